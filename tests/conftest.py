import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (gfx950) device")


def _have_gpu():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


def pytest_collection_modifyitems(config, items):
    if _have_gpu():
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(scope="session")
def orc():
    from oracle import oracle
    oracle.lib()
    return oracle


@pytest.fixture(scope="session")
def ctx():
    """One library context for the whole GPU session (workspace reuse is part of the contract)."""
    import cuspamm_amd as sp
    c = sp.SpammContext(0)
    yield c
    c.close()


@pytest.fixture(params=[0, 1], ids=["default_unit", "macro_tiles"])
def work_unit(ctx, request):
    """The session context as it is (small outputs: gate and multiply in one kernel) and with the GEMM's work unit
    fixed to whole macro tiles, so that gate, schedule and GEMM run on small outputs too."""
    import cuspamm_amd as sp
    ctx.set_option(sp.OPT_GEMM_SHAPE, request.param)
    yield request.param
    ctx.set_option(sp.OPT_GEMM_SHAPE, 0)
