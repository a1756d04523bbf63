"""The multiply calls of the Python mirror, without a GPU: what native code answers where torch throws, and what is there without it.  In
processes of their own, which an exception through the interpreter's frames would end."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a matrix "on the GPU" of exactly torch's tensor type whose sizes are symbols: torch throws where its address is asked for
SYMBOLIC = """
import torch
from cuspamm_amd import api
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import ShapeEnv
api.load_library()
mode = FakeTensorMode(shape_env=ShapeEnv())
fake = mode.from_tensor(torch.empty(64, 64), static_shapes=False)
with mode:
    fake = fake.to("cuda")
X = torch._to_functional_tensor(fake)
assert type(X) is torch.Tensor and X.is_cuda and X.dim() == 2 and X.is_contiguous()
flags = (False,) * 5
assert api._call.multiply(1, X, X, X, 32, 1.0, *flags) is None
assert api._call.multiply_noalloc(1, X, X, X, 32, 1.0, *flags[:3]) is None
"""


def python(code, **env):
    return subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=dict(os.environ, PYTHONPATH=ROOT, **env), text=True, stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, timeout=300)


@pytest.mark.parametrize("code", [SYMBOLIC], ids=["symbolic sizes"])
def test_what_torch_throws_at_is_left_to_the_checks_in_python(code):
    done = python(code)
    assert done.returncode == 0, done.stdout[-2000:]


LOADS = """
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import cuspamm_amd as sp
    from cuspamm_amd import api
    lib = sp.load_library()
assert lib.spamm_version() >= 100
ours = [str(w.message) for w in seen if "multiply calls" in str(w.message)]
"""


def package_without_native_calls(tmp_path, stand_in=None):
    """A copy of the Python files; `stand_in`: of a _spamm_call that is not this torch's."""
    pkg = tmp_path / "cuspamm_amd"
    pkg.mkdir()
    here = os.path.join(ROOT, "cuspamm_amd")
    for name in os.listdir(here):
        if name.endswith(".py"):
            shutil.copy(os.path.join(here, name), pkg / name)
    if stand_in:
        (pkg / "_spamm_call.py").write_text(stand_in)
    return tmp_path


@pytest.mark.parametrize("stand_in", [None, "torch_version = '0.1'", "def multiply(*a): return -1"], ids=["absent", "another torch's", "of unknown make"])
def test_the_engine_loads_without_native_calls(tmp_path, stand_in):
    where = package_without_native_calls(tmp_path, stand_in)
    (tmp_path / "m.csv").write_text("1,2\n3,4\n")
    code = LOADS + """
assert len(ours) == 1 and api._call is api.PythonCalls, seen
assert api._call.multiply(1, 2) is None and api._call.multiply_noalloc() is None
assert (sp.load_csv("m.csv", 2, 2) == [[1, 2], [3, 4]]).all()
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=where, text=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=300,
                          env=dict(os.environ, PYTHONPATH=str(where), SPAMM_LIBRARY_PATH=os.path.join(ROOT, "cuspamm_amd", "libspamm_gfx950.so")))
    assert done.returncode == 0, done.stdout[-2000:]


def test_native_calls_are_what_runs_where_they_were_built():
    done = python(LOADS + "assert not ours and api._call.__name__ == 'cuspamm_amd._spamm_call', ours")
    assert done.returncode == 0, done.stdout[-2000:]
