"""The multiply calls of the Python mirror, without a GPU: what native code answers where torch throws.  In a process of its own, which
an exception through the interpreter's frames would end."""
import os
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
