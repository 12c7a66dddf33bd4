"""ICIA's moments do not depend on what ran before in the process.

The grid of a moment pass decides which tiles a lane sums in FP32, so it is
that of the pass's own kernel, whichever input type, radius class or map came
first.  Each moment is taken in a process of its own."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

pytestmark = pytest.mark.gpu

_CHILD = """
import sys
sys.path.insert(0, {root!r})
import torch, tucuda_amd
g = torch.Generator(device="cuda"); g.manual_seed(7)
x = torch.rand((2160, 3840), generator=g, device="cuda") * 255
if {first}:
    tucuda_amd.icia_moment({first}[0], x.to(getattr(torch, {first}[1])), {first}[2])
m = tucuda_amd.icia_moment({sigma}, x.to(getattr(torch, {dtype!r})), {model!r})
print("bits", m.cpu().numpy().tobytes().hex(), flush=True)
"""


def _bits(sigma, dtype, model, first):
    code = _CHILD.format(root=ROOT, first=first, sigma=sigma, dtype=dtype, model=model)
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100, check=True,
                         env=os.environ)
    return [l for l in out.stdout.splitlines() if l.startswith("bits")][0]


def test_icia_moment_does_not_depend_on_the_first_call(dev):
    """The grid of a moment pass is that of its own kernel, whichever input
    type, radius class or map ran first in the process."""
    heavy, light = (3.0, "float32", "projective"), (1.0, "uint8", "affine")
    assert _bits(*heavy, first=None) == _bits(*heavy, first=light)
    assert _bits(*light, first=None) == _bits(*light, first=heavy)
