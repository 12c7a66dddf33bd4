"""Outputs whose rows lie far apart.

Sixteen rows of an output may span more than the 2 GiB that a strip's buffer
stores address, and one row more than a signed 32-bit byte pitch: such strips
store by plain 64-bit addresses.  The views here have a few rows, so that the
memory between them is reserved but never touched.  Reference: the same call
into ordinary rows; each result lies within the FP32 bar of the oracle, so two
differ by at most twice that and one unit of a 16-bit or 8-bit result."""
import numpy as np
import pytest

from tests._util import to_dev
from tests.test_gpu_row_lines import _same
from tucuda_amd import synth

pytestmark = pytest.mark.gpu

# (element type, row stride in elements, written rows)
CASES = [("float32", (1 << 29) + 16, 3),        # 2 GiB + 64 bytes a row
         ("float32", (1 << 29) + 3, 2),         # off every alignment
         ("bfloat16", (1 << 30) + 8, 2),
         ("uint8", (1 << 31) - 64, 2),          # the longest stride taken
         ("float32", 40 << 20, 20),             # 160 MiB: 16 rows pass 2 GiB
         ("uint8", 140 << 20, 20)]


def _far(nrow, ncol, stride, dtype, dev):
    import torch
    need = ((nrow - 1) * stride + ncol + 64) * dtype.itemsize
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip("not enough free device memory for rows this far apart")
    buf = torch.empty(need // dtype.itemsize, dtype=dtype, device=dev)
    out = torch.as_strided(buf, (nrow, ncol), (stride, 1), 0)
    out.fill_(7)
    return out


@pytest.mark.parametrize("name, stride, rows", CASES)
@pytest.mark.parametrize("family", ["mfma", "valu"])
def test_rows_far_apart(dev, monkeypatch, name, stride, rows, family):
    import torch
    import tucuda_amd
    for k in ("TUCU_GAUSS_PATH", "TUCU_FIR_PATH"):
        monkeypatch.setenv(k, "valu") if family == "valu" else monkeypatch.delenv(k, raising=False)
    dt = getattr(torch, name)
    g = tucuda_amd.FIRGaussianConvolver2(1.0)               # radius 4: every output has the same valid region
    ncol = 203
    img = to_dev(synth.edge_image(9, rows + 8, ncol), dev)
    x = img if dt.itemsize == 4 else img.to(dt)
    far, near = _far(rows, ncol - 8, stride, dt, dev), torch.full((rows, ncol - 8), 7, dtype=dt, device=dev)
    # one output; written at (0, 0): shift False
    g.smooth(x, far, False)
    g.smooth(x, near, False)
    torch.cuda.synchronize()
    _same(far.clone(), near, (name, stride, "smooth"))
    # the six-output kernel
    far.fill_(7)
    g.convolve6(x, {"diffH": far}, False)
    g.convolve6(x, {"diffH": near}, False)
    torch.cuda.synchronize()
    _same(far.clone(), near, (name, stride, "diffH"))


@pytest.mark.parametrize("name, stride, rows", [c for c in CASES if c[0] != "uint8"])
def test_batch_rows_far_apart(dev, name, stride, rows):
    """A batch (written at the input's places) with one such job among
    ordinary ones, each compared."""
    import torch
    import tucuda_amd
    dt = getattr(torch, name)
    ncol, nrow = 150, rows + 8                              # radius 4: rows 4 .. rows + 3 are written
    img = to_dev(synth.edge_image(10, nrow, ncol), dev).to(dt)
    small = to_dev(synth.edge_image(11, 90, 100), dev).to(dt)
    far = _far(nrow, ncol, stride, dt, dev)
    outs = {"smooth": torch.full_like(small, 7), "diffVV": torch.full_like(small, 7)}
    near, nouts = torch.full((nrow, ncol), 7, dtype=dt, device=dev), {k: torch.full_like(v, 7) for k, v in outs.items()}
    g = tucuda_amd.FIRGaussianConvolver2(1.0)
    tucuda_amd.GaussBatch([(img, {"smooth": far}, 1.0), (small, outs, 1.0)]).launch()
    g.convolve6(img, {"smooth": near})
    g.convolve6(small, nouts)
    torch.cuda.synchronize()
    _same(far.clone(), near, (name, stride, "batch"))
    for k in outs:
        _same(outs[k], nouts[k], (name, k, "ordinary job"))


def test_second_job_of_a_batch(dev):
    """Jobs of a batch of which the first has rows off 128-byte lines."""
    import torch
    import tucuda_amd
    gen = torch.Generator(device=dev)
    gen.manual_seed(5)
    for name in ("float32", "bfloat16"):
        dt = getattr(torch, name)
        x = (torch.rand((1601, 2051), generator=gen, device=dev) * 255).to(dt)
        big = torch.full_like(x, 7)
        small, ref = (tucuda_amd.array2(90, 100, dt, dev) for _ in range(2))
        for sigma in (1.2, 3.0):
            small.fill_(7)
            ref.fill_(7)
            tucuda_amd.GaussBatch([(x, {"smooth": big}, sigma), (x[:90, :100], {"smooth": small}, sigma)]).launch()
            tucuda_amd.FIRGaussianConvolver2(sigma).smooth(x[:90, :100], ref)
            torch.cuda.synchronize()
            _same(small, ref, (name, sigma))
