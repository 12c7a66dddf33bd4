"""Strips that the valid region's left or right edge cuts, at every place within
a 16-byte chunk and within a 128-byte line.

Of such a strip's rows the matrix-core kernels stream the lines that are whole,
store those that are cut ordinarily (float tile loops and batches), move a
chunk that is cut inside the region, and store a strip with less than a chunk
pixel by pixel.  Rows padded to 256 bytes; six outputs (one round), a batch and
one output (tile loop) against the oracle within the FP32 bar and, for 16-bit
results, one unit; what lies outside the valid region stays as it was."""
import numpy as np
import pytest

import oracle
from tests._util import random_lobe, to_dev, to_host
from tests.test_gpu_gauss_layouts import TYPES, _as_f32, _check, _input

pytestmark = pytest.mark.gpu

FILL = {"u8": 7, "f32": -7, "f16": -7, "bf16": 0xC0E0}


def _out(nrow, ncol, kind, dev):
    import tucuda_amd
    start = np.full((nrow, ncol), FILL[kind], TYPES[kind])
    src = to_dev(start, dev)
    out = tucuda_amd.array2(nrow, ncol, src.dtype, dev)
    out.copy_(src)
    return out


def _compare(out, lh, lv, img, ik, ok, what):
    nrow, ncol = img.shape
    start = np.full((nrow, ncol), FILL[ok], TYPES[ok])
    ref, ref_f = start.copy(), np.zeros((nrow, ncol), np.float32)
    oracle.fir2(lh, lv, img, ref, True, nthreads=8)
    oracle.fir2(lh, lv, _as_f32(img, ik), ref_f, True, nthreads=8)
    got = to_host(out)
    rv, rh = lv.size & ~1, lh.size & ~1
    inside = (slice(rv, nrow - rv), slice(rh, ncol - rh))
    border = np.ones((nrow, ncol), bool)
    border[inside] = False
    assert (got[border] == start[border]).all(), what
    _check(got[inside], ref[inside], ref_f[inside], ok, what)


# The last strip's valid pixels beyond 128, or of the only strip where there is one.
WIDTHS = [0, 1, 2, 3, 5, 7, 9, 15, 17, 31, 32, 33, 47, 48, 63]


@pytest.mark.parametrize("ik, ok", [("f32", "f32"), ("bf16", "bf16"), ("f16", "f16"), ("u8", "f32"), ("u8", "u8")])
@pytest.mark.parametrize("sigma", [0.8, 1.2, 2.4])
def test_six_outputs_and_batches(dev, ik, ok, sigma):
    import torch
    import tucuda_amd
    g = tucuda_amd.FIRGaussianConvolver2(sigma)
    lobes = oracle.gauss_lobes(sigma)
    r = max(lb.size & ~1 for lb in lobes)
    jobs = []
    for w in WIDTHS:
        nrow, ncol = 2 * r + 37, 128 + r + w
        img = _input(ik, nrow, ncol)
        x = to_dev(img, dev)
        outs = {m: _out(nrow, ncol, ok, dev) for m in tucuda_amd.METHOD_ORDER}
        g.convolve6(x, outs)
        jobs.append((img, x, outs))
    torch.cuda.synchronize()
    batched = ik == ok and ik in ("f32", "bf16")
    if batched:
        bouts = [{m: _out(*img.shape, ok, dev) for m in tucuda_amd.METHOD_ORDER} for img, _, _ in jobs]
        batch = tucuda_amd.GaussBatch([(x, b, sigma) for (_, x, _), b in zip(jobs, bouts)])
        batch.launch()
        torch.cuda.synchronize()
    for i, (img, _, outs) in enumerate(jobs):
        for m in tucuda_amd.METHOD_ORDER:
            h, v = tucuda_amd.METHOD_LOBES[m]
            what = f"{ik}->{ok} sigma {sigma} {img.shape} {m}"
            _compare(outs[m], lobes[h], lobes[v], img, ik, ok, what)
            if batched:
                assert torch.equal(bouts[i][m], outs[m]), "batch " + what


@pytest.mark.parametrize("ik, ok", [("f32", "f32"), ("bf16", "bf16"), ("f16", "f16"), ("u8", "f32"), ("u8", "u8")])
@pytest.mark.parametrize("nH, nV, w", [(9, 3, 1), (9, 2, 3), (3, 5, 6), (17, 3, 13), (17, 3, 48), (4, 3, 60)])
def test_one_output_tile_loop(dev, ik, ok, nH, nV, w):
    import torch
    import tucuda_amd
    rng = np.random.default_rng(nH * 100 + w)
    lh, lv = random_lobe(rng, nH), random_lobe(rng, nV)
    img = _input(ik, 9001, 832 + (nH & ~1) + w)
    out = _out(*img.shape, ok, dev)
    tucuda_amd.FIRFilter2().initialize(lh, lv).convolve(to_dev(img, dev), out)
    torch.cuda.synchronize()
    _compare(out, lh, lv, img, ik, ok, f"{ik}->{ok} {nH}/{nV} {img.shape}")
