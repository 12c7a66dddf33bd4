"""Taps that the matrix products cannot carry.

The matrix-core kernels scale each lobe by a power of two so that its largest
tap lies in [2^5, 2^6).  Taps that are not finite, or so small that the scale
itself is out of range, go to the FP32 form instead: every output is the sum
of the tap products, with the NaN, +Inf and -Inf of the reference's sums."""
import numpy as np
import pytest

import oracle
from tests._util import to_dev, to_host
from tests.test_gpu_nonfinite import _compare
from tucuda_amd import synth

pytestmark = pytest.mark.gpu


def _taps(n, seed):
    t = np.random.default_rng(seed).standard_normal(n)
    return (t / np.abs(t).sum()).astype(np.float32)


@pytest.mark.parametrize("nrow, ncol", [(75, 140), (1601, 2051)])     # one round of workgroups, the tile loop
@pytest.mark.parametrize("n", [9, 33])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("where", ["V", "H"])
def test_taps_that_are_not_finite(dev, nrow, ncol, n, value, where):
    import torch
    import tucuda_amd
    tv, th = np.abs(_taps(n, 1)), np.abs(_taps(n, 2))    # one sign: the order of the sums plays no part
    (tv if where == "V" else th)[n // 2 - 2] = value
    img = synth.edge_image(3, nrow, ncol) + np.float32(1)
    for kind in ("f32", "bf16"):
        x = img
        if kind == "bf16":
            x = (img.view(np.uint32) >> 16).astype(np.uint16)
        vals = img if kind == "f32" else (x.astype(np.uint32) << 16).view(np.float32)
        out = torch.full(img.shape, -5.0, device=dev)
        tucuda_amd.SeparableFilter2(th, tv).convolve(to_dev(x, dev), out)
        ref = np.full(img.shape, -5.0, np.float32)
        oracle.fir2_taps(th, tv, vals, ref)
        _compare(to_host(out), ref, f"{kind} {where} {value}")


@pytest.mark.parametrize("n", [9, 33])
@pytest.mark.parametrize("where", ["V", "H"])
@pytest.mark.parametrize("scale", [1e-38, 1e-40])
def test_taps_below_the_scale(dev, n, where, scale):
    """Taps whose power-of-two scale overflows.  The oracle sums the same
    float32 taps in double."""
    import torch
    import tucuda_amd
    tv, th = _taps(n, 5), _taps(n, 6)
    if where == "V":
        tv = (tv.astype(np.float64) * scale).astype(np.float32)
    else:
        th = (th.astype(np.float64) * scale).astype(np.float32)
    img = (synth.edge_image(4, 90, 170).astype(np.float64) * 2.0 ** 60).astype(np.float32)
    out = torch.full(img.shape, np.nan, device=dev)
    tucuda_amd.SeparableFilter2(th, tv).convolve(to_dev(img, dev), out)
    ref = np.full(img.shape, np.nan, np.float32)
    oracle.fir2_taps(th, tv, img, ref, precision="f64")
    got, ref = to_host(out).astype(np.float64), ref.astype(np.float64)
    assert (np.isnan(got) == np.isnan(ref)).all()
    ok = ~np.isnan(ref)
    assert np.abs(got[ok] - ref[ok]).max() <= 4e-5 * np.abs(ref[ok]).max()
