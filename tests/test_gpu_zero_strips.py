"""16-bit images with strips of zeros of both signs.

A strip's scale comes from its largest magnitude, and a bfloat16 strip reads
it from pairs of values.  A strip that holds zeros alone, some of them -0.0
(masked or rectified images), has the largest magnitude 0 and gradients 0:
its moments are those of the same image in float32, its filtered pixels the
oracle's.  ICIA's gradients never leave the chip, so a wrong scale there
shows in the moments only."""
import numpy as np
import pytest

import oracle
from tests._util import bf16_bits_to_f32, to_dev, to_host
from tests.test_gpu_icia import _oracle_moment

pytestmark = pytest.mark.gpu


def _masked(kind, nrow=200, ncol=330):
    """Values in the middle, zeros around them, a third of them -0.0; and a
    few of the smallest magnitudes of the type in one corner."""
    rng = np.random.default_rng(3)
    img = np.where(rng.random((nrow, ncol)) < 1 / 3, -0.0, 0.0).astype(np.float32)
    img[70:130, 140:230] = rng.integers(-255, 256, (60, 90))
    if kind == "f16":
        return img.astype(np.float16), img
    return (img.view(np.uint32) >> 16).astype(np.uint16), img      # small integers: exact in bfloat16


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("model", ["affine", "projective"])
@pytest.mark.parametrize("sigma", [1.0, 3.0])
def test_icia_moment_of_zero_strips(dev, kind, model, sigma):
    import tucuda_amd
    x, img = _masked(kind)
    got = tucuda_amd.icia_moment(sigma, to_dev(x, dev), model).cpu().numpy().astype(np.float64)
    want, absm = _oracle_moment(img, sigma, model)
    assert np.isfinite(got).all()
    np.testing.assert_array_less(np.abs(got - want), 5e-5 * absm + 1e-30)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("sigma", [1.0, 3.0])
def test_filters_of_zero_strips(dev, kind, sigma):
    """Six outputs, one output and (bfloat16) a batch; where the window holds
    zeros alone the result is exactly 0."""
    import torch
    import tucuda_amd
    x, img = _masked(kind)
    xd = to_dev(x, dev)
    g = tucuda_amd.FIRGaussianConvolver2(sigma)
    outs = {m: torch.full(img.shape, 7, dtype=xd.dtype, device=dev) for m in tucuda_amd.METHOD_ORDER}
    g.convolve6(xd, outs)
    one = torch.full_like(xd, 7)
    g.smooth(xd, one)
    results = [(m, outs[m]) for m in outs] + [("smooth", one)]
    if kind == "bf16":
        many = {m: torch.full_like(xd, 7) for m in tucuda_amd.METHOD_ORDER}
        tucuda_amd.GaussBatch([(xd, many, sigma)]).launch()
        results += [(m, many[m]) for m in many]
    torch.cuda.synchronize()
    lobes = oracle.gauss_lobes(sigma)
    eps = 2.0 ** -8 if kind == "bf16" else 2.0 ** -11
    for m, out in results:
        ref = np.full(img.shape, 7, np.float32)
        oracle.gauss(m, sigma, img, ref, lobes=lobes)
        got = to_host(out)
        got = (bf16_bits_to_f32(got) if kind == "bf16" else got.astype(np.float32)).astype(np.float64)
        assert (got[ref == 0] == 0).all(), m
        assert (np.abs(got - ref) <= eps * np.abs(ref) + 2e-5 * 255).all(), m
