"""ICIA's moments where single columns carry them.

The moments of u are summed per strip from powers of each pixel's place in it
and expanded to powers of u.  An image that is flat but for one vertical step
near the left border has all its gradient at small u, where an expansion about
a far point would cancel; its moments lie within 5e-5 of the sums of their
terms' magnitudes, the bar of tests/test_gpu_icia.py.  (Sigma 1: its taps sum
such a step so that both gradients are the oracle's to 1e-7, and the vertical
one exactly 0, wherever the step lies; with lobes whose tail alone is inside the
image, the gradients' own rounding is far above that bar.)  Large gradients
(their squares within a few thousand of the largest float) stay finite."""
import numpy as np
import pytest

from tests._util import to_dev
from tests.test_gpu_icia import _oracle_moment

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", ["affine", "projective"])
@pytest.mark.parametrize("ik", ["f32", "u8", "f16", "bf16"])
@pytest.mark.parametrize("col", [2, 3, 5, 6, 40, 68])
def test_icia_moment_of_one_step(dev, ik, model, col):
    import tucuda_amd
    img = np.zeros((150, 300), np.float32)
    img[:, col:] = 200
    x = {"f32": img, "u8": img.astype(np.uint8), "f16": img.astype(np.float16),
         "bf16": (img.view(np.uint32) >> 16).astype(np.uint16)}[ik]
    got = tucuda_amd.icia_moment(1.0, to_dev(x, dev), model).cpu().numpy().astype(np.float64)
    want, absm = _oracle_moment(img, 1.0, model)
    np.testing.assert_array_less(np.abs(got - want), 5e-5 * absm + 1e-30)


@pytest.mark.parametrize("model", ["affine", "projective"])
def test_icia_moment_of_large_gradients(dev, model):
    """Gradients of about 5e16, each moment below the largest float; within
    5e-5 of the terms' magnitudes of the same image scaled by a power of two
    (2^48) to ordinary values."""
    import tucuda_amd
    rng = np.random.default_rng(4)
    img = (rng.random((120, 260)) * 200).astype(np.float32)
    want, absm = _oracle_moment(img, 1.0, model)
    big = img * np.float32(2.0 ** 48)
    got = tucuda_amd.icia_moment(1.0, to_dev(big, dev), model).cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    np.testing.assert_array_less(np.abs(got * 2.0 ** -96 - want), 5e-5 * absm)
