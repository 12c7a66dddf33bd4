"""One output of 16-bit input at radius class 8, images larger than one round
of workgroups: the strips of the tile loop load their input themselves.

Whole interiors, edges of the image inside a strip's window on every side,
rows and columns that no tile size divides, packed odd rows; a NaN and an
infinity at a corner, in the middle and at an edge.  float32 results against
the oracle on the same values, within the FP32 bar; the valid region's border
and what lies outside it stay as they were."""
import numpy as np
import pytest

import oracle
from tests._util import bf16_bits_to_f32, random_lobe, to_dev, to_host
from tests.test_gpu_nonfinite import _compare
from tucuda_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("nrow, ncol", [(2311, 2051), (4130, 1029), (1100, 4160)])
@pytest.mark.parametrize("nH, nV", [(9, 9), (3, 8), (8, 2)])
def test_one_output_of_large_16_bit_images(dev, kind, nrow, ncol, nH, nV):
    import torch
    import tucuda_amd
    rng = np.random.default_rng(nH * 10 + nV)
    lh, lv = random_lobe(rng, nH), random_lobe(rng, nV)
    img = synth.edge_image(5, nrow, ncol)
    for y, x, v in ((0, 0, np.nan), (nrow // 2, ncol // 2, np.inf), (nrow - 1, ncol // 3, -np.inf), (7, ncol - 1, np.nan)):
        img[y, x] = v
    if kind == "f16":
        src = img.astype(np.float16)
        vals = src.astype(np.float32)
    else:
        src = (img.view(np.uint32) >> 16).astype(np.uint16)
        vals = bf16_bits_to_f32(src)
    out = torch.full(img.shape, -5.0, device=dev)
    tucuda_amd.FIRFilter2().initialize(lh, lv).convolve(to_dev(src, dev), out)
    torch.cuda.synchronize()
    ref = np.full(img.shape, -5.0, np.float32)
    oracle.fir2(lh, lv, vals, ref, nthreads=8)
    _compare(to_host(out), ref, f"{kind} {nrow}x{ncol} {nH}/{nV}")
