"""Output rows that start anywhere in a 128-byte line, and images narrower
than one 16-byte load.

The matrix-core kernels choose their stores by where output rows start (whole
lines streaming, shared lines by ordinary stores, 16-bit rows off a 4-pixel
boundary by plain addresses), large images with such rows take their tiles row
by row, and narrow element types load their window in 16-byte chunks, byte by
byte where a row is shorter than one.  Reference: the same call into rows
padded to 256 bytes; each result lies within the FP32 bar of the oracle, so two
differ by at most twice that and one unit of a 16-bit result.  Narrow images are compared with the oracle itself."""
import numpy as np
import pytest

import oracle
from tests._util import ABS_TOL, REL_TOL, random_lobe, to_dev, to_host
from tests.test_gpu_gauss_layouts import TYPES, _as_f32, _check, _input

pytestmark = pytest.mark.gpu

EPS = {"float32": 0.0, "float16": 2.0 ** -10, "bfloat16": 2.0 ** -7}


def _same(got, ref, what):
    g, r = got.double(), ref.double()
    if got.dtype.itemsize == 1:
        bad = (g - r).abs() > 1
    else:
        eps = EPS[str(got.dtype).split(".")[1]]
        bad = ~((g - r).abs() <= (2 * REL_TOL * r.abs()).clamp(min=2 * ABS_TOL) + eps * r.abs() + 1e-30)
    assert not bool(bad.any()), (what, int(bad.sum()))


def _packed(nrow, ncol, off, dtype, dev):
    """A view of nrow x ncol packed rows starting off elements into a buffer."""
    import torch
    buf = torch.full((nrow * ncol + off + 64,), 7, dtype=dtype, device=dev)
    return buf, torch.as_strided(buf, (nrow, ncol), (ncol, 1), off)


# The first size is one round of workgroups, the others the tile loop.
@pytest.mark.parametrize("nrow, ncol, off", [(130, 331, 1), (1601, 2051, 0), (1601, 2052, 3), (1601, 2056, 4),
                                             (1537, 2064, 0), (1537, 2080, 8)])
@pytest.mark.parametrize("kind, okind", [("float32", "float32"), ("bfloat16", "bfloat16"), ("float16", "float16"),
                                         ("uint8", "float32"), ("uint8", "uint8")])
@pytest.mark.parametrize("sigma", [1.2, 3.0])
def test_rows_at_any_offset(dev, nrow, ncol, off, kind, okind, sigma):
    import torch
    import tucuda_amd
    it, ot = getattr(torch, kind), getattr(torch, okind)
    gen = torch.Generator(device=dev)
    gen.manual_seed(5)
    x = (torch.rand((nrow, ncol), generator=gen, device=dev) * 255).to(it)
    g = tucuda_amd.FIRGaussianConvolver2(sigma)
    bufs, outs, refs = {}, {}, {}
    for m in tucuda_amd.METHOD_ORDER:
        bufs[m], outs[m] = _packed(nrow, ncol, off, ot, dev)
        refs[m] = tucuda_amd.array2(nrow, ncol, ot, dev)
        refs[m].fill_(7)
    g.convolve6(x, outs)
    g.convolve6(x, refs)
    for m in tucuda_amd.METHOD_ORDER:
        _same(outs[m], refs[m], (m, kind, okind))
        # outside the view, and outside the valid region
        assert bool((bufs[m][:off] == 7).all()) and bool((bufs[m][nrow * ncol + off:] == 7).all()), m
        h, v = tucuda_amd.METHOD_LOBES[m]
        n = [a.size for a in tucuda_amd.FIRGaussianConvolver2.lobes(sigma)]
        rh, rv = n[h] & ~1, n[v] & ~1
        o = outs[m]
        for edge in (o[:rv], o[nrow - rv:], o[:, :rh], o[:, ncol - rh:]):
            assert bool((edge == 7).all()), m
    # one output, and the batch
    buf, out = _packed(nrow, ncol, off, ot, dev)
    g.smooth(x, out)
    _same(out, refs["smooth"], ("smooth", kind, okind))
    if kind == okind and kind in ("float32", "bfloat16"):
        for b in bufs.values():
            b.fill_(7)
        small = tucuda_amd.array2(90, 100, ot, dev)
        batch = tucuda_amd.GaussBatch([(x, outs, sigma), (x[:90, :100], {"smooth": small}, sigma)])
        batch.launch()
        torch.cuda.synchronize()
        for m in tucuda_amd.METHOD_ORDER:
            _same(outs[m], refs[m], (m, kind, "batch"))
            assert bool((bufs[m][:off] == 7).all()) and bool((bufs[m][nrow * ncol + off:] == 7).all()), m


@pytest.mark.parametrize("ik, ok", [("u8", "u8"), ("u8", "f32"), ("bf16", "bf16"), ("f16", "f32")])
@pytest.mark.parametrize("nrow, ncol", [(5, 5), (6, 7), (40, 9), (17, 15), (90, 16), (33, 17)])
@pytest.mark.parametrize("nH, nV", [(3, 3), (2, 5), (5, 2)])
def test_narrow_images(dev, ik, ok, nrow, ncol, nH, nV):
    import torch
    import tucuda_amd
    rng = np.random.default_rng(7)
    lh, lv = random_lobe(rng, nH), random_lobe(rng, nV)
    img = _input(ik, nrow, ncol)
    fill = {"u8": 7, "bf16": 0xC0E0}.get(ok, -7)
    start = np.full((nrow, ncol), fill, TYPES[ok])
    ref, ref_f = start.copy(), np.zeros((nrow, ncol), np.float32)
    oracle.fir2(lh, lv, img, ref, True)
    oracle.fir2(lh, lv, _as_f32(img, ik), ref_f, True)
    out = to_dev(start, dev)
    tucuda_amd.FIRFilter2().initialize(lh, lv).convolve(to_dev(img, dev), out)
    torch.cuda.synchronize()
    got = to_host(out)
    rv, rh = nV & ~1, nH & ~1
    valid = np.zeros((nrow, ncol), bool)
    if nrow > 2 * rv and ncol > 2 * rh:
        valid[rv:nrow - rv, rh:ncol - rh] = True
    assert (got[~valid] == start[~valid]).all()
    if valid.any():
        cut = np.ix_(valid.any(1), valid.any(0))
        _check(got[cut], ref[cut], ref_f[cut], ok, f"{ik}->{ok} {nrow}x{ncol} {nH}/{nV}")
