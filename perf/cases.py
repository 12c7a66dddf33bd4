"""Workloads of tucuda_amd by which its speed is followed from change to change.

``listed()`` names the fixed ones, ``draw(rng)`` gives more of the same
ranges.  A case is a dict of plain values; ``prepare(case, seed)`` makes what
a program holds before the call (images, outputs, convolver, batch handle or
captured graph), ``run(state)`` is one pass through the public entry points,
``work(case)`` the bytes and operations a pass cannot do without (each input
read once, each output pixel written once, two operations a tap), and
``exact(case, seed)`` the same outputs in float64 from plain torch.
"""
import math

import numpy as np
import torch

import tucuda_amd

DTYPES = {"u8": torch.uint8, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ESIZE = {"u8": 1, "f32": 4, "f16": 2, "bf16": 2}
METHODS = ("smooth", "diffH", "diffV", "diffHH", "diffHV", "diffVV")
# (horizontal lobe, vertical lobe) of each method
METHOD_LOBES = {"smooth": (0, 0), "diffH": (1, 0), "diffV": (0, 1), "diffHH": (2, 0), "diffHV": (1, 1),
                "diffVV": (0, 2)}
RULES = {"reference": tucuda_amd.TUCU_RULE_REFERENCE, "ceil4": tucuda_amd.TUCU_RULE_CEIL4SIGMA}
# Half-extent and whether the operator reads one row only, of cu::subsample's operators drawn here.
SUB_OPS = {"identity1x1": (0, 0), "diffHV3x3": (1, 1), "sobelAbs3x3": (1, 1), "gaussian5x5": (2, 2)}


def listed():
    return [
        # The smallest call: one smoothed VGA frame (the reference's demo size), where latency is all.
        {"name": "smooth_vga_f32", "kind": "methods", "methods": 1, "nrow": 480, "ncol": 640, "in": "f32", "out": "f32",
         "sigma": 2.0, "rule": "reference", "layout": "array2"},
        # A program moved over from the reference: its six methods called one after the other.
        {"name": "methods6_1080p_f32", "kind": "methods", "methods": 6, "nrow": 1080, "ncol": 1920, "in": "f32",
         "out": "f32", "sigma": 3.0, "rule": "reference", "layout": "array2"},
        # The headline workload, one call per frame.
        {"name": "gauss6_1080p_f32", "kind": "gauss6", "nrow": 1080, "ncol": 1920, "in": "f32", "out": "f32",
         "sigma": 3.0, "rule": "reference", "layout": "array2"},
        # The headline workload as a video program issues it: 16 frames of a clip replayed from one HIP graph.
        {"name": "stream16_1080p_f32", "kind": "stream", "frames": 16, "nrow": 1080, "ncol": 1920, "in": "f32",
         "out": "f32", "sigma": 3.0, "rule": "reference", "layout": "array2"},
        # 16-bit storage on a large frame.
        {"name": "gauss6_2160p_bf16", "kind": "gauss6", "nrow": 2160, "ncol": 3840, "in": "bf16", "out": "bf16",
         "sigma": 3.0, "rule": "reference", "layout": "array2"},
        # An odd-sized photograph in plain torch tensors, rows packed at their width.
        {"name": "gauss6_odd_f32_packed", "kind": "gauss6", "nrow": 3001, "ncol": 4003, "in": "f32", "out": "f32",
         "sigma": 1.6, "rule": "ceil4", "layout": "packed"},
        # General (asymmetric) taps on a large byte image, half-precision result.
        {"name": "taps_4096_u8_f16", "kind": "taps", "nH": 17, "nV": 9, "nrow": 4096, "ncol": 4096, "in": "u8",
         "out": "f16", "layout": "array2"},
        # FIRFilter2 from bytes to bytes, as the reference instantiates it.
        {"name": "fir_2160p_u8_u8", "kind": "fir", "nH": 9, "nV": 5, "nrow": 2160, "ncol": 3840, "in": "u8",
         "out": "u8", "layout": "array2"},
        # A four-level Gaussian pyramid of a large frame.
        {"name": "pyramid4_2160p_f32", "kind": "pyramid", "levels": 4, "nrow": 2160, "ncol": 3840, "in": "f32",
         "out": "f32", "sigma": 2.0, "rule": "reference", "layout": "array2"},
        # The subsampling operator with the largest stencil.
        {"name": "subsample_2160p_f32", "kind": "subsample", "op": "gaussian5x5", "nrow": 2160, "ncol": 3840,
         "in": "f32", "out": "f32", "layout": "array2"},
        # Image alignment: the error moment of a grey camera frame.
        {"name": "icia_2160p_u8_projective", "kind": "icia", "model": "projective", "nrow": 2160, "ncol": 3840,
         "in": "u8", "sigma": 2.0, "rule": "reference", "layout": "array2"},
        # Batched mode (and what the server launches): 256 images of uneven sizes and sigmas.
        {"name": "batch256_bf16", "kind": "batch", "images": 256, "low": 240, "high": 2160, "in": "bf16", "out": "bf16",
         "rule": "ceil4", "layout": "array2", "sizes": 3},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["methods", "gauss6", "gauss6", "stream", "taps", "fir", "pyramid", "subsample", "icia", "batch",
                       "batch"])
    case = {"kind": kind, "layout": rng.choice(["array2", "array2", "packed"])}
    if kind == "batch":
        t = rng.choice(["f32", "bf16"])
        case.update({"images": size(8, 96), "low": 240, "high": 2160, "in": t, "out": t, "rule": "ceil4",
                     "sizes": rng.randrange(1 << 20)})
        return case
    hi = 2200 if kind == "stream" else 4320
    nrow, ncol = size(240, hi), size(240, hi)
    case.update({"nrow": nrow, "ncol": int(min(max(ncol, nrow / 2), 2 * nrow))})
    t = rng.choice(["f32", "f32", "bf16", "f16", "u8"])
    case["in"], case["out"] = t, "f32" if t == "u8" else t
    if kind in ("methods", "gauss6", "stream", "pyramid", "icia"):
        case["sigma"] = round(rng.uniform(0.8, 4.0), 3)
        case["rule"] = rng.choice(["reference", "ceil4"])
    if kind == "methods":
        case["methods"] = rng.choice([1, 2, 6])
    elif kind == "stream":
        case["frames"] = rng.randint(4, 16)
    elif kind == "taps":
        case["nH"], case["nV"] = 2 * rng.randint(1, 16) + 1, 2 * rng.randint(1, 16) + 1
    elif kind == "fir":
        case["nH"], case["nV"] = rng.choice([2, 3, 4, 5, 8, 9, 16, 17]), rng.choice([2, 3, 4, 5, 8, 9, 16, 17])
        if t == "u8":
            case["out"] = rng.choice(["u8", "f32", "f16"])
    elif kind == "pyramid":
        case["levels"] = rng.randint(2, 4)
    elif kind == "subsample":
        case["op"] = rng.choice(sorted(SUB_OPS)) if t != "u8" else "identity1x1"
    elif kind == "icia":
        case["model"] = rng.choice(["affine", "projective"])
        del case["out"]
    return case


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _pixels(gen, nrow, ncol):
    """Uniform [0, 255) noise with a few step edges, float32."""
    img = torch.rand((nrow, ncol), generator=gen, device="cuda") * 191.0
    par = torch.rand((4, 3), generator=gen, device="cuda")
    yy = torch.arange(nrow, device="cuda", dtype=torch.float32)[:, None]
    xx = torch.arange(ncol, device="cuda", dtype=torch.float32)[None, :]
    th = par[:, 0] * (2.0 * math.pi)
    for k in range(4):
        img += 16.0 * (((xx - par[k, 1] * ncol) * torch.cos(th[k]) + (yy - par[k, 2] * nrow) * torch.sin(th[k])) > 0.0)
    return img


def _image(case, nrow, ncol, dtype):
    if case["layout"] == "packed":
        return torch.zeros((nrow, ncol), dtype=DTYPES[dtype], device="cuda")
    return tucuda_amd.array2(nrow, ncol, DTYPES[dtype], "cuda")


def _clip(case):
    """The same output image of every frame of a clip, frames x rows x columns."""
    frames, nrow, ncol = case["frames"], case["nrow"], case["ncol"]
    return _image(case, frames * nrow, ncol, case["out"]).unflatten(0, (frames, nrow))


def _input(case, gen, nrow, ncol):
    img = _image(case, nrow, ncol, case["in"])
    img.copy_(_pixels(gen, nrow, ncol))
    return img


def _lobe(n):
    """A FIRFilter2 half-kernel of n entries, outermost first: a smoothing
    kernel (odd n, unit sum) or a derivative (even n)."""
    r = n & ~1
    s = max(r / 2.5, 0.8)
    k = np.arange(r, -1 if n & 1 else 0, -1, dtype=np.float64)
    w = np.exp(-0.5 * (k / s) ** 2)
    if n & 1:
        return (w / (2 * w[:-1].sum() + w[-1])).astype(np.float32)
    return (-k * w / (2 * (k * k * w).sum())).astype(np.float32)


def _taps(n, phase):
    """n asymmetric taps (a decaying wave), unit absolute sum."""
    i = np.arange(n, dtype=np.float64)
    w = np.exp(-i / (0.4 * n + 1)) * np.cos(0.7 * i + phase)
    return (w / np.abs(w).sum()).astype(np.float32)


def _batch_sizes(case):
    """(rows, columns, sigma) of each image: sides log-uniform, aspect within
    [0.5, 2], sigma uniform in [0.8, 4)."""
    rng = np.random.default_rng(case["sizes"])
    lo, hi = math.log(case["low"]), math.log(case["high"])
    out = []
    for a, b, c in rng.random((case["images"], 3)):
        h, w = int(round(math.exp(lo + (hi - lo) * a))), int(round(math.exp(lo + (hi - lo) * b)))
        out.append((h, int(min(max(w, h / 2), 2 * h)), float(np.float32(0.8 + 3.2 * c))))
    return out


def _batch_layout(case):
    """Offset (elements) and row pitch of each image's six outputs in one
    buffer, and its size: rows padded to 256 bytes, or packed."""
    per = 256 // ESIZE[case["out"]]
    pos, places = 0, []
    for h, w, _ in _batch_sizes(case):
        pitch = w if case["layout"] == "packed" else (w + per - 1) // per * per
        mine = []
        for _ in range(6):
            mine.append(pos)
            pos += (h * pitch + per - 1) // per * per
        places.append((pitch, mine))
    return places, pos


def _levels(case):
    return [(case["nrow"] >> k, case["ncol"] >> k) for k in range(case["levels"])]


def prepare(case, seed):
    kind, gen = case["kind"], _generator(seed)
    s = {"kind": kind}
    if kind == "batch":
        places, total = _batch_layout(case)
        buf = torch.zeros(total, dtype=DTYPES[case["out"]], device="cuda")
        jobs = []
        for (h, w, sigma), (pitch, at) in zip(_batch_sizes(case), places):
            outs = [torch.as_strided(buf, (h, w), (pitch, 1), p) for p in at]
            jobs.append((_input(case, gen, h, w), outs, sigma))
        s.update(buf=buf, jobs=jobs, batch=tucuda_amd.GaussBatch(jobs, rule=RULES[case["rule"]]))
        return s
    nrow, ncol = case["nrow"], case["ncol"]
    if kind == "pyramid":
        s["g"] = tucuda_amd.FIRGaussianConvolver2(case["sigma"], rule=RULES[case["rule"]])
        s["levels"] = [_input(case, gen, nrow, ncol)]
        s["levels"] += [_image(case, h, w, case["out"]) for h, w in _levels(case)[1:]]
        return s
    if kind == "stream":
        g = tucuda_amd.FIRGaussianConvolver2(case["sigma"], rule=RULES[case["rule"]])
        ins = [_input(case, gen, nrow, ncol) for _ in range(case["frames"])]
        clip = {m: _clip(case) for m in METHODS}        # output m of every frame, frames one after the other
        outs = [{m: clip[m][i] for m in METHODS} for i in range(len(ins))]
        g.convolve6(ins[0], outs[0])
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for x, o in zip(ins, outs):
                g.convolve6(x, o)
        s.update(g=g, ins=ins, outs=outs, clip=clip, graph=graph)
        return s
    s["x"] = _input(case, gen, nrow, ncol)
    if kind == "icia":
        s.update(sigma=case["sigma"], model=case["model"], rule=RULES[case["rule"]])
    elif kind == "subsample":
        s.update(out=_image(case, nrow // 2, ncol // 2, case["out"]), op=case["op"])
    elif kind == "fir":
        s.update(f=tucuda_amd.FIRFilter2().initialize(_lobe(case["nH"]), _lobe(case["nV"])),
                 out=_image(case, nrow, ncol, case["out"]))
    elif kind == "taps":
        s.update(f=tucuda_amd.SeparableFilter2(_taps(case["nH"], 0.3), _taps(case["nV"], -0.4)),
                 out=_image(case, nrow, ncol, case["out"]))
    else:
        n = case.get("methods", 6)
        s["g"] = tucuda_amd.FIRGaussianConvolver2(case["sigma"], rule=RULES[case["rule"]])
        s["outs"] = {m: _image(case, nrow, ncol, case["out"]) for m in METHODS[:n]}
    return s


def run(s):
    kind = s["kind"]
    if kind == "batch":
        s["batch"].launch()
        return s["buf"]
    if kind == "stream":
        s["graph"].replay()
        return s["clip"]
    if kind == "pyramid":
        lv = s["levels"]
        for k in range(len(lv) - 1):
            s["g"].smoothSubsample(lv[k], lv[k + 1])
        return lv[1:]
    if kind == "icia":
        return tucuda_amd.icia_moment(s["sigma"], s["x"], s["model"], rule=s["rule"])
    if kind == "subsample":
        tucuda_amd.subsample(s["x"], s["out"], s["op"])
        return s["out"]
    if kind in ("fir", "taps"):
        s["f"].convolve(s["x"], s["out"])
        return s["out"]
    if kind == "methods":
        for m, o in s["outs"].items():
            getattr(s["g"], m)(s["x"], o)
        return s["outs"]
    s["g"].convolve6(s["x"], s["outs"])
    return s["outs"]


# -------------------------------------------------------------------- work
def _radii(case, sigma=None):
    l0, l1, l2 = _gauss_lobes(case["sigma"] if sigma is None else sigma, case["rule"])
    return len(l0) - 1, len(l1), len(l2) - 1


def _gauss_work(case, nrow, ncol, methods, r):
    px_in = nrow * ncol
    px_out = flops = 0
    for m in methods:
        h, v = METHOD_LOBES[m]
        n = max(0, nrow - 2 * r[v]) * max(0, ncol - 2 * r[h])
        px_out += n
        flops += n * 2 * (2 * r[h] + 1)
    for v in {METHOD_LOBES[m][1] for m in methods}:         # the vertical sums are shared
        flops += px_in * 2 * (2 * r[v] + 1)
    return {"bytes": px_in * ESIZE[case["in"]] + px_out * ESIZE[case["out"]], "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_gauss_work(case, h, w, METHODS, _radii(case, sg)) for h, w, sg in _batch_sizes(case)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    nrow, ncol = case["nrow"], case["ncol"]
    es_in = ESIZE[case["in"]]
    if kind == "pyramid":
        r, lv, w = _radii(case)[0], _levels(case), {"bytes": 0, "flops": 0}
        for (h, c), (h2, c2) in zip(lv, lv[1:]):
            w["bytes"] += h * c * (es_in if (h, c) == lv[0] else ESIZE[case["out"]]) + h2 * c2 * ESIZE[case["out"]]
            w["flops"] += (h2 * c + h2 * c2) * 2 * (2 * r + 1)
        return w
    if kind == "subsample":
        ry = SUB_OPS[case["op"]][0]
        rows = nrow // 2 if ry == 0 else nrow
        out = (nrow // 2) * (ncol // 2)
        return {"bytes": rows * ncol * es_in + out * ESIZE[case["out"]], "flops": out * 2 * (2 * ry + 1) ** 2}
    if kind == "icia":
        w = _gauss_work(dict(case, out="f32"), nrow, ncol, ("diffH", "diffV"), _radii(case))
        nm = 21 if case["model"] == "affine" else 36
        return {"bytes": nrow * ncol * es_in + nm * 4, "flops": w["flops"] + nrow * ncol * 2 * nm}
    if kind in ("fir", "taps"):
        rh, rv = (case["nH"] & ~1, case["nV"] & ~1) if kind == "fir" else (case["nH"] // 2, case["nV"] // 2)
        out = (nrow - 2 * rv) * (ncol - 2 * rh)
        return {"bytes": nrow * ncol * es_in + out * ESIZE[case["out"]],
                "flops": out * 2 * (2 * rh + 1) + nrow * ncol * 2 * (2 * rv + 1)}
    w = _gauss_work(case, nrow, ncol, METHODS[:case.get("methods", 6)], _radii(case))
    return {k: v * case.get("frames", 1) for k, v in w.items()}


# ------------------------------------------------------------------- exact
def _gauss_lobes(sigma, rule):
    """The three lobes (outermost entry first) of a sigma, rounded to float32
    at each step as the library computes them."""
    f = np.float32
    sigma = f(sigma)
    dx = np.arange(17, dtype=np.float32) / sigma
    g = np.exp(f(-0.5) * (dx * dx)).astype(np.float32)
    lb = [g, -dx * g, (dx * dx - f(1)) * g]
    if rule == "ceil4":
        r = min(max(int(math.ceil(f(4) * sigma)), 1), 16)
        n = (r + 1, r, r + 1)
    else:
        n = []
        for a, even in zip(lb, (True, False, True)):
            siz = int(np.nonzero(np.abs(a) > np.abs(a).max() * f(0.01))[0][-1]) + 1
            sizes = (2, 5, 9, 17) if even else (1, 4, 8, 16)
            k = next(i for i, lim in enumerate(sizes) if siz <= lim or i == 3)
            n.append(((3, 5, 9, 17) if even else (2, 4, 8, 16))[k])
    i = np.arange(17, dtype=np.float32)

    def total(v):                                           # summed in order
        return abs(np.cumsum(v, dtype=np.float32)[-1])

    return (lb[0][:n[0]][::-1] / total(np.concatenate([lb[0][:1], f(2) * lb[0][1:n[0]]])),
            lb[1][1:n[1] + 1][::-1] / total((f(2) * i * lb[1])[:n[1]]),
            lb[2][:n[2]][::-1] / total((i * i * lb[2])[1:n[2]]))


def _full(lobe, symmetric):
    """The taps of a half-kernel, first (left / upper) tap first."""
    a = [float(v) for v in lobe]
    return a + a[-2::-1] if symmetric else a + [0.0] + [-v for v in a[::-1]]


def _correlate(x, taps, dim):
    n = x.shape[dim] - len(taps) + 1
    out = torch.zeros_like(x.narrow(dim, 0, n))
    for i, t in enumerate(taps):
        if t:
            out.add_(x.narrow(dim, i, n), alpha=t)
    return out


def _separable(x, th, tv):
    """The filtered image in float64, zero outside the valid region."""
    out = torch.zeros_like(x)
    rh, rv = len(th) // 2, len(tv) // 2
    if x.shape[0] > 2 * rv and x.shape[1] > 2 * rh:
        out[rv:x.shape[0] - rv, rh:x.shape[1] - rh] = _correlate(_correlate(x, tv, 0), th, 1)
    return out


def _gauss_exact(x, sigma, rule, methods):
    lobes = _gauss_lobes(sigma, rule)
    full = [_full(lobes[k], k != 1) for k in range(3)]
    return {m: _separable(x, full[METHOD_LOBES[m][0]], full[METHOD_LOBES[m][1]]) for m in methods}


def _subsample_exact(x, op):
    ry, rx = SUB_OPS[op]
    h, w = x.shape
    out = torch.zeros((h // 2, w // 2), dtype=x.dtype, device=x.device)
    y = [k for k in range(h // 2) if 2 * k >= ry and 2 * k + ry < h]
    c = [k for k in range(w // 2) if 2 * k >= rx and 2 * k + rx < w]
    if not y or not c:
        return out

    def p(dy, dx):
        return x[2 * y[0] + dy:2 * y[-1] + dy + 1:2, 2 * c[0] + dx:2 * c[-1] + dx + 1:2]

    if op == "identity1x1":
        v = p(0, 0).clone()
    elif op == "diffHV3x3":
        v = 0.25 * (p(-1, -1) - p(-1, 1) - p(1, -1) + p(1, 1))
    elif op == "sobelAbs3x3":
        sh = 0.125 * (p(-1, 1) - p(-1, -1) + p(1, 1) - p(1, -1)) + 0.25 * (p(0, 1) - p(0, -1))
        sv = 0.125 * (p(1, -1) - p(-1, -1) + p(1, 1) - p(-1, 1)) + 0.25 * (p(1, 0) - p(-1, 0))
        v = sh.abs() + sv.abs()
    else:
        b = (0.0625, 0.25, 0.375, 0.25, 0.0625)
        v = sum(b[i] * b[j] * p(i - 2, j - 2) for i in range(5) for j in range(5))
    out[y[0]:y[-1] + 1, c[0]:c[-1] + 1] = v
    return out


def _moment_exact(x, case):
    """Upper triangle of sum a a^T, a the derivative vector of the affine or
    projective map at (s u, s v)."""
    g = _gauss_exact(x, case["sigma"], case["rule"], ("diffH", "diffV"))
    eh, ev = g["diffH"], g["diffV"]
    s = 1.0 / max(x.shape)
    v = (s * torch.arange(x.shape[0], device=x.device, dtype=x.dtype))[:, None]
    u = (s * torch.arange(x.shape[1], device=x.device, dtype=x.dtype))[None, :]
    a = [eh * u, eh * v, eh, ev * u, ev * v, ev]
    if case["model"] == "projective":
        t = -(eh * u + ev * v)
        a += [t * u, t * v]
    return torch.stack([(a[i] * a[j]).sum() for i in range(len(a)) for j in range(i, len(a))])


def exact(case, seed):
    kind = case["kind"]
    if case.get("out") == "u8":
        return None
    gen = _generator(seed)
    if kind == "batch":
        places, total = _batch_layout(case)
        buf = torch.zeros(total, dtype=torch.float64, device="cuda")
        for (h, w, sigma), (pitch, at) in zip(_batch_sizes(case), places):
            x = _input(case, gen, h, w).double()
            for p, v in zip(at, _gauss_exact(x, sigma, case["rule"], METHODS).values()):
                torch.as_strided(buf, (h, w), (pitch, 1), p).copy_(v)
        return buf
    nrow, ncol = case["nrow"], case["ncol"]
    if kind == "stream":
        frames = [_input(case, gen, nrow, ncol).double() for _ in range(case["frames"])]
        each = [_gauss_exact(x, case["sigma"], case["rule"], METHODS) for x in frames]
        return {m: torch.stack([e[m] for e in each]) for m in METHODS}
    x = _input(case, gen, nrow, ncol).double()
    if kind == "pyramid":
        lobe, out = _full(_gauss_lobes(case["sigma"], case["rule"])[0], True), []
        for _ in range(case["levels"] - 1):
            x = _subsample_exact(_separable(x, lobe, lobe), "identity1x1")
            out.append(x)
        return out
    if kind == "icia":
        return _moment_exact(x, case)
    if kind == "subsample":
        return _subsample_exact(x, case["op"])
    if kind == "fir":
        return _separable(x, _full(_lobe(case["nH"]), case["nH"] & 1), _full(_lobe(case["nV"]), case["nV"] & 1))
    if kind == "taps":
        return _separable(x, [float(t) for t in _taps(case["nH"], 0.3)], [float(t) for t in _taps(case["nV"], -0.4)])
    return _gauss_exact(x, case["sigma"], case["rule"], METHODS[:case.get("methods", 6)])
