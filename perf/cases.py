"""The calls this framework is measured on: filters on single images and
volumes, the ridge filters, the batched plans, the learned surrogate
(inference and training), whole-slide reads and segmentation, each through the
public entry point that a user's program calls.

A case is a dict of plain values; ``kind`` names the path and the other entries
its sizes and options.
"""

import math
import os
import struct
import tempfile

import numpy as np
import torch

from cucim_amd import batch, surrogate, synthetic
from cucim_amd.clara import CuImage
from cucim_amd.skimage import color, filters, measure
from cucim_amd.skimage._vendored import ndimage as ndi

DATA = os.path.join(os.path.dirname(os.path.abspath(surrogate.__file__)), "data",
                    "frangi_surrogate.npz")


def listed():
    return [
        # one small image smoothed, as a tile loader or a viewer does per tile:
        # the smallest call, latency
        {"name": "gaussian-tile", "kind": "gaussian", "d0": 1, "d1": 256, "d2": 256,
         "dtype": "float32", "sigma": 2.0},
        # a light-sheet / CT stack smoothed before segmentation: uint16, odd extents
        {"name": "gaussian-stack", "kind": "gaussian", "d0": 201, "d1": 387, "d2": 413,
         "dtype": "uint16", "sigma": 1.5},
        # a long line filter over a large plane: the bandwidth headline
        {"name": "correlate1d-8192", "kind": "correlate1d", "d0": 8192, "d1": 8192, "axis": 1,
         "taps": 17, "dtype": "float32"},
        # a large colour photograph: gray, smooth, edges, as three calls
        {"name": "edges-photo", "kind": "edges", "d0": 4032, "d1": 3021, "sigma": 1.5},
        # 512 uneven colour tiles through one batched plan
        {"name": "tiles-512", "kind": "tiles", "count": 512, "lo": 256, "hi": 1024, "step": 128,
         "sigma": 1.5},
        # the retina panel of the reference's notebook: the ridge filters at
        # sigma 2 on a 1011 x 1011 image (its fourth, hessian, is frangi with
        # another gamma and the zeros set to 1)
        {"name": "ridge-panel", "kind": "ridges2d", "d0": 1011, "d1": 1011, "smin": 2, "smax": 2,
         "dtype": "float32"},
        # the headline volume: multi-scale Frangi of 256^3
        {"name": "frangi-256", "kind": "frangi", "d0": 256, "d1": 256, "d2": 256, "smin": 1,
         "smax": 5, "dtype": "float32"},
        # uneven volumes of a cohort as one captured graph
        {"name": "volumes-48", "kind": "volumes", "count": 48, "lo": 48, "hi": 192, "smax": 3},
        # the learned surrogate over one volume
        {"name": "surrogate-256", "kind": "surrogate", "d0": 256, "d1": 256, "d2": 256},
        # one training step of the surrogate: eight 64^3 patches
        {"name": "train-step", "kind": "train", "count": 8, "edge": 64},
        # one level of a slide into device memory: 256 x 256 JPEG tiles, 4:2:0
        {"name": "slide-4096", "kind": "slide", "d0": 4096, "d1": 4096, "x": 0, "y": 0,
         "w": 4096, "h": 4096, "sub": 2, "quality": 90},
        # threshold of a vesselness-like map and its connected components
        {"name": "segment-volume", "kind": "segment", "d0": 160, "d1": 256, "d2": 256,
         "dtype": "float32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gaussian", "gaussian", "correlate1d", "edges", "tiles", "ridges2d",
                       "frangi", "volumes", "surrogate", "train", "slide", "segment"])
    c = {"kind": kind}
    if kind == "gaussian":
        flat = rng.random() < 0.5
        c["d0"] = 1 if flat else _log(rng, 16, 256)
        c["d1"], c["d2"] = (_log(rng, 100, 8192 if flat else 500) for _ in range(2))
        c["dtype"] = rng.choice(["float32", "float32", "uint8", "uint16", "float64"])
        c["sigma"] = round(rng.uniform(0.7, 4.0), 2)
    elif kind == "correlate1d":
        c["d0"], c["d1"] = (_log(rng, 200, 8192) for _ in range(2))
        c["axis"] = rng.randrange(2)
        c["taps"] = rng.randrange(3, 42)
        c["dtype"] = rng.choice(["float32", "float32", "float32", "float64"])
        if c["dtype"] == "float64":
            c["d0"] = min(c["d0"], 4096)
    elif kind == "edges":
        c["d0"], c["d1"] = (_log(rng, 200, 4200) for _ in range(2))
        c["sigma"] = round(rng.uniform(0.7, 4.0), 2)
    elif kind == "tiles":
        c["count"] = _log(rng, 8, 512)
        c["lo"] = _log(rng, 100, 300)
        c["hi"] = c["lo"] + _log(rng, 50, 700)
        c["step"] = rng.choice([1, 1, 64])
        c["sigma"] = round(rng.uniform(0.8, 3.0), 2)
    elif kind == "ridges2d":
        c["d0"], c["d1"] = (_log(rng, 200, 2100) for _ in range(2))
        c["smin"] = rng.randrange(1, 4)
        c["smax"] = c["smin"] + rng.randrange(0, 3)
        c["dtype"] = rng.choice(["float32", "float32", "float64"])
    elif kind == "frangi":
        for k in ("d0", "d1", "d2"):
            c[k] = _log(rng, 40, 250)
        c["smin"] = rng.randrange(1, 3)
        c["smax"] = c["smin"] + rng.randrange(0, 4)
        c["dtype"] = rng.choice(["float32", "float32", "float32", "float32", "float64"])
    elif kind == "volumes":
        c["count"] = _log(rng, 4, 48)
        c["lo"] = rng.randrange(40, 80)
        c["hi"] = rng.randrange(90, 193)
        c["smax"] = rng.randrange(1, 4)
    elif kind == "surrogate":
        for k in ("d0", "d1", "d2"):
            c[k] = _log(rng, 40, 250)
    elif kind == "train":
        c["count"] = rng.randrange(1, 9)
        c["edge"] = rng.randrange(20, 65)
    elif kind == "slide":
        c["d0"], c["d1"] = (_log(rng, 700, 4096) for _ in range(2))
        c["x"], c["y"] = rng.randrange(0, 300), rng.randrange(0, 300)
        c["w"] = max(64, int((c["d1"] - c["x"]) * rng.uniform(0.3, 1.0)))
        c["h"] = max(64, int((c["d0"] - c["y"]) * rng.uniform(0.3, 1.0)))
        c["sub"] = rng.choice([2, 2, 0])
        c["quality"] = rng.choice([75, 90, 90, 95])
    else:
        if rng.random() < 0.5:
            c["d0"], c["d1"], c["d2"] = 1, _log(rng, 200, 3000), _log(rng, 200, 3000)
        else:
            c["d0"], c["d1"], c["d2"] = (_log(rng, 24, 200) for _ in range(3))
        c["dtype"] = rng.choice(["float32", "float32", "uint8"])
    return c


# ---------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _image(shape, dtype, seed):
    """A blocky scene with noise: 8 x 8 blocks of one level plus noise, the
    full range of the integer types, [0, 1] in the float types."""
    g = _gen(seed)
    coarse = torch.rand(tuple(-(-s // 8) for s in shape), generator=g, device="cuda")
    for d in range(len(shape)):
        coarse = coarse.repeat_interleave(8, d).narrow(d, 0, shape[d])
    x = (0.75 * coarse + 0.25 * torch.rand(shape, generator=g, device="cuda")).clamp_(0, 1)
    if dtype == "uint8":
        return (x * 255).to(torch.uint8)
    if dtype == "uint16":
        return (x * 65535).to(torch.int32).to(torch.uint16)
    return x.to(getattr(torch, dtype)).contiguous()


def _vessels2d(shape, dtype, seed):
    """Bright lines on a dim background with noise (a retina-like image)."""
    v = synthetic.tube_volume((12,) + tuple(shape), ntubes=24, seed=seed, noise=0.05)
    return v.amax(0).to(getattr(torch, dtype)).contiguous()


def _volume_shapes(case):
    # the shapes of a cohort are part of the case, its voxels of the seed
    r = np.random.default_rng(case["count"] * 1000003 + case["lo"] * 1009 + case["hi"])
    return [tuple(int(v) for v in r.integers(case["lo"], case["hi"] + 1, 3))
            for _ in range(case["count"])]


def _tile_edges(case):
    r = np.random.default_rng(case["count"] * 7919 + case["lo"] * 31 + case["hi"])
    e = np.arange(case["lo"], case["hi"] + 1, case["step"])
    return [int(v) for v in r.choice(e, case["count"])]


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k == "gaussian":
        shape = (case["d1"], case["d2"]) if case["d0"] == 1 else (case["d0"], case["d1"],
                                                                    case["d2"])
        s["x"] = _image(shape, case["dtype"], seed)
    elif k == "correlate1d":
        s["x"] = _image((case["d0"], case["d1"]), case["dtype"], seed)
        n = case["taps"]
        t = np.hanning(n + 2)[1:-1]
        s["w"] = t / t.sum()
    elif k == "edges":
        s["x"] = torch.stack([_image((case["d0"], case["d1"]), "uint8", 3 * seed + i)
                              for i in range(3)], -1).contiguous()
    elif k == "tiles":
        g = _gen(seed)
        ins, offs, edges = [], [0], _tile_edges(case)
        for e in edges:
            c = -(-e // 8)
            up = torch.rand((c, c, 3), generator=g, device="cuda") * 255
            up = up.repeat_interleave(8, 0).repeat_interleave(8, 1)[:e, :e]
            fine = torch.rand((e, e, 3), generator=g, device="cuda") * 32 - 16
            ins.append((up + fine).clamp(0, 255).to(torch.uint8).contiguous())
            offs.append(offs[-1] + -(-e * e // 64) * 64)
        s["flat"] = torch.zeros(offs[-1], device="cuda")
        outs = [s["flat"][o:o + e * e].view(e, e) for o, e in zip(offs, edges)]
        s["plan"] = batch.GrayGaussSobelBatch(ins, outs, sigma=case["sigma"])
    elif k == "ridges2d":
        s["x"] = _vessels2d((case["d0"], case["d1"]), case["dtype"], seed)
        s["sigmas"] = list(range(case["smin"], case["smax"] + 1))
    elif k == "frangi":
        s["x"] = synthetic.tube_volume((case["d0"], case["d1"], case["d2"]), ntubes=24,
                                       seed=seed).to(getattr(torch, case["dtype"]))
        s["sigmas"] = list(range(case["smin"], case["smax"] + 1))
    elif k == "volumes":
        vols = [synthetic.tube_volume(sh, ntubes=3, seed=seed * 64 + i, noise=0.08)
                for i, sh in enumerate(_volume_shapes(case))]
        s["plan"] = batch.FrangiBatch3D(vols, sigmas=range(1, case["smax"] + 1))
        s["graph"] = s["plan"].capture()
    elif k == "surrogate":
        s["x"] = synthetic.tube_volume((case["d0"], case["d1"], case["d2"]), ntubes=24, seed=seed)
        s["model"] = surrogate.FrangiSurrogate.load(DATA)
    elif k == "train":
        e, h = case["edge"], surrogate.HALO
        s["model"] = surrogate.FrangiSurrogate(seed=seed)
        s["xs"], s["ts"] = [], []
        for i in range(case["count"]):
            v = synthetic.tube_volume((e,) * 3, ntubes=4, seed=seed * 16 + i, noise=0)
            g = _gen(seed * 16 + i)
            n = 0.05 * torch.randn(v.shape, generator=g, device="cuda")
            s["xs"].append((v + n).to(torch.bfloat16).view(e, e, e, 1).contiguous())
            s["ts"].append((0.6 * v * v)[h:-h, h:-h, h:-h].contiguous())
    elif k == "slide":
        s["dir"] = tempfile.TemporaryDirectory()
        path = os.path.join(s["dir"].name, "slide.tif")
        with open(path, "wb") as f:
            f.write(_slide(case, seed))
        s["image"] = CuImage(path)
    else:
        shape = (case["d0"], case["d1"], case["d2"])
        v = synthetic.tube_volume(shape if shape[0] > 1 else (8,) + shape[1:], ntubes=16,
                                  seed=seed, noise=0.12)
        v = (v if shape[0] > 1 else v[4]).clamp(0, 1).contiguous()
        s["x"] = (v * 255).to(torch.uint8) if case["dtype"] == "uint8" else v
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "gaussian":
        return filters.gaussian(s["x"], sigma=c["sigma"])
    if k == "correlate1d":
        return ndi.correlate1d(s["x"], s["w"], axis=c["axis"], mode="reflect")
    if k == "edges":
        gray = color.rgb2gray(s["x"])
        smooth = filters.gaussian(gray, sigma=c["sigma"])
        return gray, smooth, filters.sobel(smooth)
    if k == "tiles":
        s["plan"].run()
        return s["flat"]
    if k == "ridges2d":
        return [f(s["x"], sigmas=s["sigmas"], black_ridges=False)
                for f in (filters.meijering, filters.sato, filters.frangi)]
    if k == "frangi":
        return filters.frangi(s["x"], sigmas=s["sigmas"], black_ridges=False)
    if k == "volumes":
        s["graph"].replay()
        return s["plan"].outputs
    if k == "surrogate":
        return s["model"](s["x"])
    if k == "train":
        loss = s["model"].train_step(s["xs"], s["ts"], lr=1e-3)
        return {"loss": loss, "w": s["model"].w, "b": s["model"].b}
    if k == "slide":
        return s["image"].read_region((c["x"], c["y"]), (c["w"], c["h"]), 0, device="cuda",
                                      num_workers=8)
    t = filters.threshold_otsu(s["x"])
    return t, measure.label(s["x"] > t)


# ------------------------------------------------------------ work, errors --
_SIZE = {"uint8": 1, "uint16": 2, "float32": 4, "float64": 8}


def _radii(sigmas):
    return [int((8 if s > 1 else 100) * s / math.sqrt(2) + 0.5) for s in sigmas]


def _hessian_taps(s):
    """Taps of the order-0 kernel that are not zero in 32 bits (those past
    about 14 standard deviations are)."""
    return 2 * min(_radii([s])[0], int(14.4 * s / math.sqrt(2))) + 1


def work(case):
    k = case["kind"]
    if k == "gaussian":
        n = case["d0"] * case["d1"] * case["d2"]
        ndim = 2 if case["d0"] == 1 else 3
        out = 8 if case["dtype"] == "float64" else 4
        return {"bytes": n * (_SIZE[case["dtype"]] + out),
                "flops": 2.0 * n * ndim * (2 * int(4 * case["sigma"] + 0.5) + 1)}
    if k == "correlate1d":
        n = case["d0"] * case["d1"]
        return {"bytes": 2 * n * _SIZE[case["dtype"]], "flops": 2.0 * n * case["taps"]}
    if k == "edges":
        n = case["d0"] * case["d1"]
        return {"bytes": n * (3 + 4 + 4 + 4),
                "flops": n * (5 + 4.0 * (2 * int(4 * case["sigma"] + 0.5) + 1) + 20)}
    if k == "tiles":
        n = sum(e * e for e in _tile_edges(case))
        return {"bytes": 7 * n,
                "flops": n * (5 + 4.0 * (2 * int(4 * case["sigma"] + 0.5) + 1) + 20)}
    if k in ("ridges2d", "frangi"):
        n = case["d0"] * case["d1"] * case.get("d2", 1)
        nf = 3 if k == "ridges2d" else 1
        per = 7 if k == "ridges2d" else 27  # 1-D sweeps that the Hessian needs per sigma
        taps = sum(_hessian_taps(s) for s in range(case["smin"], case["smax"] + 1))
        return {"bytes": n * (1 + nf) * _SIZE[case["dtype"]], "flops": 2.0 * n * per * taps * nf}
    if k == "volumes":
        n = sum(a * b * c for a, b, c in _volume_shapes(case))
        taps = sum(_hessian_taps(s) for s in range(1, case["smax"] + 1))
        return {"bytes": 8 * n, "flops": 2.0 * n * 27 * taps}
    if k == "surrogate":
        n = case["d0"] * case["d1"] * case["d2"]
        return {"bytes": 8 * n, "flops": float(n) * _NET_FLOPS}
    if k == "train":
        e, n = case["edge"], case["count"]
        fl = sum(54.0 * ci * co * (e - 2 * (i + 1)) ** 3
                 for i, (ci, co, _) in enumerate(surrogate.LAYERS))
        # forward, weight gradients, input gradients of all layers but the first
        return {"bytes": n * (2 * e ** 3 + 4 * (e - 10) ** 3) + 32 * 48049,
                "flops": n * (3 * fl - 54.0 * 24 * (e - 2) ** 3)}
    if k == "slide":
        return {"bytes": case["w"] * case["h"] * (3 + 0.3), "flops": 0}
    n = case["d0"] * case["d1"] * case["d2"]
    return {"bytes": n * (_SIZE[case["dtype"]] + 4), "flops": 0}


_NET_FLOPS = sum(54 * ci * co for ci, co, _ in surrogate.LAYERS)


def tolerance(case):
    """Four times the largest relative error seen against 64 bits over the
    listed and drawn cases of the kind (or, where the call computes integers
    or bytes, equality).  Single voxels of the ridge filters move by more: the
    vesselness jumps where two eigenvalues of opposite sign swap their order
    by magnitude; so does a weight whose gradient is near zero, as Adam's
    first steps follow the gradient's sign."""
    k = case["kind"]
    if k in ("slide", "segment"):
        return "exact"
    ridge = k in ("frangi", "ridges2d")
    if case.get("dtype") == "float64":
        return {"rel": 1e-6, "max": 0.99} if ridge else {"rel": 1e-12}
    t = {"rel": {"gaussian": 5e-7, "correlate1d": 3e-7, "edges": 2e-6, "tiles": 2e-6,
                 "ridges2d": 4e-4, "frangi": 6e-4, "volumes": 6e-4, "surrogate": 2e-2,
                 "train": 6e-3}[k]}
    return dict(t, max=0.99) if ridge or k in ("volumes", "train") else t


# --------------------------------------------------- the results in 64 bits --
def _index(n, r, mode):
    i = np.arange(-r, n + r)
    if mode == "nearest":
        i = np.clip(i, 0, n - 1)
    else:  # reflect: d c b a | a b c d | d c b a
        i = np.mod(i, 2 * n)
        i = np.where(i >= n, 2 * n - 1 - i, i)
    return torch.from_numpy(i)


def _corr(x, w, axis, mode, anchor=None):
    """sum_t w[t] x[i + t - anchor] along an axis, the ends extended."""
    n, r = x.shape[axis], len(w)
    a = r // 2 if anchor is None else anchor
    xe = x.index_select(axis, _index(n, r, mode).to(x.device))
    out = torch.zeros_like(x)
    for t, v in enumerate(w):
        if v != 0:
            out.add_(xe.narrow(axis, r + t - a, n), alpha=float(v))
    return out


def _gauss(sigma, order, radius):
    t = np.arange(-radius, radius + 1, dtype=np.float64)
    g = np.exp(-0.5 * (t / sigma) ** 2)
    g /= g.sum()
    # a correlation kernel: the derivative's sign is that of the flipped one
    return g if order == 0 else g * t / sigma ** 2


def _smooth(x, sigma, mode="nearest"):
    w = _gauss(sigma, 0, int(4 * sigma + 0.5))
    for d in range(x.dim()):
        x = _corr(x, w, d, mode)
    return x


def _sobel(x):
    e, s = np.array([-1.0, 0, 1]) / 2, np.array([1.0, 2, 1]) / 4
    a = _corr(_corr(x, e, 0, "reflect"), s, 1, "reflect")
    b = _corr(_corr(x, s, 0, "reflect"), e, 1, "reflect")
    return torch.sqrt((a * a + b * b) * 2)  # edge weights are 1, 0, -1 over sqrt(2)


def _gray(x):
    return (x.double() / 255) @ torch.tensor([0.2125, 0.7154, 0.0721], dtype=torch.float64,
                                             device=x.device)


def _eigenvalues(x, sigma):
    """Eigenvalues of the Hessian by Gaussian derivatives, ascending."""
    nd, sq = x.dim(), sigma / math.sqrt(2)
    r = _radii([sigma])[0]
    w = [_gauss(sq, o, r) for o in (0, 1)]
    grad = []
    for a in range(nd):
        y = x
        for d in range(nd):
            y = _corr(y, w[int(d == a)], d, "reflect")
        grad.append(y)
    h = {}
    for a in range(nd):
        for b in range(a, nd):
            y = grad[a]
            for d in range(nd):
                y = _corr(y, w[int(d == b)], d, "reflect")
            h[a, b] = y
    if nd == 2:
        m, q = (h[0, 0] + h[1, 1]) / 2, (h[0, 0] - h[1, 1]) / 2
        s = torch.sqrt(q * q + h[0, 1] ** 2)
        return [m - s, m + s]
    q = (h[0, 0] + h[1, 1] + h[2, 2]) / 3
    a, b, c = h[0, 0] - q, h[1, 1] - q, h[2, 2] - q
    d, e, f = h[0, 1], h[0, 2], h[1, 2]
    p = torch.sqrt((a * a + b * b + c * c + 2 * (d * d + e * e + f * f)) / 6)
    det = a * (b * c - f * f) - d * (d * c - f * e) + e * (d * f - b * e)
    phi = torch.acos((det / (2 * p ** 3)).nan_to_num(1.0).clamp(-1, 1)) / 3
    hi = q + 2 * p * torch.cos(phi)
    lo = q + 2 * p * torch.cos(phi + 2 * math.pi / 3)
    return [lo, 3 * q - hi - lo, hi]


def _by_size(ev):
    v = torch.stack(ev)
    return list(v.gather(0, v.abs().argsort(dim=0, stable=True)))


def _frangi(x, sigmas, alpha=0.5, beta=0.5):
    """Of the negated image (bright ridges)."""
    out = g2 = None
    for s in sigmas:
        ev = _by_size(_eigenvalues(-x, s))
        rg = sum(e * e for e in ev)
        if g2 is None:
            g2 = max(float(rg.max()) / 2, 1e-10) if float(rg.max()) else 2.0
        v = -torch.expm1(-rg / g2)
        l2 = ev[1].clamp_min(1e-10)
        if len(ev) == 2:
            v = v * torch.exp(-(ev[0] / l2) ** 2 / (2 * beta ** 2))
        else:
            l3 = ev[2].clamp_min(1e-10)
            v = v * torch.exp(-ev[0] ** 2 / (l2 * l3) / (2 * beta ** 2))
            v = v * -torch.expm1(-(l2 / l3) ** 2 / (2 * alpha ** 2))
        out = v if out is None else torch.maximum(out, v)
    return out


def _sato(x, sigmas):
    out = torch.zeros_like(x)
    for s in sigmas:
        ev = torch.stack(_eigenvalues(-x, s)[1:]).clamp_min(0)
        out = torch.maximum(out, s * s * ev.prod(0) ** (1 / len(ev)))
    return out


def _meijering(x, sigmas):
    out, al = torch.zeros_like(x), 1 / (x.dim() + 1)
    for s in sigmas:
        ev = _eigenvalues(-x, s)
        v = torch.stack([e + al * sum(o for o in ev if o is not e) for e in ev])
        v = v.gather(0, v.abs().argmax(0, keepdim=True))[0].clamp_min(0)
        out = torch.maximum(out, v / v.max() if float(v.max()) > 0 else v)
    return out


def _conv(x, w, b):
    """Valid 3 x 3 x 3 convolution, channels last; w: (27, ci, co)."""
    d, h, wd = (s - 2 for s in x.shape[:3])
    y = b.expand(d * h * wd, -1)
    for t in range(27):
        z, u, v = t // 9, t // 3 % 3, t % 3
        y = y + x[z:z + d, u:u + h, v:v + wd].reshape(d * h * wd, -1) @ w[t]
    return y.view(d, h, wd, -1)


def _gelu(x):
    return x * torch.sigmoid(2 * math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3))


def _net(x, ws, bs):
    for i, (w, b) in enumerate(zip(ws, bs)):
        x = _conv(x, w, b)
        if i < len(ws) - 1:
            x = _gelu(x)
    return x[..., 0]


def exact(case, seed):
    k = case["kind"]
    if k == "slide":
        return None  # bytes
    s = prepare(dict(case, count=1) if k == "volumes" else case, seed)
    if k == "gaussian":
        top = {"uint8": 255.0, "uint16": 65535.0}.get(case["dtype"], 1.0)
        return _smooth(s["x"].double() / top, case["sigma"])
    if k == "correlate1d":
        return _corr(s["x"].double(), s["w"], case["axis"], "reflect")
    if k == "edges":
        g = _gray(s["x"])
        m = _smooth(g, case["sigma"])
        return g, m, _sobel(m)
    if k == "tiles":
        out = torch.zeros(s["flat"].numel(), dtype=torch.float64, device="cuda")
        for x, o in zip(s["plan"].inputs, s["plan"].outputs):
            y = _sobel(_smooth(_gray(x), case["sigma"]))
            out.narrow(0, o.storage_offset(), o.numel()).copy_(y.reshape(-1))
        return out
    if k == "ridges2d":
        x = s["x"].double()
        return [_meijering(x, s["sigmas"]), _sato(x, s["sigmas"]), _frangi(x, s["sigmas"])]
    if k == "frangi":
        return _frangi(s["x"].double(), s["sigmas"])
    if k == "volumes":
        vols = [synthetic.tube_volume(sh, ntubes=3, seed=seed * 64 + i, noise=0.08)
                for i, sh in enumerate(_volume_shapes(case))]
        return [_frangi(v.double(), range(1, case["smax"] + 1)) if i < 6 else None
                for i, v in enumerate(vols)]
    if k == "surrogate":
        m, h = s["model"], surrogate.HALO
        x = s["x"].double()
        for d in range(3):
            x = x.index_select(d, _index(x.shape[d], h, "reflect").to(x.device))
        y = _net(x[..., None], [w.double() for w in m.w], [b.double() for b in m.b])
        return y.clamp(0, 1)
    if k == "train":
        m = s["model"]
        p = [t.double().requires_grad_() for t in m.w + m.b]
        n, total = len(m.w), 0.0
        for x, t in zip(s["xs"], s["ts"]):
            loss = ((_net(x.double(), p[:n], p[n:]) - t.double()) ** 2).mean() / case["count"]
            loss.backward()
            total += float(loss.detach())
        # the first Adam step: both moments divided by their bias are g and g^2
        new = [(t - 1e-3 * t.grad / (t.grad.abs() + 1e-8)).detach() for t in p]
        return {"loss": torch.tensor([total], dtype=torch.float64), "w": new[:n], "b": new[n:]}
    x = s["x"].cpu().numpy()
    lo, hi = x.min(), x.max()
    if case["dtype"] == "uint8":
        cnt, mid = np.bincount(x.ravel() - lo).astype(np.float64), np.arange(lo, hi + 1.0)
    else:
        cnt, e = np.histogram(x.astype(np.float64), 256, (float(lo), float(hi)))
        mid = (e[1:] + e[:-1]) / 2
    w1, m1 = np.cumsum(cnt), np.cumsum(cnt * mid)
    with np.errstate(divide="ignore", invalid="ignore"):
        var = w1 * (w1[-1] - w1) * (m1 / w1 - (m1[-1] - m1) / (w1[-1] - w1)) ** 2
    return np.float64(mid[np.nanargmax(var[:-1])]), None


# ------------------------------------------------------- a slide in a file --
# Baseline JPEG tiles with the tables of ITU-T T.81 annex K, in a tiled TIFF.
_ZIGZAG = [int(v) for v in np.argsort([
    (i + j) * 64 + (j if (i + j) % 2 == 0 else i) for i in range(8) for j in range(8)])]
_QY = ("16 11 10 16 24 40 51 61 12 12 14 19 26 58 60 55 14 13 16 24 40 57 69 56 14 17 22 29 51 "
       "87 80 62 18 22 37 56 68 109 103 77 24 35 55 64 81 104 113 92 49 64 78 87 103 121 120 101 "
       "72 92 95 98 112 100 103 99")
_QC = ("17 18 24 47 99 99 99 99 18 21 26 66 99 99 99 99 24 26 56 99 99 99 99 99 47 66 99 99 99 99 "
       "99 99 " + "99 " * 32)
_DC = [("00010501010101010100000000000000", "000102030405060708090a0b"),
       ("00030101010101010101010000000000", "000102030405060708090a0b")]
_AC = [("0002010303020403050504040000017d",
        "01020300041105122131410613516107227114328191a1082342b1c11552d1f02433627282090a161718191a25"
        "262728292a3435363738393a434445464748494a535455565758595a636465666768696a737475767778797a83"
        "8485868788898a92939495969798999aa2a3a4a5a6a7a8a9aab2b3b4b5b6b7b8b9bac2c3c4c5c6c7c8c9cad2d3"
        "d4d5d6d7d8d9dae1e2e3e4e5e6e7e8e9eaf1f2f3f4f5f6f7f8f9fa"),
       ("00020102040403040705040400010277",
        "000102031104052131061241510761711322328108144291a1b1c109233352f0156272d10a162434e125f11718"
        "191a262728292a35363738393a434445464748494a535455565758595a636465666768696a737475767778797a"
        "82838485868788898a92939495969798999aa2a3a4a5a6a7a8a9aab2b3b4b5b6b7b8b9bac2c3c4c5c6c7c8c9ca"
        "d2d3d4d5d6d7d8d9dae2e3e4e5e6e7e8e9eaf2f3f4f5f6f7f8f9fa")]


def _codes(bits, vals):
    """(code, length) of every symbol of a canonical Huffman table."""
    code, table, at = 0, np.zeros((256, 2), np.int64), 0
    vals = bytes.fromhex(vals)
    for i, n in enumerate(bytes.fromhex(bits)):
        for _ in range(n):
            table[vals[at]] = code, i + 1
            code, at = code + 1, at + 1
        code <<= 1
    return table


def _segment(marker, payload):
    return struct.pack(">BBH", 255, marker, len(payload) + 2) + payload


def _scene(h, w, seed):
    """Smooth tissue-like colour with sensor noise."""
    g = _gen(seed)
    r = np.random.default_rng(seed)
    y = torch.arange(h, device="cuda", dtype=torch.float32)[:, None]
    x = torch.arange(w, device="cuda", dtype=torch.float32)[None, :]
    px = []
    for _ in range(3):
        a = torch.zeros((h, w), device="cuda")
        for _ in range(6):
            fy, fx, ph = r.uniform(0.01, 0.08), r.uniform(0.01, 0.08), r.uniform(0, 6.3)
            a += torch.sin(y * fy + x * fx + ph)
        px.append(a * 17 + 120 + 6 * torch.randn((h, w), generator=g, device="cuda"))
    return torch.stack(px).clamp(0, 255).floor()


def _blocks(plane, q, tile, dct):
    """Quantised zigzag coefficients: (tiles, rows, columns, 64) of 8 x 8
    blocks, the tiles in raster order."""
    h, w = plane.shape
    ny, nx, n = h // tile, w // tile, tile // 8
    b = (plane - 128).view(ny, n, 8, nx, n, 8)
    b = b.permute(0, 3, 1, 4, 2, 5).reshape(-1, 8, 8)
    c = torch.round((dct @ b @ dct.T).reshape(-1, 64) / q)
    return c[:, _ZIGZAG].to(torch.int64).view(ny * nx, n, n, 64)


def _bits(v):
    return torch.where(v == 0, 0, torch.floor(torch.log2(v.abs().double().clamp_min(1))).long() + 1)


def _slide(case, seed, tile=256):
    h, w, f = case["d0"], case["d1"], 2 if case["sub"] else 1
    hp, wp = -(-h // tile) * tile, -(-w // tile) * tile
    px = _scene(hp, wp, seed)
    dev = px.device
    m = torch.tensor([[0.299, 0.587, 0.114], [-0.168736, -0.331264, 0.5],
                      [0.5, -0.418688, -0.081312]], device=dev)
    ycc = torch.einsum("ij,jhw->ihw", m, px)
    ycc[1:] += 128
    k = torch.arange(8, device=dev, dtype=torch.float32)
    dct = torch.cos((2 * k[None, :] + 1) * k[:, None] * math.pi / 16) / 2
    dct[0] /= math.sqrt(2)
    s = 5000 // case["quality"] if case["quality"] < 50 else 200 - 2 * case["quality"]
    qt = [np.clip((np.array(t.split(), np.int64) * s + 50) // 100, 1, 255) for t in (_QY, _QC)]
    ql = [torch.from_numpy(t).to(dev).float() for t in qt]
    y = _blocks(ycc[0], ql[0], tile, dct)
    nt, nb = y.shape[0], tile // 8 // f
    chroma = [torch.nn.functional.avg_pool2d(c[None, None], f)[0, 0] if f > 1 else c
              for c in ycc[1:]]
    chroma = [_blocks(c, ql[1], tile // f, dct) for c in chroma]
    # minimum coded units: f x f luma blocks, then one of each colour
    y = y.view(nt, nb, f, nb, f, 64).permute(0, 1, 3, 2, 4, 5).reshape(nt, nb * nb, f * f, 64)
    co = torch.cat([y] + [c.reshape(nt, nb * nb, 1, 64) for c in chroma], 2)
    u = f * f + 2
    # differences of the DC values within each tile and component
    for lo, hi in ((0, f * f), (f * f, f * f + 1), (f * f + 1, u)):
        dc = co[:, :, lo:hi, 0].reshape(nt, -1)
        co[:, :, lo:hi, 0] = torch.diff(dc, dim=1, prepend=dc[:, :1] * 0).view(nt, -1, hi - lo)
    co = co.reshape(-1, 64)
    comp = (torch.arange(u, device=dev) >= f * f).long().repeat(nt * nb * nb)
    dct_, act = (torch.from_numpy(np.stack([_codes(*t) for t in tb])).to(dev)
                 for tb in (_DC, _AC))
    size = _bits(co)
    extra = torch.where(co < 0, co + (1 << size) - 1, co)
    # zero run before each coefficient that is not zero
    pos = torch.arange(64, device=dev).expand_as(co)
    nz = torch.where((co != 0) | (pos == 0), pos, 0)
    before = torch.cummax(nz, 1).values
    run = pos - torch.cat([before[:, :1], before[:, :-1]], 1) - 1
    ac = act[comp[:, None], ((run.clamp_min(0) % 16) << 4) + size]
    zrl, eob = act[comp, 0xF0], act[comp, 0]
    val, num = (ac[..., 0] << size) + extra, ac[..., 1] + size
    for n in (3, 2, 1):  # runs of 16 zeros before the symbol
        many = run // 16 >= n
        val += torch.where(many, zrl[:, None, 0] << num, 0)
        num += torch.where(many, zrl[:, None, 1].expand_as(num), 0)
    keep = co != 0
    d = dct_[comp, size[:, 0]]
    val[:, 0], num[:, 0], keep[:, 0] = (d[:, 0] << size[:, 0]) + extra[:, 0], \
        d[:, 1] + size[:, 0], True
    end = (before[:, -1] < 63).long()
    val = torch.cat([torch.where(keep, val, 0), (eob[:, 0] * end)[:, None]], 1).view(nt, -1)
    num = torch.cat([torch.where(keep, num, 0), (eob[:, 1] * end)[:, None]], 1).view(nt, -1)
    length = num.sum(1)
    head = _segment(0xC0, struct.pack(">BHHB", 8, tile, tile, 3)
                    + bytes([1, 16 * f + f, 0, 2, 17, 1, 3, 17, 1])) \
        + _segment(0xDA, bytes([3, 1, 0, 2, 17, 3, 17, 0, 63, 0]))
    blobs = []
    for t in range(0, nt, 64):  # some tiles at a time: the bits take 8 bytes each
        v, n, ln = val[t:t + 64], num[t:t + 64], length[t:t + 64]
        nbyte = (ln + 7) // 8
        start = torch.cumsum(nbyte, 0) - nbyte
        at = (torch.cumsum(n, 1) - n + 8 * start[:, None]).reshape(-1)
        v, n = v.reshape(-1), n.reshape(-1)
        use = n > 0
        v, n, at = v[use], n[use], at[use]
        which = torch.repeat_interleave(torch.arange(n.numel(), device=dev), n)
        off = torch.arange(which.numel(), device=dev) - (torch.cumsum(n, 0) - n)[which]
        bit = torch.ones(8 * int(nbyte.sum()), dtype=torch.uint8, device=dev)
        bit[at[which] + off] = ((v[which] >> (n[which] - 1 - off)) & 1).to(torch.uint8)
        by = (bit.view(-1, 8) << torch.arange(7, -1, -1, dtype=torch.uint8, device=dev)).sum(
            1, dtype=torch.int64).to(torch.uint8).cpu().numpy().tobytes()
        for o, c in zip(start.tolist(), nbyte.tolist()):
            blobs.append(b"\xff\xd8" + head + by[o:o + c].replace(b"\xff", b"\xff\x00")
                         + b"\xff\xd9")
    tables = b"\xff\xd8" + b"".join(
        _segment(0xDB, bytes([i]) + bytes(int(q) for q in qt[i][_ZIGZAG])) for i in range(2))
    for cls, tb in ((0, _DC), (16, _AC)):
        for i, (bits, vals) in enumerate(tb):
            tables += _segment(0xC4, bytes([cls + i]) + bytes.fromhex(bits) + bytes.fromhex(vals))
    return _tiff(w, h, tile, f, blobs, tables + b"\xff\xd9")


def _tiff(w, h, tile, f, blobs, tables):
    """One level of JPEG tiles as a classic little-endian TIFF."""
    offs, at = [], 8
    for b in blobs:
        offs.append(at)
        at += len(b) + len(b) % 2
    tags = {256: (4, [w]), 257: (4, [h]), 258: (3, [8, 8, 8]), 259: (3, [7]), 262: (3, [6]),
            277: (3, [3]), 284: (3, [1]), 322: (3, [tile]), 323: (3, [tile]), 324: (4, offs),
            325: (4, [len(b) for b in blobs]), 347: (7, tables), 530: (3, [f, f])}
    ifd, extra = struct.pack("<H", len(tags)), b""
    base = at + 2 + 12 * len(tags) + 4
    for tag, (typ, v) in sorted(tags.items()):
        raw = v if typ == 7 else struct.pack("<%d%s" % (len(v), "HI"[typ == 4]), *v)
        ifd += struct.pack("<HHI", tag, typ, len(v))
        if len(raw) <= 4:
            ifd += raw.ljust(4, b"\0")
        else:
            ifd += struct.pack("<I", base + len(extra))
            extra += raw + b"\0" * (len(raw) % 2)
    body = b"".join(b + b"\0" * (len(b) % 2) for b in blobs)
    return struct.pack("<2sHI", b"II", 42, at) + body + ifd + b"\0\0\0\0" + extra
