"""Performance cases: the work that users of iqhip have it do, through its
public entry points, from one tile-sized problem to the largest configuration.

A case is a dict of plain values; extents are texts such as "100x100x50".
  kind "plan"          a plan held by the program; a pass is one simulation of
                       every realization and the download of grids and picks
  kind "call"          one iqsim call on host arrays, plan creation included
  kind "fastdistance"  one fastdistance call on host arrays
  kind "graphcut"      one graphcut call on host arrays
Training images: grf32 / grf64 (continuous, Float32 / Float64), binary64
(a thresholded field in Float64), facies8 (three facies in UInt8).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "imagequilting.jl_amd"))

import iqhip  # noqa: E402
from iqhip import prep, synth  # noqa: E402


def _ext(text):
    return tuple(int(v) for v in text.split("x"))


def _txt(ext):
    return "x".join(str(int(v)) for v in ext)


def _sim(name, kind, data, ti, tile, grid, overlap, tol=0.1, path="raster", nreal=1, grids=1, soft=0, hard=0,
         learned=False):
    return {"name": name, "kind": kind, "data": data, "ti": ti, "tile": tile, "grid": grid, "overlap": overlap,
            "tol": tol, "path": path, "nreal": nreal, "grids": grids, "soft": soft, "hard": hard, "learned": learned}


def listed():
    return [
        # a first try on a small picture: every launch is tiny, latency is all
        _sim("sim2d_f32_small", "plan", "grf32", "48x40", "12x12", "60x60", 0.25),
        # the usual script: one call on a binary 2-D image, nothing kept
        _sim("call2d_binary64", "call", "binary64", "200x200", "30x30", "400x400", 1 / 6),
        # Float64 is what arrays hold by default; random path, odd extents
        _sim("sim2d_f64_random", "plan", "grf64", "201x187", "31x27", "300x311", 0.2, path="random", nreal=2),
        # an ordinary 3-D Float32 realization
        _sim("sim3d_f32", "plan", "grf32", "100x100x50", "20x20x5", "200x200x50", 0.2),
        # the same kind of work in Float64, at a smaller size
        _sim("sim3d_f64", "plan", "grf64", "80x80x40", "16x16x5", "120x120x40", 0.25),
        # an ensemble of categorical models on grids of different sizes
        _sim("batch3d_facies8", "plan", "facies8", "150x150x30", "24x24x6", "100x300x30", 0.25, grids=16),
        # conditioning on a soft variable and wells, a small ensemble
        _sim("sim2d_soft_hard", "plan", "grf32", "512x512", "48x48", "1024x1024", 1 / 6, tol=0.05, nreal=4, soft=1,
             hard=500),
        # conditioning on point data alone: most tiles hold none, the path starts from the data
        _sim("sim2d_hard", "plan", "grf32", "256x256", "32x32", "500x500", 0.25, nreal=2, hard=60),
        # the largest training image, every candidate scanned
        _sim("sim3d_large_scan", "plan", "grf32", "256x256x64", "32x32x8", "384x384x64", 0.25, nreal=2),
        # the same with the learned shortlist, an ensemble in lockstep
        _sim("sim3d_large_learned", "plan", "grf32", "256x256x64", "32x32x8", "384x384x64", 0.25, nreal=8,
             learned=True),
        # single functions swapped into a host program: a distance map ...
        {"name": "fastdistance3d_f32", "kind": "fastdistance", "data": "grf32", "ti": "100x100x50",
         "tile": "20x20x5", "overlap": 0.2},
        # ... and a boundary cut
        {"name": "graphcut3d_f32", "kind": "graphcut", "data": "grf32", "slab": "8x32x8", "dim": 0},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["small", "plane", "plane", "volume", "volume", "facies", "soft", "hard", "large", "call",
                         "fastdistance", "graphcut"])
    data = rng.choice(["grf32", "grf64"])
    path = rng.choice(["raster", "raster", "random", "dilation"])
    tol = rng.choice([0.05, 0.1, 0.1, 0.2])
    overlap = rng.choice([1 / 6, 0.2, 0.25, 1 / 3])
    if family == "small":
        t = [rng.randint(8, 16) for _ in range(2)]
        return _sim("", "plan", rng.choice(["grf32", "grf64", "binary64"]), _txt([rng.randint(3 * v, 6 * v) for v in t]),
                    _txt(t), _txt([rng.randint(4 * v, 6 * v) for v in t]), overlap, tol, path)
    if family in ("plane", "call"):
        t = [rng.randint(18, 40) for _ in range(2)]
        return _sim("", "call" if family == "call" else "plan", rng.choice([data, "binary64"]),
                    _txt([_logint(rng, 5 * v, 12 * v) for v in t]), _txt(t),
                    _txt([_logint(rng, 6 * v, 14 * v) for v in t]), overlap, tol, path, nreal=rng.choice([1, 1, 2, 4]))
    if family == "volume":
        t = [rng.randint(14, 22), rng.randint(14, 22), rng.randint(4, 7)]
        big = data == "grf32"
        return _sim("", "plan", data, _txt([_logint(rng, 4 * v, (6 if big else 5) * v) for v in t]), _txt(t),
                    _txt([_logint(rng, 5 * v, (9 if big else 6) * v) for v in t]), overlap, tol, path)
    if family == "facies":
        t = [rng.randint(18, 26), rng.randint(18, 26), 6]
        return _sim("", "plan", "facies8", _txt([rng.randint(110, 150), rng.randint(110, 150), 30]), _txt(t),
                    _txt([100, rng.randint(150, 300), 30]), 0.25, 0.1, "raster", grids=rng.choice([2, 4, 8]))
    if family in ("soft", "hard"):
        t = [rng.randint(24, 48) for _ in range(2)]
        return _sim("", "plan", "grf32" if family == "soft" else data, _txt([rng.randint(5 * v, 8 * v) for v in t]),
                    _txt(t), _txt([rng.randint(6 * v, 12 * v) for v in t]), overlap, tol, "raster",
                    nreal=rng.choice([1, 2, 4]), soft=1 if family == "soft" else 0, hard=_logint(rng, 10, 200))
    if family == "large":
        return _sim("", "plan", "grf32", _txt([rng.randint(120, 200), rng.randint(120, 200), rng.randint(40, 60)]),
                    "32x32x8", _txt([rng.randint(150, 300), rng.randint(150, 300), rng.randint(40, 64)]), 0.25, 0.1,
                    "raster", nreal=rng.choice([1, 2, 4]), learned=rng.random() < 0.5)
    if family == "fastdistance":
        t = [rng.randint(8, 24), rng.randint(8, 24), rng.randint(1, 6)]
        return {"name": "", "kind": "fastdistance", "data": data,
                "ti": _txt([_logint(rng, 3 * v, 6 * v) for v in t[:2]] + [_logint(rng, t[2], 8 * t[2])]),
                "tile": _txt(t), "overlap": overlap}
    s = [_logint(rng, 4, 32), _logint(rng, 4, 32), _logint(rng, 1, 8)]
    dim = rng.randint(0, 1)
    s[dim] = rng.randint(3, 9)
    return {"name": "", "kind": "graphcut", "data": data, "slab": _txt(s), "dim": dim}


def _field(shape, ranges, gen, dtype):
    """Gaussian random field of exponential covariance exp(-3 |h / range|), periodic, mean 0, variance 1."""
    h2 = 0.0
    for d, (n, r) in enumerate(zip(shape, ranges)):
        a = torch.minimum(torch.arange(n), n - torch.arange(n)).to(torch.float64) / float(r)
        h2 = h2 + (a ** 2).reshape([-1 if e == d else 1 for e in range(len(shape))])
    lam = torch.fft.rfftn(torch.exp(-3.0 * torch.sqrt(h2))).real.clamp_(min=0.0)
    z = torch.fft.rfftn(torch.randn(shape, generator=gen, dtype=torch.float64))
    x = torch.fft.irfftn(z * torch.sqrt(lam), s=shape)
    x = (x - x.mean()) / x.std()
    return x.numpy().astype(dtype)


def _image(case, seed):
    shape = _ext(case["ti"])
    gen = torch.Generator().manual_seed(seed)
    if case["data"] == "facies8":
        return synth.channels(shape, np.random.default_rng(seed))
    ranges = [max(2.0, n / 8) for n in shape]
    if case["data"] == "binary64":
        x = _field(shape, ranges, gen, np.float64)
        return (x > np.quantile(x, 0.7)).astype(np.float64)
    return _field(shape, ranges, gen, np.float32 if case["data"] == "grf32" else np.float64)


def _conditioning(case, T, seed):
    """Soft pairs and hard data of a conditioned simulation (a reference field
    of the grid's extents gives both)."""
    grid = _ext(case["grid"])
    rng = np.random.default_rng(seed + 1)
    soft, hard = [], None
    if case["soft"] or case["hard"]:
        gen = torch.Generator().manual_seed(seed + 1)
        F = _field(grid, [max(2.0, n / 8) for n in T.shape], gen, T.dtype)
        for _ in range(case["soft"]):
            soft.append(tuple((synth.box_blur(x, 9) + rng.normal(0, 0.1, x.shape)).astype(T.dtype) for x in (F, T)))
        flat = rng.choice(F.size, case["hard"], replace=False)
        hard = {tuple(int(c) for c in np.unravel_index(i, grid)): float(F.flat[i]) for i in flat} or None
    return soft, hard


def _grids(case):
    g = _ext(case["grid"])
    if case["grids"] == 1:
        return [g]
    # "100x300x30": plan extents between the first two numbers, the third fixed
    rng = np.random.default_rng(case["grids"])  # the case's own sizes, the same for every seed
    lo, hi = min(g[:2]), max(g[:2])
    return [(int(rng.integers(lo, hi + 1)), int(rng.integers(lo, hi + 1)), g[2]) for _ in range(case["grids"])]


def prepare(case, seed):
    if case["kind"] == "graphcut":
        # two windows that agree roughly, as a pick and the pasted grid do
        s = _ext(case["slab"])
        gen = torch.Generator().manual_seed(seed)
        dt = np.float32 if case["data"] == "grf32" else np.float64
        pad = tuple(max(n + 1, 16) for n in s)
        cut = tuple(slice(0, n) for n in s)
        base, d1, d2 = (_field(pad, [12] * 3, gen, np.float64)[cut] for _ in range(3))
        return {"case": case, "A": np.asfortranarray((base + 0.4 * d1).astype(dt)),
                "B": np.asfortranarray((base + 0.4 * d2).astype(dt))}
    T = _image(case, seed)
    if case["kind"] == "fastdistance":
        t = _ext(case["tile"])
        rng = np.random.default_rng(seed + 3)
        o = [int(rng.integers(0, n - m + 1)) for n, m in zip(T.shape, t)]
        kern = T[tuple(slice(a, a + m) for a, m in zip(o, t))].astype(np.float64)
        kern = kern + 0.3 * rng.standard_normal(t)
        w = np.zeros(t, dtype=bool)
        for d in range(2):
            w[tuple(slice(0, math.ceil(case["overlap"] * t[d])) if e == d else slice(None) for e in range(3))] = True
        return {"case": case, "T": np.asfortranarray(T), "kern": np.asfortranarray(kern), "w": np.asfortranarray(w)}
    tile = _ext(case["tile"])
    kw = dict(overlap=(case["overlap"],) * len(tile), tol=case["tol"], path=case["path"])
    soft, hard = _conditioning(case, T, seed)
    rng = np.random.default_rng(seed + 4)
    if case["kind"] == "call":
        return {"case": case, "T": T, "tile": tile, "grid": _ext(case["grid"]), "seed": seed + 4,
                "kw": dict(kw, nreal=case["nreal"], soft=soft, hard=hard)}
    grids = _grids(case)
    plan, _ = iqhip.make_plan_multi(T, tile, grids, soft=soft, hard=None if hard is None else [hard] * len(grids),
                                    nreal=case["nreal"], rng=rng, **kw)
    if case["learned"]:
        plan.learn()
        plan.set_proposal(True, K=2048, check_every=16, min_recall=0.99, check_queries=32)
    n = sum(int(np.prod(p)) for p in plan.real_padsize)
    return {"case": case, "plan": plan, "buf": plan.ctx.pinned_empty(n, plan.dtype),
            "uniforms": [rng.random(k) for k in plan.real_npath]}


def run(state):
    kind = state["case"]["kind"]
    if kind == "plan":
        plan = state["plan"]
        plan.run(state["uniforms"])
        res = plan.results(grids=True, chosen=True, out=state["buf"])
        return {"grids": list(res["grids"]), "chosen": [np.asarray(c) for c in res["chosen"]]}
    if kind == "call":
        return iqhip.iqsim(state["T"], state["tile"], state["grid"], rng=np.random.default_rng(state["seed"]),
                           **state["kw"])
    if kind == "fastdistance":
        return iqhip.fastdistance(state["T"], state["kern"], state["w"])
    return iqhip.graphcut(state["A"], state["B"], state["case"]["dim"])


def _esize(case):
    return 4 if case["data"] == "grf32" else 8


def work(case):
    if case["kind"] == "graphcut":
        n = float(np.prod(_ext(case["slab"])))
        # both slabs in, the mask out; three edges a voxel, each weighed once
        return {"bytes": n * (2 * _esize(case) + 1), "flops": n * 3 * 8}
    ti, t = _ext(case["ti"]), _ext(case["tile"])
    P = float(np.prod([a - b + 1 for a, b in zip(ti, t)]))
    if case["kind"] == "fastdistance":
        o = [math.ceil(case["overlap"] * v) for v in t[:2]]
        V = float(np.prod(t) - (t[0] - o[0]) * (t[1] - o[1]) * t[2])
        return {"bytes": float(np.prod(ti)) * _esize(case) + float(np.prod(t)) * 9 + P * 8, "flops": 4 * P * V}
    nbytes, flops = float(np.prod(ti)) * _esize(case) * (1 + case["soft"]), 0.0
    for grid in _grids(case):
        geo = prep.geometry(ti, t, grid, (case["overlap"],) * len(t))
        # overlap voxels of a raster path's tiles (2-D: the third axis has one tile)
        V = 0.0
        for i in np.ndindex(*geo["ntiles"]):
            keep = [a - (o if k > 0 and o > 1 else 0) for a, o, k in zip(t, geo["ovlsize"], i)]
            V += np.prod(t) - np.prod(keep)
        steps = float(np.prod(geo["ntiles"]))
        vox = float(np.prod(geo["padsize"]))
        nbytes += case["nreal"] * vox * _esize(case) + case["soft"] * vox * 8
        per = 2 * 64 * steps if case["learned"] else 2 * V
        flops += case["nreal"] * P * (per + case["soft"] * 2 * float(np.prod(t)) * steps)
    if case["learned"]:
        nbytes += P * (64 * 2 + 4)
    return {"bytes": float(nbytes), "flops": float(flops)}


def exact(case, seed):
    """Simulated grids are copies of training-image values chosen step by step
    and cuts are labels: neither has a value of its own in other arithmetic."""
    if case["kind"] != "fastdistance":
        return None
    s = prepare(case, seed)
    T = torch.from_numpy(np.ascontiguousarray(s["T"], dtype=np.float64))[None, None]
    w = torch.from_numpy(np.ascontiguousarray(s["w"], dtype=np.float64))[None, None]
    k = torch.from_numpy(np.ascontiguousarray(s["kern"]))[None, None] * w
    a2 = torch.nn.functional.conv3d(T * T, w)
    ab = torch.nn.functional.conv3d(T, k)
    return torch.abs((a2 - 2.0 * ab) + (k * k).sum())[0, 0].numpy()
