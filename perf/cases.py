"""The join-and-clip work that a user of this library has it do, as cases that
can be timed: what each stands for is said beside it in listed().

A case is a dict of plain values; its "kind" says which public calls one pass
makes.  Inputs are made on the GPU, from the seed alone, with the
distributions of the library's own generators (star-shaped and six-sinusoid
rings, layers in the unit square, log-normal pair sizes, rings with holes).
The layers stay resident on the device, and one context serves the whole
process, as a serving program keeps them; results come back whole through
gcmf_join_get and gcmf_clip_get, the only calls that return them, into result
buffers in pinned host memory that are sized for the case (counts say how much
of them is filled).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gcmf-gh_amd"))

import gcmf_amd as G  # noqa: E402

TAU = 2.0 * math.pi
_ctx = None


def context():
    """The process's context: one stream and its grow-only workspace."""
    global _ctx
    if _ctx is None:
        _ctx = G.Context(0)
    return _ctx


def listed():
    return [
        # one clip request of a served stream by itself: launches and
        # read-backs are all there is
        {"name": "pair_64x48", "kind": "pair", "shape": "star", "n_p": 64, "n_q": 48,
         "snap": 0.0, "cleanup": True},
        # the ordinary single pair, two detailed parcels; with the clean-up
        # off, as area computations take it
        {"name": "pair_2000x1500", "kind": "pair", "shape": "star", "n_p": 2000, "n_q": 1500,
         "snap": 0.0, "cleanup": False},
        # digitised boundaries on a coordinate grid: shared vertices and
        # collinear edges all along the rings
        {"name": "pair_grid_8001x2003", "kind": "pair", "shape": "wavy", "n_p": 8001,
         "n_q": 2003, "snap": 1e-3, "cleanup": True},
        # the largest single pair: a coastline against a district boundary
        {"name": "pair_1000000x100000", "kind": "pair", "shape": "wavy", "n_p": 1000000,
         "n_q": 100000, "snap": 0.0, "cleanup": True},
        # what a serving loop admits at once under load: a small ragged batch
        {"name": "batch_37", "kind": "batch", "pairs": 37, "median": 64.0, "n_max": 2000,
         "cleanup": True},
        # an overlay job's own pairs, very uneven sizes, three in ten apart
        {"name": "batch_20000", "kind": "batch", "pairs": 20000, "median": 64.0,
         "n_max": 50000, "cleanup": True},
        # a served join of two small resident layers
        {"name": "join_1000", "kind": "join", "base": 1000, "over": 1000, "n_min": 16,
         "n_max": 512, "r_min": 1e-4, "r_max": 5e-3},
        # layers of many small polygons (buildings against land cover)
        {"name": "join_300000x250007", "kind": "join", "base": 300000, "over": 250007,
         "n_min": 8, "n_max": 8, "r_min": 3.4e-4, "r_max": 8.5e-4},
        # the headline workload: join of two layers, then the clip of every
        # joined pair
        {"name": "join_clip_20000", "kind": "join_clip", "base": 20000, "over": 20000,
         "n_min": 16, "n_max": 512, "r_min": 1e-4, "r_max": 5e-3},
        # multi-ring polygons (holes, islands): intersection of a layer's
        # pairs, and the union of a few
        {"name": "complex_intersection_300", "kind": "complex", "pairs": 300, "union": False},
        {"name": "complex_union_7", "kind": "complex", "pairs": 7, "union": True},
        # the exported device primitives on one column: offsets of the
        # counts, indices of the survivors, order of the keys
        {"name": "primitives_3000017", "kind": "primitives", "n": 3000017, "bits": 64},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "batch", "join", "join", "join_clip", "complex",
                       "primitives"])
    if kind == "pair":
        shape = rng.choice(["star", "wavy", "grid"])
        if shape == "star":
            n_p = _log(rng, 8, 5000)
            return {"kind": kind, "shape": "star", "n_p": n_p, "n_q": _log(rng, 8, 4000),
                    "snap": 0.0, "cleanup": rng.random() < 0.7}
        if shape == "wavy":
            n_p = _log(rng, 5000, 900000)
            return {"kind": kind, "shape": "wavy", "n_p": n_p,
                    "n_q": _log(rng, 1000, max(1001, n_p // 9)), "snap": 0.0, "cleanup": True}
        n_p = _log(rng, 500, 8000)
        return {"kind": kind, "shape": "wavy", "n_p": n_p, "n_q": _log(rng, 200, 2000),
                "snap": 1e-3, "cleanup": True}
    if kind == "batch":
        return {"kind": kind, "pairs": _log(rng, 2, 16000), "median": float(rng.randint(24, 72)),
                "n_max": _log(rng, 500, 40000), "cleanup": rng.random() < 0.7}
    if kind == "join":
        if rng.random() < 0.5:
            return {"kind": kind, "base": _log(rng, 1000, 20000), "over": _log(rng, 1000, 20000),
                    "n_min": 16, "n_max": 512, "r_min": 1e-4, "r_max": 5e-3}
        b = _log(rng, 30000, 300000)
        r = 0.9 / math.sqrt(b)
        return {"kind": kind, "base": b, "over": _log(rng, 20000, 250000),
                "n_min": 5, "n_max": rng.randint(6, 10), "r_min": 0.2 * r, "r_max": 0.5 * r}
    if kind == "join_clip":
        return {"kind": kind, "base": _log(rng, 500, 18000), "over": _log(rng, 500, 18000),
                "n_min": 16, "n_max": rng.randint(100, 512), "r_min": 1e-4, "r_max": 5e-3}
    if kind == "complex":
        return {"kind": kind, "pairs": _log(rng, 1, 290), "union": rng.random() < 0.5}
    return {"kind": kind, "n": _log(rng, 3000, 2900000), "bits": rng.choice([32, 64])}


# ------------------------------------------------------------- inputs ----
def _uniform(g, n, lo, hi):
    return lo + (hi - lo) * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _ring_index(n):
    """Ring of every vertex and the vertex's place in it, for ring sizes n."""
    ring = torch.repeat_interleave(torch.arange(len(n), device=n.device), n)
    first = torch.cumsum(n, 0) - n
    return ring, torch.arange(len(ring), device=n.device) - first[ring]


def _stars(g, n, cx, cy, r, amp, sign=None):
    """Star-shaped rings of n[i] vertices about (cx, cy): vertex k at angle
    2 pi (k + U(-0.4, 0.4)) / n, radius r (1 + amp U(-1, 1))."""
    ring, k = _ring_index(n)
    th = TAU / n[ring] * (k + _uniform(g, len(ring), -0.4, 0.4))
    if sign is not None:
        th = th * sign[ring]
    rad = r[ring] * (1.0 + amp * _uniform(g, len(ring), -1.0, 1.0))
    return torch.stack([cx[ring] + rad * torch.cos(th), cy[ring] + rad * torch.sin(th)], 1)


def _wavy(g, n, cx, cy, shape):
    """One ring of radius 1 + 0.2/6 sum_k sin(2^k th + phase_k) + 0.02 U(-1, 1).
    The phases, and with them how the two boundaries of a pair run into each
    other, belong to the case; the seed moves the vertices."""
    k = torch.arange(n, device="cuda")
    th = TAU / n * (k + _uniform(g, n, -0.4, 0.4))
    s = sum(torch.sin((1 << j) * th + shape.uniform(0.0, TAU)) for j in range(6))
    rad = 1.0 + 0.2 * (s / 6.0) + 0.02 * _uniform(g, n, -1.0, 1.0)
    return torch.stack([cx + rad * torch.cos(th), cy + rad * torch.sin(th)], 1)


def _snap(xy, grid):
    """Vertices on a grid, consecutive duplicates dropped."""
    xy = torch.round(xy / grid) * grid
    return xy[(xy != torch.roll(xy, 1, 0)).any(1)]


def _sizes(g, count, lo, hi):
    """Log-uniform whole numbers in [lo, hi]."""
    v = torch.exp(_uniform(g, count, math.log(lo), math.log(hi + 1.0)))
    return torch.clamp(torch.floor(v), lo, hi).to(torch.int64)


class Layer:
    """A layer resident on the device in the library's layout: closed rings,
    their sizes and prefix sums, MBRs and their integer keys (12 fractional
    digits, offset 9e15)."""

    def __init__(self, n, xy):
        ring, k = _ring_index(n)
        first = torch.cumsum(n, 0) - n
        closed = n + 1
        start = torch.cumsum(closed, 0) - closed
        coords = torch.empty((int(closed.sum()), 2), dtype=torch.float64, device="cuda")
        coords[start[ring] + k] = xy
        coords[start + n] = xy[first]
        at = ring.unsqueeze(1).expand(-1, 2)
        lo = torch.zeros((len(n), 2), dtype=torch.float64, device="cuda")
        lo = lo.scatter_reduce(0, at, xy, "amin", include_self=False)
        hi = torch.zeros_like(lo).scatter_reduce(0, at, xy, "amax", include_self=False)
        self.n, self.xy = n, xy
        self.coords = coords
        self.vnum = closed.to(torch.int32)
        self.vpsnum = torch.cumsum(closed, 0)
        self.mbr2 = torch.cat([lo, hi], 1).contiguous()
        self.mbr = (torch.trunc(self.mbr2 * 1e12).to(torch.int64) + 9000000000000000)
        self.desc = G.DLayer(len(n), self.coords.data_ptr(), self.vnum.data_ptr(),
                             self.vpsnum.data_ptr(), self.mbr.data_ptr(), self.mbr2.data_ptr())


def _zeros(n):
    return torch.zeros(n, dtype=torch.float64, device="cuda")


def _layers(case, seed):
    """The two layers of a case, and its pairs or parts (None for a join)."""
    g = torch.Generator("cuda")
    g.manual_seed(int(seed))
    kind = case["kind"]
    if kind == "pair":
        rings = []
        shape = np.random.RandomState(case["n_p"] * 31 + case["n_q"])
        for n, x, y in ((case["n_p"], 0.0, 0.0), (case["n_q"], 0.3, 0.2)):
            if case["shape"] == "wavy":
                xy = _wavy(g, n, x, y, shape)
            else:
                one = torch.ones(1, dtype=torch.float64, device="cuda")
                xy = _stars(g, torch.tensor([n], device="cuda"), one * x, one * y, one, 0.3)
            if case["snap"] > 0.0:
                xy = _snap(xy, case["snap"])
            rings.append(Layer(torch.tensor([len(xy)], device="cuda"), xy.contiguous()))
        return rings[0], rings[1], torch.zeros((1, 2), dtype=torch.int32, device="cuda")
    if kind == "batch":
        M = case["pairs"]
        sizes = [torch.clamp(torch.round(torch.exp(
            math.log(case["median"]) + 1.5 * torch.randn(M, generator=g, device="cuda",
                                                         dtype=torch.float64))),
            8, case["n_max"]).to(torch.int64) for _ in range(2)]
        d = _uniform(g, M, 0.0, 1.4)
        d[torch.rand(M, generator=g, device="cuda") >= 0.7] = 3.0  # 70 % overlap
        ph = _uniform(g, M, 0.0, TAU)
        one = torch.ones(M, dtype=torch.float64, device="cuda")
        p = Layer(sizes[0], _stars(g, sizes[0], _zeros(M), _zeros(M), one, 0.3))
        q = Layer(sizes[1], _stars(g, sizes[1], d * torch.cos(ph), d * torch.sin(ph), one, 0.3))
        k = torch.arange(M, dtype=torch.int32, device="cuda")
        return p, q, torch.stack([k, k], 1).contiguous()
    if kind in ("join", "join_clip"):
        out = []
        for count in (case["base"], case["over"]):
            n = _sizes(g, count, case["n_min"], case["n_max"])
            cx, cy = _uniform(g, count, 0.0, 1.0), _uniform(g, count, 0.0, 1.0)
            r = torch.exp(_uniform(g, count, math.log(case["r_min"]), math.log(case["r_max"])))
            out.append(Layer(n, _stars(g, n, cx, cy, r, 0.3)))
        return out[0], out[1], None
    # complex: an outer ring, up to two holes, an island in the first hole
    M = case["pairs"]
    rs = np.random.RandomState(seed & 0x7fffffff)
    sides, parts = [], np.zeros((M, 4), np.int32)
    for side in range(2):
        rows = []
        for k in range(M):
            s = 100.0 if side == 0 else 80.0
            x, y = (0.0, 0.0) if side == 0 else rs.uniform(-60.0, 60.0, 2)
            parts[k, 2 * side] = len(rows)
            rows.append((rs.randint(12, 60), x, y, s, 1.0))
            holes = rs.randint(0, 3)
            for h in range(holes):
                a = TAU * h / holes
                hx, hy = x + 0.45 * s * math.cos(a), y + 0.45 * s * math.sin(a)
                rows.append((rs.randint(8, 30), hx, hy, 0.2 * s, -1.0))
                if h == 0:
                    rows.append((rs.randint(6, 12), hx, hy, 0.07 * s, 1.0))
            parts[k, 2 * side + 1] = len(rows) - parts[k, 2 * side]
        t = torch.tensor(np.array(rows, np.float64), device="cuda")
        n = t[:, 0].to(torch.int64)
        sides.append(Layer(n, _stars(g, n, t[:, 1], t[:, 2], t[:, 3], 0.25, t[:, 4])))
    return sides[0], sides[1], torch.from_numpy(parts).cuda()


def _column(case, seed):
    g = torch.Generator("cuda")
    g.manual_seed(int(seed))
    n, bits = case["n"], case["bits"]
    keys = torch.randint(0, 1 << 32, (n,), generator=g, device="cuda", dtype=torch.int64)
    if bits == 64:
        keys = (keys << 32) | torch.randint(0, 1 << 32, (n,), generator=g, device="cuda",
                                            dtype=torch.int64)
    counts = torch.randint(0, 100, (n,), generator=g, device="cuda", dtype=torch.int32)
    flags = (torch.rand(n, generator=g, device="cuda") < 0.5).to(torch.int32)
    vals = torch.arange(n, dtype=torch.int32, device="cuda")
    return keys, vals, counts, flags


def _mean_lognormal(median, cap):
    """Mean ring size of a batch: log-normal, sigma 1.5, clamped to [8, cap]."""
    phi = lambda z: 0.5 * (1.0 + math.erf(z / math.sqrt(2.0)))  # noqa: E731
    m, s = math.log(median), 1.5
    a, b = (math.log(8.0) - m) / s, (math.log(cap) - m) / s
    return (8.0 * phi(a) + math.exp(m + s * s / 2) * (phi(b - s) - phi(a - s)) +
            cap * (1.0 - phi(b)))


def _mean_sizes(case):
    """Mean ring size of a join's layers."""
    lo, hi = case["n_min"], case["n_max"]
    return lo if lo == hi else (hi + 1.0 - lo) / math.log((hi + 1.0) / lo)


def _candidates(case):
    """Expected number of a join's pairs whose MBRs overlap: 4 E[(ra + rb)^2]
    per pair in the unit square, a ring's MBR reaching about 1.2 r (1.02 r for
    a few vertices)."""
    lo, hi = case["r_min"], case["r_max"]
    x = math.log(hi / lo)
    r1, r2 = (hi - lo) / x, (hi * hi - lo * lo) / (2 * x)
    reach = 1.2 if case["n_min"] >= 16 else 1.02
    return case["base"] * case["over"] * 4.0 * reach * reach * (2 * r2 + 2 * r1 * r1)


def _room(case):
    """(candidate pairs, pairs clipped, result vertices) that the case's result
    buffers have room for: about twice what its inputs give."""
    kind = case["kind"]
    if kind == "pair":
        nv, nn = case["n_p"] + case["n_q"], case["n_p"] * case["n_q"]
        return 0, 1, int(2 * nv + (nn / 150 if case["shape"] == "star" else nn * 4e-5)) + 64
    if kind == "batch":
        m = case["pairs"] * 2 * _mean_lognormal(case["median"], case["n_max"])
        return 0, case["pairs"], int(0.8 * m) + 12 * case["n_max"] + 64
    if kind == "complex":
        return 0, case["pairs"], 260 * case["pairs"] + 64
    c = _candidates(case)
    c = int(1.25 * c + 10 * math.sqrt(c)) + 64
    return c, c, int(0.9 * c * _mean_sizes(case)) if kind == "join_clip" else 0


def prepare(case, seed):
    """Device-resident inputs, the context, and the buffers that receive the
    results: pinned host memory, device memory for the primitives."""
    s = {"case": case, "ctx": context()}
    if case["kind"] == "primitives":
        n = case["n"]
        s["in"] = _column(case, seed)
        s["keys"] = torch.empty(n, dtype=torch.int64, device="cuda")
        s["vals"] = torch.empty(n, dtype=torch.int32, device="cuda")
        s["offsets"] = torch.empty(n + 1, dtype=torch.int64, device="cuda")
        s["index"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    else:
        s["base"], s["over"], s["pairs"] = _layers(case, seed)
        c, m, v = _room(case)

        def room(n, dtype):
            return torch.zeros(n, dtype=dtype, pin_memory=True)

        if case["kind"] in ("join", "join_clip"):
            s["join"] = {"pairs": room(2 * c, torch.int32), "joined": room(2 * c, torch.int32)}
        if case["kind"] != "join":
            s["clip"] = {"status": room(m, torch.int32), "comp_off": room(m + 1, torch.int64),
                         "comp_sizes": room(v // 3, torch.int32), "xy": room(2 * v, torch.float64)}
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------- a pass ----
def _fetch(ctx, get, fields, out, name, count):
    """One result field, whole, into its buffer."""
    if count > len(out[name]):
        raise RuntimeError("%s: %d values, room for %d" % (name, count, len(out[name])))
    if count:
        ctx._check(get(ctx.h, fields[name][0], ctypes.c_void_p(out[name].data_ptr()), int(count)),
                   name)


def _clip_results(state, st):
    get, f, out = G.hip_lib().gcmf_clip_get, G.C_FIELDS, state["clip"]
    for name, count in (("status", st.pairs), ("comp_off", st.pairs + 1),
                        ("comp_sizes", st.total_comps), ("xy", 2 * st.total_verts)):
        _fetch(state["ctx"], get, f, out, name, count)
    return dict(out, counts=np.array([st.pairs, st.total_comps, st.total_verts]))


def _join_results(state, st):
    get, f, out = G.hip_lib().gcmf_join_get, G.J_FIELDS, state["join"]
    _fetch(state["ctx"], get, f, out, "pairs", 2 * st.candidates)
    _fetch(state["ctx"], get, f, out, "joined", 2 * st.joined)
    return dict(out, counts=np.array([st.candidates, st.joined]))


def run(state):
    """One pass through the public calls, and its results."""
    L, ctx, case = G.hip_lib(), state["ctx"], state["case"]
    kind = case["kind"]
    if kind == "primitives":
        keys, vals, counts, flags = state["in"]
        n = case["n"]
        ctx._check(L.gcmf_scan_i32_i64(ctx.h, counts.data_ptr(), state["offsets"].data_ptr(), n),
                   "scan")
        kept = ctypes.c_long()
        ctx._check(L.gcmf_compact_flags(ctx.h, flags.data_ptr(), n, state["index"].data_ptr(),
                                        ctypes.byref(kept)), "compact")
        ctx._check(L.gcmf_radix_sort_u64(ctx.h, keys.data_ptr(), vals.data_ptr(),
                                         state["keys"].data_ptr(), state["vals"].data_ptr(), n,
                                         case["bits"]), "radix_sort")
        return {"offsets": state["offsets"], "index": state["index"], "kept": kept.value,
                "keys": state["keys"], "vals": state["vals"]}
    base, over = state["base"].desc, state["over"].desc
    js, cs = G.JoinStats(), G.ClipStats()
    flags = G.CLIP_NORMALIZE
    if kind == "join":
        ctx._check(L.gcmf_join(ctx.h, ctypes.byref(base), ctypes.byref(over),
                               ctypes.byref(js)), "join")
        return _join_results(state, js)
    if kind == "join_clip":
        ctx._check(L.gcmf_join_clip(ctx.h, ctypes.byref(base), ctypes.byref(over), flags,
                                    ctypes.byref(js), ctypes.byref(cs)), "join_clip")
        return {"join": _join_results(state, js), "clip": _clip_results(state, cs)}
    pairs = state["pairs"]
    if kind == "complex":
        flags |= G.CLIP_UNION if case["union"] else 0
        ctx._check(L.gcmf_clip_complex(ctx.h, ctypes.byref(base), ctypes.byref(over),
                                       pairs.data_ptr(), len(pairs), flags, ctypes.byref(cs)),
                   "clip_complex")
    else:
        flags |= 0 if case["cleanup"] else G.CLIP_NO_CLEANUP
        ctx._check(L.gcmf_clip(ctx.h, ctypes.byref(base), ctypes.byref(over), pairs.data_ptr(),
                               len(pairs), flags, ctypes.byref(cs)), "clip")
    return _clip_results(state, cs)


# ------------------------------------------------------------ its floor ----
def work(case):
    """Bytes and FP64 operations of one pass that no way of doing it can leave
    out: every ring and MBR read once, every result written once; 32 flops
    for each edge pair that does intersect and 7 for its point.  The counts
    of results are the distributions' own (per vertex: about a third of the
    vertices of both rings come out of an overlapping pair, and a pair of
    star rings has about one intersection per four vertices)."""
    kind = case["kind"]
    if kind == "primitives":
        n = case["n"]
        return {"bytes": n * (4 + 8) + n * (4 + 2) + n * 2 * 12, "flops": 0}
    if kind in ("join", "join_clip"):
        b, o, nv, cand = case["base"], case["over"], _mean_sizes(case), _candidates(case)
        near = min(1.0, cand / max(b, o))  # share of the polygons that meet another
        by = 64 * (b + o) + 16 * nv * (b + o) * near + 8 * cand * 1.9
        if kind == "join":
            return {"bytes": by, "flops": 32 * cand}
        joined = 0.75 * cand
        return {"bytes": by + 16 * 0.35 * 2 * nv * joined,
                "flops": (32 + 7) * 0.25 * 2 * nv * joined}
    if kind == "pair":
        v, share = case["n_p"] + case["n_q"], 0.7
    elif kind == "batch":
        v, share = 2 * case["pairs"] * _mean_lognormal(case["median"], case["n_max"]), 0.7 * 0.7
    else:
        v, share = 2 * 70 * case["pairs"], 0.9
    return {"bytes": 16 * v + 16 * 0.5 * share * v, "flops": (32 + 7) * 0.25 * share * v}


# ------------------------------------------------- the same in 64 bits ----
def _area2(p, q, r):
    return (q[0] - p[0]) * (r[1] - p[1]) - (q[1] - p[1]) * (r[0] - p[0])


def _inside(ring, p):
    """Whether p is in the ring (crossing number)."""
    x0, y0 = ring[:, 0], ring[:, 1]
    x1, y1 = np.roll(x0, -1), np.roll(y0, -1)
    c = (y0 > p[1]) != (y1 > p[1])
    with np.errstate(all="ignore"):
        return bool(np.count_nonzero(c & (p[0] < (x1 - x0) * (p[1] - y0) / (y1 - y0) + x0)) & 1)


def _clean(pts, frame):
    """Vertices whose doubled turn area with their neighbours, in the pair's
    frame, is below 1e-7 go, one after another round the ring."""
    f = (pts - frame[0]) * frame[1]
    n = len(pts)
    nxt, prv = [(i + 1) % n for i in range(n)], [(i - 1) % n for i in range(n)]
    root, left = 0, n

    def small(i):
        return abs(_area2(f[prv[i]], f[i], f[nxt[i]])) < 1e-7

    def drop(i):
        nxt[prv[i]], prv[nxt[i]] = nxt[i], prv[i]

    while left and small(root):
        drop(root)
        root, left = nxt[root], left - 1
    if not left:
        return pts[:0]
    i, out = nxt[root], [root]
    while i != root:
        if small(i):
            drop(i)
        else:
            out.append(i)
        i = nxt[i]
    return pts[out]


def _clip_plain(P, Q, cleanup):
    """Components of P and Q's intersection, rings in general position, by
    the crossings of all edge pairs; None where two edges meet closer to an
    end than a predicate's epsilon tells."""
    if len(P) < len(Q):
        P, Q = Q, P
    lo = np.maximum(P.min(0), Q.min(0))
    hi = np.minimum(P.max(0), Q.max(0))
    if (lo > hi).any():
        return []
    e = float((hi - lo).max())
    scale = 2.0 ** max(0.0, math.ceil(math.log2(math.sqrt(len(P) * len(Q)) / 1024.0)))
    frame = (lo, scale / e if e > 0 else 1.0)
    dP, dQ = np.roll(P, -1, 0) - P, np.roll(Q, -1, 0) - Q
    hits = []
    for i0 in range(0, len(P), 256):  # blocks of P edges against all of Q
        p, d = P[i0:i0 + 256, None], dP[i0:i0 + 256, None]
        w = Q[None] - p
        det = d[..., 0] * dQ[None, :, 1] - d[..., 1] * dQ[None, :, 0]
        with np.errstate(all="ignore"):
            a = (w[..., 0] * dQ[None, :, 1] - w[..., 1] * dQ[None, :, 0]) / det
            b = (w[..., 0] * d[..., 1] - w[..., 1] * d[..., 0]) / det
        i, j = np.nonzero((a > -1e-6) & (a < 1 + 1e-6) & (b > -1e-6) & (b < 1 + 1e-6))
        hits += [(i0 + x, y, a[x, y], b[x, y]) for x, y in zip(i, j)]
    if any(min(a, b, 1 - a, 1 - b) < 1e-6 for _, _, a, b in hits):
        return None
    if not hits:
        out = [P] if _inside(Q, P[0]) else [Q] if _inside(P, Q[0]) else []
    else:
        pts = [(1.0 - a) * P[i] + a * (P[i] + dP[i]) for i, _, a, _ in hits]
        rings, place = [], []
        for side, R in enumerate((P, Q)):
            # ring with its crossings in order: (edge, parameter, crossing)
            seq = sorted([(k, -1.0, -1) for k in range(len(R))] +
                         [(h[side], h[2 + side], c) for c, h in enumerate(hits)])
            inside = _inside((Q, P)[side], R[0])
            at, entry = {}, {}
            for n, (_, _, c) in enumerate(seq):
                if c >= 0:
                    inside = not inside
                    at[c], entry[c] = n, inside
            rings.append([R[k] if c < 0 else pts[c] for k, _, c in seq])
            place.append((seq, at, entry))
        out, done = [], set()
        for _, _, c0 in place[0][0]:
            if c0 < 0 or c0 in done:
                continue
            comp, side, c = [], 0, c0
            while True:
                done.add(c)
                seq, at, entry = place[side]
                n, step = at[c], 1 if entry[c] else -1
                while True:
                    n = (n + step) % len(seq)
                    comp.append(rings[side][n])
                    if seq[n][2] >= 0:
                        break
                c = seq[n][2]
                done.add(c)
                if c == c0:
                    break
                side = 1 - side
            out.append(np.array(comp))
    out = [_clean(c, frame) for c in out] if cleanup else out
    return [c for c in out if len(c)]


def exact(case, seed):
    """The vertices of single-ring clips in general position as plain numpy
    gives them; everything else a pass returns is whole numbers, or a trace
    over degenerate or nested rings that no short program restates."""
    if case["kind"] not in ("pair", "batch"):
        return None
    if case["kind"] == "pair" and (case["snap"] > 0.0 or case["n_p"] * case["n_q"] > 2e7):
        return None
    if case["kind"] == "batch" and case["pairs"] > 150:
        return None
    p, q, _ = _layers(case, seed)
    rings = []
    for lay in (p, q):
        ends = np.cumsum(lay.n.cpu().numpy())
        xy = lay.xy.cpu().numpy()
        rings.append(np.split(xy, ends[:-1]))
    if sum(len(a) * len(b) for a, b in zip(*rings)) > 2e7:
        return None
    out = []
    for a, b in zip(*rings):
        r = _clip_plain(a, b, case["cleanup"])
        if r is None:
            return None
        out += [c.reshape(-1) for c in r]
    xy = np.zeros(2 * _room(case)[2])  # as the result buffer: what is not filled is 0
    got = np.concatenate(out) if out else xy[:0]
    xy[:len(got)] = got
    return {"status": None, "comp_off": None, "comp_sizes": None, "counts": None,
            "xy": torch.from_numpy(xy)}
