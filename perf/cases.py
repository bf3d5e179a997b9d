"""Timed cases of the triangulator: what its users have it do, through the public entry points.

Every case is one call (or the pair of calls that belong together) on inputs that are already
where such a program holds them: device arrays for the solvers, numpy arrays for
``gcdt_amd.solve``.  The inputs are those of ``gcdt_amd.gen``'s workloads (uniform points with
rows of segments, clustered points with rings, lattices with diagonals, star polygons with
holes), drawn on the GPU so that they are quick to make.  All outputs are whole numbers.
"""
from __future__ import annotations

import ctypes
import math

import torch

import gcdt_amd
from gcdt_amd import api
from gcdt_amd.lib import Stats, check, lib

BITS = 20               # coordinates are drawn in [0, 2^20) and mapped to the 2^30 grid
SIDE = 1 << BITS
HPOINT = api.HPOINT_DTYPE.itemsize


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # one small request, as a server gets it: all launches and waits, hardly any work
        {"name": "solve_300", "kind": "solve", "points": "uniform", "cons": "rings", "n": 300, "c": 12, "adj": False},
        # a small mesh with adjacency, for a program that walks it afterwards
        {"name": "solve_2k_adj", "kind": "solve", "points": "uniform", "cons": "rings", "n": 2053, "c": 80,
         "adj": True},
        # an ordinary request: polygon boundaries of a few percent of the points
        {"name": "solve_20k", "kind": "solve", "points": "uniform", "cons": "rings", "n": 20011, "c": 600,
         "adj": False},
        # plain CDT, small: 100k uniform points and 1,000 horizontal segments
        {"name": "rows_100k", "kind": "solve", "points": "uniform", "cons": "rows", "n": 100_000, "c": 1000,
         "adj": False},
        # the largest request of the serving workload
        {"name": "solve_1m", "kind": "solve", "points": "uniform", "cons": "rings", "n": 1_000_000, "c": 30_000,
         "adj": False},
        # plain CDT, large: 80% uniform, 20% clustered points and 1,000 rings of 100 segments
        {"name": "cluster_10m", "kind": "solve", "points": "cluster", "cons": "rings", "n": 10_000_000,
         "c": 100_000, "adj": False},
        # degenerate input: a lattice (everything cocircular) with diagonals through many vertices
        {"name": "lattice_4m", "kind": "solve", "points": "lattice", "cons": "diagonals", "n": 2048 * 2048, "c": 121,
         "adj": False},
        # a few small instances that waited together in a server's queue
        {"name": "batch_32", "kind": "batch", "instances": 32, "nmin": 64, "nmax": 8192},
        # many instances at once, log-uniform sizes
        {"name": "batch_1k", "kind": "batch", "instances": 1024, "nmin": 64, "nmax": 65536},
        # the triangles inside polygons: a solve with constraint bits, then even-odd carving
        {"name": "carve_200k", "kind": "carve", "points": "uniform", "cons": "rings", "n": 200_003, "c": 8000},
        # numpy arrays in, numpy arrays out
        {"name": "host_200k", "kind": "host", "points": "cluster", "cons": "rings", "n": 200_000, "c": 4000},
        # constraints that cross each other, with exact crossing vertices
        {"name": "crossing_30k", "kind": "crossing", "points": "uniform", "cons": "crossing", "n": 30_000, "c": 24},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "solve", "solve", "batch", "batch", "carve", "host", "crossing"])
    if kind == "batch":
        k = log(2, 1024)
        lo = log(16, 512)
        # the largest size so that the batch stays below the largest listed one
        hi = log(lo, max(lo, 65536))
        return {"kind": kind, "instances": k, "nmin": lo, "nmax": hi}
    if kind == "crossing":
        return {"kind": kind, "points": "uniform", "cons": "crossing", "n": log(300, 100_000), "c": rng.randint(4, 24)}
    points = rng.choice(["uniform", "uniform", "cluster", "lattice"])
    n = log(100, {"solve": 10_000_000, "carve": 1_000_000, "host": 1_000_000}[kind])
    if points == "lattice":
        side = max(8, min(2048, math.isqrt(n)))
        n = side * side
        case = {"kind": kind, "points": points, "cons": "diagonals", "n": n, "c": rng.randint(1, max(1, side // 16))}
    else:
        cons = "rings" if kind == "carve" else rng.choice(["rings", "rings", "rows", "none"])
        share = rng.uniform(0.002, 0.05)
        c = 0 if cons == "none" else max(12, min(100_000, int(n * share)))
        if cons == "rows":
            c = min(c, 1000)
        case = {"kind": kind, "points": points, "cons": cons, "n": n, "c": c}
    if kind == "solve":
        case["adj"] = rng.random() < 0.4
    return case


# ------------------------------------------------------------------ inputs


def _unit(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _points(case, m, g):
    """m integer coordinates in [0, 2^20)^2, repeated ones among them."""
    xy = torch.randint(0, SIDE, (m, 2), generator=g, device="cuda")
    if case["points"] == "cluster":
        centre = torch.randint(0, SIDE, (64, 2), generator=g, device="cuda")
        which = torch.randint(0, 64, (m,), generator=g, device="cuda")
        offset = torch.randn(m, 2, generator=g, device="cuda", dtype=torch.float64) * 4096
        near = (centre[which] + offset.round().long()).clamp(0, SIDE - 1)
        xy = torch.where(_unit(g, m, 1) < 0.2, near, xy)
    return xy


def _segments(case, g):
    """(c, 2, 2) endpoints; but for "crossing" no two segments cross."""
    c = case["c"]
    if c == 0:
        return torch.zeros(0, 2, 2, dtype=torch.int64, device="cuda")
    if case["cons"] == "rows":
        y = torch.randperm(SIDE, generator=g, device="cuda")[:c]
        x = torch.randperm(SIDE, generator=g, device="cuda")[: 2 * c].view(c, 2)
        return torch.stack([x, y[:, None].expand(c, 2)], 2)
    if case["cons"] == "crossing":
        a = _unit(g, c) * 2 * math.pi
        mid = SIDE * (0.25 + 0.5 * _unit(g, c, 2))
        d = torch.stack([a.cos(), a.sin()], 1) * (SIDE * (0.03 + 0.17 * _unit(g, c, 1)))
        return torch.stack([mid - d, mid + d], 1).round().long()
    if case["cons"] == "diagonals":
        # one diagonal in each of c blocks of the lattice, upwards or downwards
        k = math.isqrt(case["n"])
        side = math.ceil(math.sqrt(c))
        block = k // side
        at = torch.arange(c, device="cuda")
        corner = torch.stack([at // side, at % side], 1) * block
        length = 1 + (_unit(g, c) * (block - 1)).long().clamp(max=block - 2)
        up = _unit(g, c) < 0.5
        x0, y0 = corner[:, 0], corner[:, 1] + torch.where(up, 0, length)
        x1, y1 = x0 + length, y0 + torch.where(up, length, -length)
        return torch.stack([torch.stack([x0, y0], 1), torch.stack([x1, y1], 1)], 1) * (SIDE // k)
    # rings: one k-gon in each of a grid of squares
    k = max(6, min(100, c // 2))
    rings = max(1, c // k)
    side = math.ceil(math.sqrt(rings))
    cell = SIDE / side
    at = torch.arange(rings, device="cuda")
    r = cell * (0.1 + 0.3 * _unit(g, rings, 1))
    mid = (torch.stack([at // side, at % side], 1) + 0.5) * cell + (_unit(g, rings, 2) - 0.5) * (0.96 * cell - 2 * r)
    a = torch.arange(k, device="cuda", dtype=torch.float64) * (2 * math.pi / k)
    v = (mid[:, None] + r[:, None] * torch.stack([a.cos(), a.sin()], 1)).round().long()
    return torch.stack([v, v.roll(-1, 1)], 2).reshape(-1, 2, 2)


def _order(corner, other, groups, want, g):
    """Point keys in the order a program has them: all of `corner` (segment ends, distinct ones
    are kept) and the first of `other` that are no repeats, want[i] points of group i (the key
    above the coordinates) in all, each group shuffled.  Returns the keys and the segment ends' places."""
    corner_key, ids = torch.unique(corner, return_inverse=True)
    other = torch.unique(other)
    other = other[~torch.isin(other, corner_key)]
    key = torch.cat([corner_key, other])
    rank = torch.rand(len(key), generator=g, device="cuda", dtype=torch.float64)
    rank[: len(corner_key)] -= 1  # segment ends first, then as many others as are wanted
    by = rank.argsort()
    by = by[(key[by] >> (2 * BITS)).argsort(stable=True)]
    group = key[by] >> (2 * BITS)
    count = torch.bincount(group, minlength=groups)
    by = by[torch.arange(len(by), device="cuda") - (count.cumsum(0) - count)[group] < want[group]]
    # shuffled again inside each group, so that segment ends lie anywhere
    by = by[torch.randperm(len(by), generator=g, device="cuda")]
    by = by[(key[by] >> (2 * BITS)).argsort(stable=True)]
    place = torch.full((len(key),), -1, dtype=torch.int64, device="cuda")
    place[by] = torch.arange(len(by), device="cuda")
    return key[by], place[ids]


def _to_grid(key):
    xy = torch.stack([(key >> BITS) & (SIDE - 1), key & (SIDE - 1)], 1)
    return ((xy << 10) + 512).to(torch.int32).contiguous()


def _key(p):
    return (p[:, 0] << BITS) | p[:, 1]


def _single(case, g):
    n = case["n"]
    segs = _segments(case, g).reshape(-1, 2)
    if case["points"] == "lattice":
        i = torch.arange(math.isqrt(n), device="cuda") * (SIDE // math.isqrt(n))
        xy = torch.cartesian_prod(i, i)
    else:
        xy = _points(case, n + n // 50 + 64, g)
        n += len(torch.unique(_key(segs)))
    key, ends = _order(_key(segs), _key(xy), 1, torch.tensor([n], device="cuda"), g)
    return _to_grid(key), ends.view(-1, 2).to(torch.int32)


def _stars(case, g):
    """Star polygons with up to four star-shaped holes and uniform points between them: flat
    points, flat constraints with local ids, and both lists' offsets.  The sizes are
    log-uniform, in an order of the seed's."""
    K = case["instances"]
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    at = torch.randperm(K, generator=g, device="cuda")
    n = (lo + (hi - lo) * (at + 0.5) / K).exp().round().long()
    R = SIDE * (0.25 + 0.2 * _unit(g, K))
    outer = torch.minimum(16 + (497 * _unit(g, K)).long(), n // 2).clamp(min=3)
    holes = torch.randint(0, 5, (K, 1), generator=g, device="cuda")
    hole = torch.where(torch.arange(4, device="cuda") < holes, 16 + (49 * _unit(g, K, 4)).long(), 0)
    hole = torch.where((n // 2 - outer >= 4 * 64)[:, None], hole, 0)
    turn = (torch.arange(4, device="cuda") + 0.4 * _unit(g, K, 4)) * (math.pi / 2)
    hx, hy = SIDE / 2 + 0.38 * R[:, None] * turn.cos(), SIDE / 2 + 0.38 * R[:, None] * turn.sin()
    hr = R[:, None] * (0.05 + 0.1 * _unit(g, K, 4))
    # all polygons as one list: instance, size, centre and radius of each
    inst = torch.arange(K, device="cuda")
    pi = torch.cat([inst, inst.repeat_interleave(4)])
    pm = torch.cat([outer, hole.reshape(-1)])
    mid = torch.full((K,), SIDE / 2, device="cuda", dtype=torch.float64)
    px, py, pr = torch.cat([mid, hx.reshape(-1)]), torch.cat([mid, hy.reshape(-1)]), torch.cat([R, hr.reshape(-1)])
    first = pm.cumsum(0) - pm
    poly = torch.arange(len(pm), device="cuda").repeat_interleave(pm)
    j = torch.arange(len(poly), device="cuda") - first[poly]
    a = (j + 0.5 * _unit(g, len(poly))) * (2 * math.pi) / pm[poly]
    rad = pr[poly] * (0.7 + 0.3 * _unit(g, len(poly)))
    v = torch.stack([(px[poly] + rad * a.cos()).round().long(), (py[poly] + rad * a.sin()).round().long()], 1)
    corner = (pi[poly] << (2 * BITS)) | _key(v)
    # points inside the outer polygon's inner circle, none in a hole's outer circle: more than
    # are wanted, as some fall into holes
    who = inst.repeat_interleave(n + n // 2 + 32)
    a, d = _unit(g, len(who)) * (2 * math.pi), _unit(g, len(who)).sqrt() * 0.65 * R[who]
    x, y = SIDE / 2 + d * a.cos(), SIDE / 2 + d * a.sin()
    clear = torch.ones_like(who, dtype=torch.bool)
    for h in range(4):
        off = (x - hx[who, h]) ** 2 + (y - hy[who, h]) ** 2 > (1.05 * hr[who, h]) ** 2
        clear &= off | (hole[who, h] == 0)
    other = ((who << (2 * BITS)) | _key(torch.stack([x.floor().long(), y.floor().long()], 1)))[clear]
    key, ends = _order(corner, other, K, n, g)
    poff = torch.zeros(K + 1, dtype=torch.int64, device="cuda")
    poff[1:] = n.cumsum(0)
    cons = torch.stack([ends, ends[first[poly] + (j + 1) % pm[poly]]], 1) - poff[pi[poly]][:, None]
    by = pi[poly].argsort(stable=True)
    coff = torch.zeros(K + 1, dtype=torch.int64, device="cuda")
    coff[1:] = torch.bincount(pi[poly], minlength=K).cumsum(0)
    return _to_grid(key), poff.cpu().numpy(), cons[by].to(torch.int32).contiguous(), coff.cpu().numpy()


class _Dev:
    """A tensor as the device buffer that the entry points take."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


def _ints(*shape):
    return torch.zeros(*shape, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = case["kind"]
    if kind == "batch":
        pts, poff, cons, coff = _stars(case, g)
        tris = _ints(2 * len(pts) + 2 * case["instances"], 3)
        return {"kind": kind, "pts": _Dev(pts), "poff": poff, "cons": _Dev(cons), "coff": coff, "tris": _Dev(tris)}
    pts, cons = _single(case, g)
    n, c = len(pts), len(cons)
    if kind == "host":
        return {"kind": kind, "pts": pts.cpu().numpy(), "cons": cons.cpu().numpy()}
    s = {"kind": kind, "pts": _Dev(pts), "n": n, "cons": _Dev(cons), "c": c}
    room = 2 * n + 2
    if kind == "crossing":
        s["most"] = c * c
        room += 2 * s["most"]
        s["points"] = _Dev(torch.zeros(HPOINT * s["most"], dtype=torch.uint8, device="cuda"))
    s["tris"] = _Dev(_ints(room, 3))
    if kind != "solve" or case["adj"]:
        s["adj"] = _Dev(_ints(room, 3))
    if kind in ("carve", "crossing"):
        s["cflag"] = _Dev(_ints(room))
    if kind == "carve":
        s["inside"] = _Dev(_ints(room))
    return s


# ------------------------------------------------------------------ one pass


def run(s):
    kind = s["kind"]
    if kind == "host":
        tris, _ = gcdt_amd.solve(s["pts"], s["cons"])
        return tris
    if kind == "batch":
        api.solve_batch_device(s["pts"], s["poff"], s["cons"], s["coff"], s["tris"])
        return s["tris"].t
    if kind == "solve":
        api.solve_device(s["pts"], s["n"], s["cons"], s["c"], s["tris"], s.get("adj"))
        return [s[k].t for k in ("tris", "adj") if k in s]
    nt, more, st = ctypes.c_int(0), ctypes.c_int(0), Stats()
    cons = s["cons"].ptr if s["c"] else None
    if kind == "crossing":
        check(lib().gcdt_solve_steiner(s["pts"].ptr, s["n"], cons, s["c"], s["most"], s["tris"].ptr, s["adj"].ptr,
                                       s["cflag"].ptr, s["points"].ptr, ctypes.byref(nt), ctypes.byref(more),
                                       ctypes.byref(st), None), "gcdt_solve_steiner")
        return [nt.value, more.value] + [s[k].t for k in ("tris", "adj", "cflag", "points")]
    check(lib().gcdt_solve_flags(s["pts"].ptr, s["n"], cons, s["c"], s["tris"].ptr, s["adj"].ptr, s["cflag"].ptr,
                                 ctypes.byref(nt), ctypes.byref(st), None), "gcdt_solve_flags")
    check(lib().gcdt_carve(s["tris"].ptr, s["adj"].ptr, s["cflag"].ptr, nt.value, s["n"], s["inside"].ptr,
                           ctypes.byref(more), None), "gcdt_carve")
    return [s[k].t for k in ("tris", "adj", "cflag", "inside")]


def work(case):
    """Points and segments in, triangles (and what else is asked for) out, each once; the
    predicates: about three in-circle tests and three orientations a triangle."""
    if case["kind"] == "batch":
        lo, hi = case["nmin"], case["nmax"]
        n = case["instances"] * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        c = 200 * case["instances"]
    else:
        n, c = case["n"], case["c"]
    per = 12
    if case["kind"] == "solve" and case["adj"] or case["kind"] == "crossing":
        per = 24 + 4 * (case["kind"] == "crossing")
    elif case["kind"] == "carve":
        per = 32
    return {"bytes": 8 * n + 8 * c + per * (2 * n + 2), "flops": 2 * n * 3 * (30 + 7)}


def exact(case, seed):
    """All outputs are whole numbers: there is nothing to be off by."""
    return None
