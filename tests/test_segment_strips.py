"""Vertices on segments, found cell by cell: the lanes that share a segment's
strips change at 1, 2, 4, ... 64 strips, and several lanes share the points of
a cell where strips are few.  Segments through many vertices at those widths,
in the four directions that choose the strips, with crowded cells among them."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.emu import emu

STEP = 349_524  # a third of a cell's side, and a multiple of 12
WIDTHS = [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 64, 65, 130]
DIRECTIONS = {"row": (STEP, 0), "column": (0, STEP), "flat": (STEP, -STEP // 12), "steep": (STEP // 3, STEP)}


def lines(direction, crowd):
    """One segment per width, its vertices three to a strip; `crowd` more
    points in the first cell of every third one.  Points, segments, pieces."""
    rng = np.random.default_rng(8)
    d = np.array(DIRECTIONS[direction])
    flat = abs(d[0]) > abs(d[1])
    pts, cons, more = [], [], [rng.integers(1, (1 << 30) - 1, (400, 2))]
    n = 0
    for i, w in enumerate(WIDTHS):
        steps = max(2, 3 * (w - 1))
        at = np.array([20, 60 + 8 * i] if flat else [60 + 8 * i, 20]) * (1 << 20) + 1000
        pts.append(at + np.arange(steps + 1)[:, None] * d)
        cons.append([n, n + steps] if i % 2 else [n + steps, n])
        n += steps + 1
        if i % 3 == 0:
            more.append(rng.integers(0, 1 << 20, (crowd, 2)) + (at >> 20 << 20))
    line = np.concatenate(pts)
    other = np.unique(np.concatenate(more), axis=0)
    key = lambda p: p[:, 0] << 32 | p[:, 1]  # noqa: E731
    off = ~np.isin(key(other), key(line))
    for (a, b), w in zip(cons, WIDTHS):  # and on no segment
        A, D = line[min(a, b)], d
        cross = (other[:, 0] - A[0]) * D[1] - (other[:, 1] - A[1]) * D[0]
        off &= cross != 0
    xy = np.concatenate([line, other[off]])
    perm = rng.permutation(len(xy))
    inv = np.empty_like(perm)
    inv[perm] = np.arange(len(xy))
    return xy[perm].astype(np.int32), inv[np.array(cons)].astype(np.int32), n - len(WIDTHS)


def check(g, cons, tris, pieces, want):
    assert pieces == want
    v = O.validate(g, tris, cons)
    assert v["valid"], v
    if v["unique"]:
        ref, _ = O.cdt(g, cons)
        assert np.array_equal(O.canonical(tris), O.canonical(ref))


@pytest.mark.parametrize("direction", list(DIRECTIONS))
def test_vertices_on_segments(direction):
    emu.build()
    g, cons, want = lines(direction, 90)
    tris, _, st = emu.solve(g, cons)
    check(g, cons, tris, st["segments"], want)


@pytest.mark.gpu
@pytest.mark.parametrize("crowd", [90, 5000])
@pytest.mark.parametrize("direction", list(DIRECTIONS))
def test_vertices_on_segments_on_the_gpu(direction, crowd):
    from gcdt_amd import solve
    g, cons, want = lines(direction, crowd)
    tris, st = solve(g, cons)
    check(g, cons, tris, st["segments"], want)


@pytest.mark.gpu
def test_short_segments_in_one_crowded_cell():
    """20,000 segments whose one cell holds all 200,000 points are 4e9 tests:
    shared by all lanes about 5 ms, by one lane of a wave above 200."""
    from gcdt_amd import solve
    rng = np.random.default_rng(4)
    g = np.unique(rng.integers(0, 1 << 20, (204_000, 2)), axis=0)
    g = rng.permutation(g)[:200_000] + (768 << 20)
    block = ((g - (768 << 20)) * 141 >> 20) @ np.array([1000, 1])
    by = np.argsort(block, kind="stable")
    start = np.flatnonzero(np.r_[True, np.diff(block[by]) > 0])
    end = np.r_[start[1:], len(by)] - 1
    some = end > start
    cons = np.stack([by[start[some]], by[end[some]]], 1).astype(np.int32)
    g = g.astype(np.int32)
    assert len(cons) > 19_000
    solve(g, cons)
    tris, st = solve(g, cons)
    assert O.validate(g, tris, cons)["valid"]
    assert st["ms_constraints"] < 50, st
