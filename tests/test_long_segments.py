"""Constraint segments that cross many triangles: walked in parts, claimed and
retriangulated by waves and workgroups (cavities above 12 crossed triangles),
along rows, columns and slanted lines.

Every path gives the arrays of every other one, so the emulator build with
small caps (cavities above 4, 8 and 20 triangles take the wave, the large
workgroup and its out-of-LDS form) must give the default build's arrays bit for
bit; and every result must equal the oracle's CDT where that is unique."""
import os
import subprocess
import sys

import numpy as np
import pytest

from gcdt_amd import gen
from oracle import oracle as O
from tests.emu import emu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SMALL = (("GCDT_CAV_WAVE_K=4", "GCDT_CAV_MID_K=8", "GCDT_CAV_LDS_K=20"),
         os.path.join(os.path.dirname(emu.LIB), "libgcdt_emu_longcap.so"))


def segments(kind: str, n: int, c: int, seed: int = 5):
    """"online": many vertices on each segment.  Else n random points and c disjoint parallel segments of up to the square's
    side: rows, columns, or lines of slope 3 or 1/3 (steep, flat)."""
    rng = np.random.default_rng(seed)
    side = 1 << 20
    if kind == "online":
        # n points on each of c rows, which the segments run along, and as many anywhere
        at = (np.arange(c) * 2 + 1) * (side // (2 * c))
        x = np.sort(rng.permutation(side - 2)[:n] + 1)
        on = np.stack(np.meshgrid(x, at), 2).reshape(-1, 2)
        segs = np.stack([np.stack([np.zeros(c, int), at], 1), np.stack([np.full(c, side - 1), at], 1)], 1)
        xy, ids = gen.dedup(np.concatenate([rng.integers(0, side, (n, 2)), on, segs.reshape(-1, 2)]))
        return gen.to_grid(xy), ids[n + len(on):].reshape(-1, 2).astype(np.int32)
    pts = rng.integers(0, side, (n, 2))
    at = (np.arange(c) * 2 + 1) * (side // (2 * c))
    lo = rng.integers(0, side // 3, c)
    hi = rng.integers(side // 2, side - 1, c)
    if kind in ("rows", "columns"):
        a, b = np.stack([lo, at], 1), np.stack([hi, at], 1)
    else:
        # lines through (at, 0) before scaling, cut to the square
        lo, hi = lo // 3, hi // 3
        a, b = np.stack([at * 0.6 + lo, 3 * lo], 1), np.stack([at * 0.6 + hi, 3 * hi], 1)
    if kind in ("columns", "flat"):
        a, b = a[:, ::-1], b[:, ::-1]
    segs = np.stack([a, b], 1).astype(np.int64).clip(0, side - 1)
    # the same points twice over collinear ones: every other segment gets a vertex at its middle
    mid = segs[::2].sum(1)
    mid = mid[(mid % 2 == 0).all(1)] // 2
    xy, ids = gen.dedup(np.concatenate([pts, mid, segs.reshape(-1, 2)]))
    return gen.to_grid(xy), ids[n + len(mid):].reshape(-1, 2).astype(np.int32)


def check(g, cons, tris):
    v = O.validate(g, tris, cons)
    assert v["valid"], v
    if v["unique"]:
        ref, _ = O.cdt(g, cons)
        assert np.array_equal(O.canonical(tris), O.canonical(ref))


CASES = [("rows", 400, 3), ("rows", 5000, 40), ("columns", 5000, 40), ("steep", 3000, 25), ("flat", 3001, 25),
         ("columns", 60, 2),
         # more vertices on the segments than the first buffer holds; more than one wave sorts (1,024)
         ("online", 900, 3), ("online", 1100, 1)]


def emulated(lib, case, seed):
    code = ("import sys, numpy as np; from tests import test_long_segments as t; from tests.emu import emu; "
            f"g, c = t.segments(*{case!r}); tris, adj, _ = emu.solve(g, c); "
            "np.savez(sys.argv[1], tris=tris, adj=adj)")
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "o.npz")
        env = dict(os.environ, EMU_SEED=str(seed), EMU_CONC="8", EMU_YIELD_ATOMICS="1", EMU_LIB=lib)
        r = subprocess.run([sys.executable, "-c", code, out], cwd=ROOT, env=env, capture_output=True, text=True,
                           timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        z = np.load(out)
        return z["tris"], z["adj"]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}")
def test_every_cavity_path_gives_the_same_arrays(case):
    default, small = emu.build(), emu.build(SMALL)
    g, cons = segments(*case)
    tris, adj = emulated(default, case, 1)
    check(g, cons, tris)
    tris2, adj2 = emulated(small, case, 2)
    assert np.array_equal(tris, tris2) and np.array_equal(adj, adj2)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + [("rows", 200_000, 7), ("steep", 100_000, 1200), ("flat", 30_000, 3)],
                         ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}")
def test_long_segments_on_the_gpu(case):
    from gcdt_amd import solve
    g, cons = segments(*case)
    tris, _ = solve(g, cons)
    check(g, cons, tris)
    again, _ = solve(g, cons)
    assert np.array_equal(tris, again)
