"""The routes of the insertion and flip rounds: lists in LDS and in memory, tests
by edges and by triangles, settling beside relocation and before it, tails that
start from a launched round.  The route is chosen by list lengths alone, so an
emulator build with small caps sends the same inputs down the other routes and
must give the same arrays; on the GPU, sizes at the real caps must equal the
oracle's CDT and repeat bit for bit."""
import os
import subprocess
import sys
import tempfile

import numpy as np
import pytest

from gcdt_amd import gen
from oracle import oracle as O
from tests.emu import emu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SMALL = (("GCDT_INS_LIST=200", "GCDT_SHORT_MAX=16", "GCDT_FLIP_WG_LIST=64", "GCDT_FLIP_SHORT_MAX=300",
          "GCDT_INS_SPLIT_MAX=100"),
         os.path.join(os.path.dirname(emu.LIB), "libgcdt_emu_routes.so"))


def points(kind, n, seed=3):
    rng = np.random.default_rng(seed)
    if kind == "lattice":  # every point but the first few on an edge or a circle of others
        k = int(n ** 0.5)
        x, y = np.meshgrid(np.arange(k), np.arange(k))
        xy = np.stack([x.ravel(), y.ravel()], 1) * (1 << 12)
    elif kind == "cluster":  # nearly all in one sample cell: long chains of flips
        xy = np.concatenate([rng.normal(1 << 19, 300, (n, 2)).astype(int), rng.integers(0, 1 << 20, (9, 2))])
    else:
        xy = rng.integers(0, 1 << 20, (n, 2))
    xy, _ = gen.dedup(np.asarray(xy).clip(0, (1 << 20) - 1))
    return gen.to_grid(xy)


def emulated(lib, kind, n, seed, env):
    code = ("import sys, numpy as np; from tests import test_round_routes as t; from tests.emu import emu; "
            f"tris, adj, _ = emu.solve(t.points({kind!r}, {n}), np.zeros((0, 2), np.int32)); "
            "np.savez(sys.argv[1], tris=tris, adj=adj)")
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "o.npz")
        e = dict(os.environ, EMU_SEED=str(seed), EMU_CONC="8", EMU_YIELD_ATOMICS="1", EMU_LIB=lib, **env)
        r = subprocess.run([sys.executable, "-c", code, out], cwd=ROOT, env=e, capture_output=True, text=True,
                           timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        z = np.load(out)
        return z["tris"], z["adj"]


def check(g, tris):
    none = np.zeros((0, 2), np.int32)
    v = O.validate(g, tris, none)
    assert v["valid"], v
    if v["unique"]:
        ref, _ = O.cdt(g, none)
        assert np.array_equal(O.canonical(tris), O.canonical(ref))


# insertion rounds above the threshold are launched; flips have one tester above it
@pytest.mark.parametrize("threshold", [4096, 1024, 0])
@pytest.mark.parametrize("kind,n", [("uniform", 2), ("uniform", 199), ("uniform", 201), ("uniform", 2500),
                                    ("lattice", 1600), ("cluster", 1500)])
def test_every_route_gives_the_same_arrays(kind, n, threshold):
    env = {"GCDT_TAIL_THRESHOLD": str(threshold)}
    default, small = emu.build(), emu.build(SMALL)
    tris, adj = emulated(default, kind, n, 1, env)
    check(points(kind, n), tris)
    tris2, adj2 = emulated(small, kind, n, 2, env)
    assert np.array_equal(tris, tris2) and np.array_equal(adj, adj2)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [("uniform", 128), ("uniform", 129), ("uniform", 4095), ("uniform", 4097),
                                    ("uniform", 32_767), ("uniform", 200_000), ("lattice", 70_000),
                                    ("cluster", 40_000)])
def test_sizes_at_the_caps_on_the_gpu(kind, n):
    from gcdt_amd import solve
    g = points(kind, n)
    none = np.zeros((0, 2), np.int32)
    tris, _ = solve(g, none)
    check(g, tris)
    again, _ = solve(g, none)
    assert np.array_equal(tris, again)
