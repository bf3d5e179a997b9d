"""Inputs packed into few cells: thousands of cells above the cap that one
workgroup sorts, among the points' cells and among the leaves'.  The arrays
must not depend on the order in which the atomics arrive."""
import os
import subprocess
import sys
import tempfile

import numpy as np
import pytest

from oracle import oracle as O
from tests.emu import emu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# a cell of more than two elements is sorted by a workgroup, of more than four
# by the merge of all such cells; any number of long pieces is many, and those of
# up to 24 triangles on average get a wave or a workgroup by their own size
# (test_cavity_sizes.py); all flip rounds below the tail threshold run in one
# workgroup (test_round_counts.py)
TINY = (("GCDT_CELL_RANK_MAX=2", "GCDT_CELL_BLOCK_MAX=4", "GCDT_CAV_WAVE_K=4", "GCDT_CAV_MID_K=24", "GCDT_CAV_LDS_K=30",
         "GCDT_CAV_FEW=0", "GCDT_FLIP_WG_LIST=4096"),
        os.path.join(os.path.dirname(emu.LIB), "libgcdt_emu_tinycap.so"))
NONE = np.zeros((0, 2), np.int32)


def packed(n, side, seed=4):
    """n distinct grid points in a square of `side` of the whole one's side."""
    rng = np.random.default_rng(seed)
    w = int(side * (1 << 30))
    lo = 1 << 20
    key = np.unique(rng.integers(0, w, n + n // 100) << 32 | rng.integers(0, w, n + n // 100))
    g = np.stack([key >> 32, key & 0xFFFFFFFF], 1) + lo
    return np.ascontiguousarray(rng.permutation(g)[:n].astype(np.int32))


def pieces(cells, each, seed=4):
    """`each` points in every cell of cells x cells of the 1024 x 1024 ones."""
    rng = np.random.default_rng(seed)
    x, y = np.meshgrid(np.arange(8, 8 + cells), np.arange(8, 8 + cells))
    base = np.repeat(np.stack([x.ravel(), y.ravel()], 1), each, 0) << 20
    g = np.unique(base + rng.integers(0, 1 << 20, base.shape), axis=0)
    return np.ascontiguousarray(rng.permutation(g).astype(np.int32))


CASES = {
    "points": lambda: pieces(64, 6),          # 4,096 cells of six points
    "leaves": lambda: packed(30_000, 0.354),  # about 8,200 of 65,536 leaf cells hold 60,002 leaves
}


def emulated(case, seed, conc):
    code = ("import sys, numpy as np; from tests import test_crowded_cells as t; from tests.emu import emu; "
            f"tris, adj, _ = emu.solve(t.CASES[{case!r}](), t.NONE); np.savez(sys.argv[1], tris=tris, adj=adj)")
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "o.npz")
        e = dict(os.environ, EMU_SEED=str(seed), EMU_CONC=str(conc), EMU_YIELD_ATOMICS="1", EMU_LIB=emu.build(TINY))
        r = subprocess.run([sys.executable, "-c", code, out], cwd=ROOT, env=e, capture_output=True, text=True,
                           timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        z = np.load(out)
        return z["tris"], z["adj"]


@pytest.mark.parametrize("case", list(CASES))
def test_arrays_do_not_depend_on_the_interleaving(case):
    tris, adj = emulated(case, 1, 1)
    v = O.validate(CASES[case](), tris, NONE)
    assert v["valid"], v
    for seed, conc in ((2, 8), (3, 16)):
        t, a = emulated(case, seed, conc)
        assert np.array_equal(tris, t) and np.array_equal(adj, a)


# 2,600 cells of 2,290 points; 2,800 leaf cells of 2,100 leaves
@pytest.mark.gpu
@pytest.mark.parametrize("n,side", [(6_000_000, 0.05), (3_000_000, 0.026)])
def test_thousands_of_crowded_cells_on_the_gpu(n, side):
    from gcdt_amd import solve
    g = packed(n, side)
    t1, _, a1 = solve(g, NONE, with_adj=True)
    t2, _, a2 = solve(g, NONE, with_adj=True)
    assert np.array_equal(t1, t2) and np.array_equal(a1, a2)
