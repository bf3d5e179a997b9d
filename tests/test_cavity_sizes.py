"""Rounds with many long pieces: the smaller cavities by a wave each and the
larger ones by a workgroup, or all of them by workgroups, as the pieces' number
and average length say.  Every choice must give the same arrays."""
import numpy as np
import pytest

from tests.emu import emu
from tests.test_crowded_cells import TINY
from tests.test_long_segments import check, emulated, segments


@pytest.mark.parametrize("case", [("rows", 300, 8), ("columns", 400, 8), ("steep", 500, 9), ("rows", 2000, 12)],
                         ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}")
def test_both_sizes_give_the_default_arrays(case):
    default, both = emu.build(), emu.build(TINY)
    g, cons = segments(*case)
    tris, adj = emulated(default, case, 1)
    check(g, cons, tris)
    tris2, adj2 = emulated(both, case, 2)
    assert np.array_equal(tris, tris2) and np.array_equal(adj, adj2)


# 1,500 long pieces of about 90 and 400 triangles
@pytest.mark.gpu
@pytest.mark.parametrize("case", [("rows", 12_000, 1500), ("rows", 300_000, 1500)],
                         ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}")
def test_many_long_segments_on_the_gpu(case):
    from gcdt_amd import solve
    g, cons = segments(*case)
    tris, _, adj = solve(g, cons, with_adj=True)
    check(g, cons, tris)
    again, _, adj2 = solve(g, cons, with_adj=True)
    assert np.array_equal(tris, again) and np.array_equal(adj, adj2)
