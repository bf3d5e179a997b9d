"""gcdt_solve_noalloc takes or refuses an input by its array's size alone.  The
limit follows from the input (points, sample, segments, crowded cells, the cells
that the sample's triangles meet), whatever buffers the phases make do with; a
refused input is one that gcdt_solve solves."""
import numpy as np
import pytest

from gcdt_amd import gen
from oracle import oracle as O
from tests.emu import emu

SCRATCH = 6  # GCDT_ERR_SCRATCH
NONE = np.zeros((0, 2), np.int32)
# the largest inputs of each kind that the array has taken since it is there
DIAGONAL, LATTICE, ONE_CELL = 81, 816, 529_084


def diagonal(n):
    """n points evenly along a diagonal: with the square's corners, triangles
    whose bounding boxes are most of the square."""
    x = (np.arange(n) * 2 + 1) * ((1 << 30) // (2 * n))
    return np.stack([x, x], 1).astype(np.int32)


def lattice(k):
    i = np.arange(k) * ((1 << 20) // k)
    x, y = np.meshgrid(i, i)
    return gen.to_grid(np.stack([x.ravel(), y.ravel()], 1))


def one_cell(n):
    """n points on every other column and row of one of the 1024 x 1024 cells:
    a lattice of a width of 1,000, its last row unfinished."""
    i = np.arange(n)
    g = np.stack([i % 1000, i // 1000], 1) * 1024 + (512 << 20) + 7
    return g.astype(np.int32)


def statuses(solve, inputs):
    out = []
    for g in inputs:
        try:
            solve(g)
            out.append(0)
        except Exception as e:
            out.append(e.status)
    return out


def test_location_counts_the_cells_of_the_samples_triangles():
    emu.build()
    emu.check(emu.load().gcdt_pool_init(), "gcdt_pool_init")
    inputs = [diagonal(n) for n in (40, DIAGONAL, DIAGONAL + 1, 400)]
    assert statuses(lambda g: emu.solve(g, NONE, entry="gcdt_solve_noalloc"), inputs) == [0, 0, SCRATCH, SCRATCH]
    assert O.validate(inputs[3], emu.solve(inputs[3], NONE)[0], NONE)["valid"]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,most", [(diagonal, DIAGONAL), (lattice, LATTICE), (one_cell, ONE_CELL)],
                         ids=["diagonal", "lattice", "one_cell"])
def test_limit_on_the_gpu(kind, most):
    from gcdt_amd import solve
    from gcdt_amd.lib import check, lib
    from tests.test_zz_no_alloc import _run
    check(lib().gcdt_pool_init(), "gcdt_pool_init")
    inputs = [kind(most), kind(most + 1)]
    assert statuses(lambda g: _run(lib().gcdt_solve_noalloc, g, NONE), inputs) == [0, SCRATCH]
    solve(inputs[1])
