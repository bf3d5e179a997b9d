"""Constraints that cross more than 2^30 triangles in one round between them."""
import numpy as np
import pytest

from gcdt_amd import gen
from gcdt_amd.api import DeviceBuffer, solve_device

pytestmark = pytest.mark.gpu


def test_copies_of_one_long_segment():
    """180,000 copies of a segment across 6,800 triangles: one of them wins and
    the others find its edge in the next round.  Their paths are 1.2e9 words."""
    n, copies = 10_000_000, 180_000
    rng = np.random.default_rng(6)
    side = 1 << 20
    ends = np.array([[500, side // 2], [side - 500, side // 2 + 1]])
    xy, ids = gen.dedup(np.concatenate([rng.integers(0, side, (n, 2)), ends]))
    g = gen.to_grid(xy)
    cons = np.ascontiguousarray(np.broadcast_to(ids[n:].astype(np.int32), (copies, 2)))
    dp, dc, dt = DeviceBuffer.from_array(g), DeviceBuffer.from_array(cons), DeviceBuffer(12 * (2 * len(g) + 2))
    try:
        _, st = solve_device(dp, len(g), dc, copies, dt)
        tris = dt.to_array(np.int32, (2 * len(g) + 2, 3))
        one = DeviceBuffer.from_array(cons[:1])
        _, st1 = solve_device(dp, len(g), one, 1, dt)
        assert np.array_equal(tris, dt.to_array(np.int32, (2 * len(g) + 2, 3)))
    finally:
        for b in (dp, dc, dt):
            b.free()
    assert st["constraint_rounds"] >= 1 and st["segments"] == copies * st1["segments"]
