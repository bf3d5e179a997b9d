"""The pool's peak of a batch stays within what the server admits it by, also
for small instances, nearly all of whose points are in their samples."""
import ctypes

import pytest

from gcdt_amd import gen
from gcdt_amd.api import DeviceBuffer, pack_instances, solve_batch_device
from gcdt_amd.lib import check, lib
from gcdt_amd.serve import batch_footprint

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,n", [(1000, 16), (1000, 100), (500, 250), (3000, 60), (64, 2000)])
def test_batch_peak_within_its_footprint(count, n):
    some = []
    for i in range(64):
        p, c = gen.polygon_instance(gen.Stream(i + 1), n)
        some.append((gen.to_grid(p), c))
    inst = [some[i % 64] for i in range(count)]
    pts, poff, cons, coff, toff = pack_instances(inst)
    dp, dc, dt = DeviceBuffer.from_array(pts), DeviceBuffer.from_array(cons), DeviceBuffer(12 * int(toff[-1]))
    in_use, cached, peak = (ctypes.c_size_t(0) for _ in range(3))
    check(lib().gcdt_pool_reset_peak(), "gcdt_pool_reset_peak")
    check(lib().gcdt_pool_stats(ctypes.byref(in_use), ctypes.byref(cached), ctypes.byref(peak)), "gcdt_pool_stats")
    own = sum(b.nbytes for b in (dp, dc, dt))
    before = in_use.value
    solve_batch_device(dp, poff, dc, coff, dt)
    check(lib().gcdt_pool_stats(ctypes.byref(in_use), ctypes.byref(cached), ctypes.byref(peak)), "gcdt_pool_stats")
    for b in (dp, dc, dt):
        b.free()
    assert peak.value - before + own <= batch_footprint([len(g) for g, _ in inst])
