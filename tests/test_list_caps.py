"""Lists of exactly the lengths at which the rounds change their route, and one
more: insertion lists of 4,096 (held in LDS) and 131,072 points (settled beside
the relocation), flip lists of 256 (held in LDS), 1,024 (one workgroup) and
65,536 triangles (tested by edges).  The arrays are those of the emulator, whose
small-cap builds give the same on every route, bit for bit."""
import hashlib

import numpy as np
import pytest

from gcdt_amd import gen
from oracle import dropin as D
from oracle import oracle as O
from tests.emu import emu

NONE = np.zeros((0, 2), np.int32)


def uniform(n):
    """n points: 2 n + 2 triangles to flip."""
    xy, _ = gen.dedup(np.random.default_rng(17).integers(0, 1 << 20, (n + 4, 2)))
    return gen.to_grid(xy[:n])


def cells(side, each, more):
    """`each` points in every cell of side x side of the 256 x 256 sample cells
    and `more` others: side^2 sample points, the rest inserted after them."""
    rng = np.random.default_rng(23)
    x, y = np.meshgrid(np.arange(side), np.arange(side))
    at = np.repeat(np.stack([x.ravel(), y.ravel()], 1) * (256 // side), each, 0)
    at = np.concatenate([at, at[:more]])
    off = rng.choice(1 << 24, len(at), replace=False) if each > 1 else rng.integers(0, 1 << 24, len(at))
    return gen.to_grid(rng.permutation((at << 12) + np.stack([off >> 12, off & 4095], 1)))


# inputs whose lists have the length that is named, and the digest of triangles and neighbours
CASES = {
    "insert_4096": (lambda: cells(64, 1, 0), "af80195eebe0171c"),
    "insert_4097": (lambda: np.concatenate([cells(64, 1, 0), np.array([[(3 << 22) + 9, 5]], np.int32)]), "88db8b1554675df9"),
    "insert_131072": (lambda: cells(64, 33, 0), "fe00deb7b52f2e6b"),
    "insert_131073": (lambda: cells(64, 33, 1), "6de022ded058fb34"),
    "flip_256": (lambda: uniform(127), "bb06959abc8b5399"),
    "flip_258": (lambda: uniform(128), "c150dd9030ebe393"),
    "flip_1024": (lambda: uniform(511), "97b5f1c22bf3f315"),
    "flip_1026": (lambda: uniform(512), "144440f7604e9521"),
    "flip_65536": (lambda: uniform(32_767), "d2a38020c71a65dc"),
    "flip_65538": (lambda: uniform(32_768), "8d322d5e2b1c1670"),
}


def digest(tris, adj):
    return hashlib.sha256(np.ascontiguousarray(tris).tobytes() + np.ascontiguousarray(adj).tobytes()).hexdigest()[:16]


def check(g, tris, adj):
    v = O.validate(g, tris, NONE)
    assert v["valid"], v
    if v["unique"]:
        ref, _ = O.cdt(g, NONE)
        assert np.array_equal(O.canonical(tris), O.canonical(ref))
    assert D.adj_violations(O.with_corners(g), tris, adj) == []


@pytest.mark.parametrize("case", [k for k in CASES if "131" not in k and "655" not in k])
def test_emulated(case):
    emu.build()
    g = CASES[case][0]()
    tris, adj, _ = emu.solve(g, NONE)
    check(g, tris, adj)
    assert digest(tris, adj) == CASES[case][1]


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_on_the_gpu(case):
    from gcdt_amd import solve
    g = CASES[case][0]()
    tris, _, adj = solve(g, NONE, with_adj=True)
    check(g, tris, adj)
    assert digest(tris, adj) == CASES[case][1]
