"""The double filters of the crossing pass: over rational points of every
spread -- the whole grid, neighbouring cells, crossings that coincide or lie on
one line or circle -- a filter gives the exact sign or 0, and it settles nearly
all points in general position.  The exact determinants are held to Python's
integers on the same points."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host_filters.cpp")
LIB = os.path.join(HERE, "libhost_filters.so")
GRID = (1 << 30) - 1


@pytest.fixture(scope="module")
def lib():
    cmd = [os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-fPIC", "-shared", "--offload-arch=gfx950", "-Xclang",
           "-target-feature", "-Xclang", "-packed-fp32-ops", "-o", LIB, SRC]
    subprocess.run(cmd, check=True, capture_output=True)
    return ctypes.CDLL(LIB)


def crossing(P1, P2, Q1, Q2):
    """The crossing of two lines in homogeneous integers, W > 0; None if parallel."""
    dx, dy, ex, ey = P2[0] - P1[0], P2[1] - P1[1], Q2[0] - Q1[0], Q2[1] - Q1[1]
    W = dx * ey - dy * ex
    if W == 0:
        return None
    t = (Q1[0] - P1[0]) * ey - (Q1[1] - P1[1]) * ex
    X, Y = P1[0] * W + dx * t, P1[1] * W + dy * t
    if W < 0:
        X, Y, W = -X, -Y, -W
    return (X, Y, W) if 0 <= X <= GRID * W and 0 <= Y <= GRID * W else None


def sgn(v):
    return (v > 0) - (v < 0)


def orient(p, q, r):
    return sgn((p[0] * r[2] - r[0] * p[2]) * (q[1] * r[2] - r[1] * q[2])
               - (p[1] * r[2] - r[1] * p[2]) * (q[0] * r[2] - r[0] * q[2]))


def incircle(a, b, c, d):
    rows = []
    for p in (a, b, c):
        x, y = p[0] * d[2] - d[0] * p[2], p[1] * d[2] - d[1] * p[2]
        w = p[2] * d[2]
        rows.append((x * w, y * w, x * x + y * y))
    (ax, ay, al), (bx, by, bl), (cx, cy, cl) = rows
    return sgn(al * (bx * cy - by * cx) + bl * (cx * ay - cy * ax) + cl * (ax * by - ay * bx))


def points(rng, kind, span):
    """Four points of one item."""
    base = [rng.randrange(0, GRID - span + 1) for _ in range(2)]

    def g():
        return (base[0] + rng.randrange(span + 1), base[1] + rng.randrange(span + 1))

    def x():
        while True:
            c = crossing(g(), g(), g(), g())
            if c:
                return c

    if kind == "grid":
        return [g() + (1,) for _ in range(4)]
    if kind == "crossings":
        return [x() if rng.random() < 0.7 else g() + (1,) for _ in range(4)]
    if kind == "one line":
        a, b = g(), g()
        while a == b:
            b = g()
        out = [a + (1,), b + (1,)]
        while len(out) < 4:
            c = crossing(a, b, g(), g())
            if c:
                out.append(c)
        rng.shuffle(out)
        return out
    if kind == "one circle":
        (px, py), r, s = g(), rng.randrange(1, span + 1), rng.randrange(1, span + 1)
        q = [(px, py), (px + r, py), (px + r, py + s), (px, py + s)]
        q = [(min(u, GRID), min(v, GRID), 1) for u, v in q]
        rng.shuffle(q)
        return q
    p = x()  # "coincident"
    return [p, p, x(), g() + (1,)]


@pytest.mark.parametrize("span", [1, 7, 1 << 10, 1 << 20, GRID])
@pytest.mark.parametrize("kind", ["grid", "crossings", "one line", "one circle", "coincident"])
def test_filter_is_exact_or_open(lib, kind, span):
    rng = random.Random(len(kind) * 1000003 + span)
    n = 400
    items = [points(rng, kind, span) for _ in range(n)]
    w = np.zeros((n, 4, 5), np.uint64)
    for i, it in enumerate(items):
        for j, (X, Y, W) in enumerate(it):
            w[i, j] = [X & (2**64 - 1), X >> 64, Y & (2**64 - 1), Y >> 64, W]
    out = np.zeros((n, 4), np.int32)
    lib.host_filters(w.ctypes.data_as(ctypes.c_void_p), n, out.ctypes.data_as(ctypes.c_void_p))
    for it, (of, oe, cf, ce) in zip(items, out.tolist()):
        assert oe == orient(*it[:3]) and ce == incircle(*it)
        assert of in (0, oe) and cf in (0, ce)
    if kind in ("grid", "crossings") and span >= 1 << 20:
        assert np.mean(out[:, 0] == out[:, 1]) > 0.95 and np.mean(out[:, 2] == out[:, 3]) > 0.9
