"""The half-plane form of the coverage rule against the span rule, on the CPU.

The rasteriser evaluates convex polygons as half planes and the rest by the
reference's spans (src/Pipeline/SetupRoutine.cpp:550-621).  Here both rules,
and the predicate that picks between them, are written out over integers and
compared at every sample point around random polygons: triangles of every
kind, and polygons of 4 and 5 vertices that the predicate accepts."""
import numpy as np
import pytest


def span_rule(poly, d, x, y):
    n = len(poly)
    left = np.zeros(x.shape, bool)
    right = np.zeros(x.shape, bool)
    for i in range(n):
        (xa, ya), (xb, yb) = poly[(i + 1 - d) % n], poly[(i + d) % n]
        swap = yb < ya
        x1, y1, x2, y2 = (xb, yb, xa, ya) if swap else (xa, ya, xb, yb)
        e = (y2 - y1) * (x - x1) - (x2 - x1) * (y - y1)
        rows = (y1 <= y) & (y < y2)
        if swap:
            right = np.where(rows, e < 0, right)
        else:
            left = np.where(rows, e >= 0, left)
    return left & right


def half_plane_rule(poly, d, x, y):
    n = len(poly)
    inside = np.ones(x.shape, bool)
    for i in range(n):
        a, b = poly[i], poly[(i + 1) % n]
        (xa, ya), (xb, yb) = (a, b) if d else (b, a)
        dx, dy = xb - xa, yb - ya
        closed = dy > 0 or (dy == 0 and dx < 0)
        inside &= dy * (x - xa) - dx * (y - ya) - (0 if closed else 1) >= 0
    return inside


def convex(poly):
    n = len(poly)
    left = right = back = False
    dirs = []
    for i in range(n):
        p, q, r = poly[i - 1], poly[i], poly[(i + 1) % n]
        dx0, dy0, dx1, dy1 = q[0] - p[0], q[1] - p[1], r[0] - q[0], r[1] - q[1]
        c = dx0 * dy1 - dy0 * dx1
        left |= c > 0
        right |= c < 0
        back |= c == 0 and dx0 * dx1 + dy0 * dy1 <= 0
        if dy1:
            dirs.append(dy1 > 0)
    changes = sum(dirs[k] != dirs[k - 1] for k in range(len(dirs)))
    return not (left and right) and not back and changes == 2


def points(poly):
    p = np.array(poly)
    lo, hi = p.min(0) - 2, p.max(0) + 3
    return np.meshgrid(np.arange(lo[0], hi[0]), np.arange(lo[1], hi[1]))


@pytest.mark.parametrize("span", [3, 6, 40])
def test_every_triangle(span):
    rng = np.random.default_rng(span)
    for _ in range(1500):
        tri = [tuple(int(v) for v in rng.integers(0, span, 2)) for _ in range(3)]
        x, y = points(tri)
        for d in (0, 1):
            assert np.array_equal(span_rule(tri, d, x, y), half_plane_rule(tri, d, x, y)), (tri, d)


@pytest.mark.parametrize("n,span", [(4, 4), (4, 9), (4, 60), (5, 5), (5, 12), (5, 60)])
def test_accepted_polygons(n, span):
    rng = np.random.default_rng(100 * n + span)
    accepted = 0
    while accepted < 300:
        if rng.integers(0, 2):  # any vertices, in any order
            poly = [tuple(int(v) for v in rng.integers(0, span, 2)) for _ in range(n)]
        else:  # on a circle, rounded: convex or nearly so, either way round
            a = np.sort(rng.uniform(0, 2 * np.pi, n))[::rng.choice([-1, 1])]
            poly = [(int(round(span * np.cos(t) / 2)), int(round(span * np.sin(t) / 2))) for t in a]
        if not convex(poly):
            continue
        accepted += 1
        x, y = points(poly)
        for d in (0, 1):
            assert np.array_equal(span_rule(poly, d, x, y), half_plane_rule(poly, d, x, y)), (poly, d)


@pytest.mark.parametrize("poly", [
    [(0, 0), (0, 0), (8, 0), (8, 8)],             # a repeated vertex
    [(0, 0), (8, 0), (4, 0), (4, 8)],             # back along an edge
    [(0, 0), (8, 0), (4, 2), (4, 8)],             # a reflex corner
    [(0, 8), (6, 0), (12, 8), (0, 4), (12, 4)],   # a star: two revolutions
    [(0, 0), (4, 4), (8, 8), (4, 4)],             # no area
])
def test_rejected_polygons(poly):
    assert not convex(poly)
