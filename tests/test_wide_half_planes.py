"""The half planes of polygons with long edges, as the rasteriser evaluates
them over an 8x8 block (origin term in 64 bits clamped to +-2^30; an edge that
has the whole block on one side is a constant there or drops the polygon, a
short one takes steps by 16-bit products; the blocks that a long one crosses
are left to the spans), against the span rule with exact integers, on the CPU."""
import numpy as np
import pytest

from test_half_plane_coverage import convex, span_rule

SAMPLES = {1: [(0, 0)], 4: [(-2, -6), (6, -2), (-6, 2), (2, 6)]}


def block_rule(poly, d, ox, oy, sx, sy):
    """sx, sy: 28.4 offsets of the samples from the block's origin pixel.  None: left to the spans."""
    n, inside, spans = len(poly), np.full(sx.shape, 1 << 30), False
    for i in range(n):
        a, b = poly[i], poly[(i + 1) % n]
        (xa, ya), (xb, yb) = (a, b) if d else (b, a)
        dx, dy = xb - xa, yb - ya
        closed = dy > 0 or (dy == 0 and dx < 0)
        v = dy * (16 * ox - xa) - dx * (16 * oy - ya)
        f = max(-(1 << 30), min(1 << 30, v)) - (0 if closed else 1)
        reach = (abs(dx) + abs(dy)) * 128
        assert reach < 1 << 29
        if f < -reach:
            return np.zeros(sx.shape, bool)
        if f <= reach:
            spans |= max(abs(dx), abs(dy)) > 32767
            inside = np.minimum(inside, dy * sx - dx * sy + f)
    return None if spans else inside >= 0


@pytest.mark.parametrize("ms", [1, 4])
@pytest.mark.parametrize("n", [3, 4, 5])
@pytest.mark.parametrize("lim", [40000, 1 << 18, (1 << 20) - 1])
def test_blocks_along_the_edges(lim, n, ms):
    rng = np.random.default_rng(lim + 7 * n + ms)
    cx, cy = np.meshgrid(np.arange(8), np.arange(8))
    done, compared, left = 0, 0, 0
    while done < 40:
        a = np.sort(rng.uniform(0, 2 * np.pi, n))[::rng.choice([-1, 1])]
        r = lim * rng.uniform(0.5, 1.0)
        poly = [(int(r * np.cos(t)), int(r * np.sin(t))) for t in a]
        if rng.random() < 0.3:
            poly[1] = (poly[0][0], poly[1][1])  # a vertical edge
        if rng.random() < 0.3:
            poly[2] = (poly[2][0], poly[1][1])  # a horizontal one
        if n > 3 and not convex(poly):
            continue
        done += 1
        for _ in range(24):
            i, t = int(rng.integers(n)), rng.random()
            p, q = np.array(poly[i]), np.array(poly[(i + 1) % n])
            ox, oy = (int(v) // 128 * 8 for v in p + (q - p) * t + rng.integers(-200, 200, 2))
            for kx, ky in SAMPLES[ms]:
                sx, sy = 16 * cx + kx, 16 * cy + ky
                for d in (0, 1):
                    got = block_rule(poly, d, ox, oy, sx, sy)
                    left += got is None
                    if got is not None:
                        compared += 1
                        want = span_rule(poly, d, 16 * ox + sx, 16 * oy + sy)
                        assert np.array_equal(want, got), (poly, d, ox, oy)
    assert compared > 100 and left > 100
