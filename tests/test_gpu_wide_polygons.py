"""Polygons with edges beyond 2047 pixels (28.4 extents above 32767), whose
half planes hold in the blocks that no such edge crosses, against the oracle,
bit for bit: triangles clipped to several vertices over wide and tall targets,
long lines of several widths, extents around the limit, one and four samples,
both windings, tiles past the known pair capacity."""
import numpy as np
import pytest

from oracle_runner import oracle_render
from swiftshader_amd import abi, runtime
from swiftshader_amd.scenes import DrawData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu

BLEND = (abi.BLEND_FACTOR_SRC_ALPHA, abi.BLEND_FACTOR_ONE_MINUS_SRC_ALPHA, abi.BLEND_OP_ADD) * 2
SIZES = [(4100, 21), (19, 4100), (2500, 90)]


def _draw(w, h, xy, **kw):
    """Triangles (lines) with the given clip-space xy and random depths and colours."""
    rng = np.random.default_rng(len(xy) + w)
    z = rng.uniform(0.05, 0.95, (len(xy), 1))
    pos = np.concatenate([xy, z, np.ones_like(z)], 1).astype(np.float32)
    return DrawData(width=w, height=h, positions=pos, colors=rng.uniform(0, 1, (len(xy), 4)).astype(np.float32),
                    shader=abi.SHADER_INTERPOLATE, blend_enable=1, blend=BLEND, **kw)


def _check(name, draw):
    print(f"[wide polygons] {name}", flush=True)
    _compare(name, oracle_render(draw), gpu_render(draw))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("size", SIZES)
def test_clipped_triangles(size, samples):
    """Vertices up to three times outside: three to seven vertices after clipping."""
    rng = np.random.default_rng(size[0] + samples)
    xy = rng.uniform(-3.0, 3.0, (120, 2))
    xy[:30] = rng.choice([-1.0, 1.0], (30, 2)) * rng.choice([1.0, 1.5], (30, 1))  # borders, corners and repeated vertices
    _check(f"clipped {size} x{samples}", _draw(*size, xy, samples=samples))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("width", [1.0, 7.0, 40.0])
@pytest.mark.parametrize("mode", [abi.LINE_RASTERIZATION_DEFAULT, abi.LINE_RASTERIZATION_RECTANGULAR])
def test_long_lines(mode, width, samples):
    rng = np.random.default_rng(int(width) + samples)
    xy = rng.uniform(-1.2, 1.2, (40, 2))
    xy[::2, 0] = rng.uniform(-1.1, -0.7, 20)
    xy[1::2, 0] = rng.uniform(0.7, 1.1, 20)
    _check(f"lines {width} mode {mode} x{samples}",
           _draw(3000, 60, xy, samples=samples, topology=abi.TOPOLOGY_LINE_LIST, line_width=width,
                 line_rasterization_mode=mode))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("extent", [32766, 32767, 32768, 32783])
def test_extents_around_the_limit(extent, samples):
    """Triangles and lines as wide as `extent` sixteenths of a pixel, to one sixteenth."""
    w, h, n = 2064, 37, 40
    rng = np.random.default_rng(extent + samples)
    x0 = rng.integers(0, 16 * w - extent, (n, 1))
    x = np.concatenate([x0, x0 + extent, x0 + rng.integers(0, extent, (n, 1))], 1) / 16.0
    y = rng.integers(0, 16 * h, (n, 3)) / 16.0
    flip = rng.random(n) < 0.5
    x[flip], y[flip] = x[flip][:, [1, 0, 2]], y[flip][:, [1, 0, 2]]
    xy = np.stack([2 * x / w - 1, 2 * y / h - 1], 2).reshape(-1, 2)
    _check(f"extent {extent} x{samples}", _draw(w, h, xy, samples=samples))


def test_past_the_known_capacity():
    rng = np.random.default_rng(12)
    draw = _draw(4100, 40, rng.uniform(-1.6, 1.6, (900, 2)))
    want = oracle_render(draw)
    runtime.check(runtime.lib().swr_release(), "swr_release")  # forget the learnt capacity
    gpu_render(_draw(16, 16, np.array([[-1, -1], [1, -1], [-1, 1]])))
    print("[wide polygons] past the capacity", flush=True)
    _compare("past the capacity", want, gpu_render(draw))
