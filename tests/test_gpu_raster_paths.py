"""The rasteriser's coverage and shading paths where they can go wrong, against
the oracle, bit for bit: clipped polygons (triangles over the target's edges
and corners), triangles wider than the 16-bit edge extents, wide lines and
points over the corners, targets that end inside a block; unblended draws
with every kind of colour mask, several primitives in one pixel's samples,
and depth compares with and without hierarchical depth."""
import dataclasses

import numpy as np
import pytest

from oracle_runner import oracle_render
from swiftshader_amd import abi, scenes
from swiftshader_amd.scenes import DrawData, TextureData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu


def _check(name, draw):
    print(f"[raster paths] {name}", flush=True)
    _compare(name, oracle_render(draw), gpu_render(draw))


def _edge_triangles(w, h, n, area_hi, seed, **kw):
    """Triangles centred on the target's borders and corners."""
    rng = np.random.default_rng(seed)
    pos, _, col = scenes.screen_triangles(rng, n, w, h, area_hi=area_hi)
    p = pos.reshape(n, 3, 4)
    c = (p[..., :2] / p[..., 3:]).mean(1)
    shift = np.where(np.abs(c) == np.abs(c).max(1, keepdims=True), np.sign(c) - c, 0.0)
    shift[: n // 4] = np.sign(c[: n // 4]) - c[: n // 4]  # a quarter on the corners
    p[..., :2] += (shift[:, None, :] * p[..., 3:]).astype(np.float32)
    return DrawData(width=w, height=h, positions=pos, colors=col, shader=abi.SHADER_INTERPOLATE, **kw)


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("size,area", [((8, 8), 40), ((61, 35), 900), ((130, 9), 400), ((17, 97), 3000)])
def test_clipped_polygons(size, area, samples):
    _check(f"clipped {size} x{samples}", _edge_triangles(*size, 400, area, 31 + size[0], samples=samples))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("size", [(2047, 24), (2048, 24), (2300, 17), (24, 2300)])
def test_triangles_wider_than_the_edge_extents(size, samples):
    """Unclipped triangles as wide (high) as the target, and clipped ones."""
    w, h = size
    rng = np.random.default_rng(w + samples)
    xy = rng.uniform(-1.0, 1.0, (30 * 3, 2))
    xy[::2, int(w < h)] = rng.choice([-1.0, 1.0], 45)
    xy[60:] *= 1.3
    z = rng.uniform(0.0, 1.0, (90, 1))
    pos = np.concatenate([xy, z, np.ones((90, 1))], 1).astype(np.float32)
    col = rng.uniform(0.0, 1.0, (90, 4)).astype(np.float32)
    _check(f"wide {size} x{samples}", DrawData(width=w, height=h, positions=pos, colors=col, samples=samples,
                                                shader=abi.SHADER_INTERPOLATE))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("topology", [abi.TOPOLOGY_LINE_LIST, abi.TOPOLOGY_POINT_LIST])
def test_lines_and_points_over_the_borders(topology, samples):
    rng = np.random.default_rng(77 + topology)
    n = 240
    pos = np.concatenate([rng.uniform(-1.15, 1.15, (n, 2)), rng.uniform(0, 1, (n, 1)), np.ones((n, 1))], 1)
    pos[::3, 0] = np.sign(pos[::3, 0])
    col = rng.uniform(0, 1, (n, 4)).astype(np.float32)
    _check(f"topology {topology} x{samples}",
           DrawData(width=75, height=43, positions=pos.astype(np.float32), colors=col, samples=samples,
                    shader=abi.SHADER_INTERPOLATE, topology=topology, line_width=3.0,
                    point_sizes=rng.uniform(1.0, 30.0, n).astype(np.float32)))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("fmt", [abi.FORMAT_R8G8B8A8_UNORM, abi.FORMAT_B8G8R8A8_UNORM, abi.FORMAT_B8G8R8A8_SRGB,
                                 abi.FORMAT_R32G32B32A32_SFLOAT])
@pytest.mark.parametrize("mask", [0x0, 0x5, 0xE, 0xF])
def test_unblended_colour_masks(fmt, mask, samples):
    """Small triangles, so that a pixel's samples have several last writers,
    over a cleared target whose masked channels must stay."""
    rng = np.random.default_rng(mask + samples)
    tex = TextureData(format=abi.FORMAT_R8G8B8A8_UNORM,
                      levels=scenes.box_mip_chain(scenes.noise_texture_rgba8(rng, 32)))
    pos, uv, col = scenes.screen_triangles(rng, 900, 45, 29, area_hi=60)
    _check(f"mask {mask:x} format {fmt} x{samples}",
           DrawData(width=45, height=29, positions=pos, colors=col, texcoords=uv, samples=samples, color_format=fmt,
                    shader=abi.SHADER_MODULATE, texture=tex, color_write_mask=mask,
                    clear_color=(0.25, 0.5, 0.75, 0.125)))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("blend", [0, 1])
@pytest.mark.parametrize("compare", range(8))
def test_depth_compares_in_deep_blocks(compare, blend, samples):
    """About 60 layers: the hierarchical depth bound is re-tested many times
    in a block (LESS, LESS_OR_EQUAL), or never."""
    base = scenes.textured_1080p(seed=50 + compare, triangles=700, width=50, height=34, tex_size=32)
    draw = dataclasses.replace(base, depth_compare=compare, blend_enable=blend, samples=samples, clear_depth=0.5)
    _check(f"compare {compare} blend {blend} x{samples}", draw)
