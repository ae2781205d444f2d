"""The general raster kernels' stencil table and depth compares against the
oracle, bit for bit: every op on failure, depth failure and passing, both faces
apart, partial and empty compare and write masks, references beyond 8 bits,
values that clamp and wrap, every depth compare (stored NaN included), one and
four samples, tiles of one wave and of four, blended or not."""
import ctypes

import numpy as np
import pytest

from oracle_runner import oracle_render
from swiftshader_amd import abi, runtime, scenes
from swiftshader_amd.scenes import DrawData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu

BLEND = (abi.BLEND_FACTOR_SRC_ALPHA, abi.BLEND_FACTOR_ONE_MINUS_SRC_ALPHA, abi.BLEND_OP_ADD) * 2
MASKS = [(0xFF, 0xFF), (0x3C, 0xA7), (0x07, 0x100FF), (0xFF, 0x00)]  # compare, write


def _scene(seed, **kw):
    rng = np.random.default_rng(seed)
    pos, _, col = scenes.screen_triangles(rng, 900, 61, 44, area_hi=400)
    return DrawData(width=61, height=44, positions=pos, colors=col, shader=abi.SHADER_INTERPOLATE, blend=BLEND,
                    has_stencil=True, stencil_test=1, **kw)


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("op", range(8))
def test_every_op_of_both_faces(op, samples):
    for k, (cmask, wmask) in enumerate(MASKS):
        front = dict(fail_op=op, depth_fail_op=(op + 3) % 8, pass_op=(op + 5) % 8, compare_op=(op + k) % 8,
                     compare_mask=cmask, write_mask=wmask, reference=0x104 + 3 * k)
        back = dict(fail_op=(op + 6) % 8, depth_fail_op=(op + 1) % 8, pass_op=op, compare_op=(5 - op + k) % 8,
                    compare_mask=wmask, write_mask=0xFF, reference=5 + 2 * k)
        draw = _scene(70 + op, samples=samples, front=front, back=back, blend_enable=k & 1, depth_test=k != 2,
                      depth_write=k != 2, clear_depth=0.6, depth_compare=abi.COMPARE_LESS_OR_EQUAL,
                      clear_stencil=(3, 254, 0, 5, 255, 7, 1, 250)[op])
        print(f"[stencil table] op {op} x{samples} masks {cmask:x} {wmask:x}", flush=True)
        _compare(f"op {op} x{samples} masks {cmask:x} {wmask:x}", oracle_render(draw), gpu_render(draw))


@pytest.mark.parametrize("clear_depth", [0.5, float("nan")])
@pytest.mark.parametrize("compare", range(8))
def test_depth_compares_with_stencil(compare, clear_depth):
    face = dict(fail_op=abi.STENCIL_OP_INVERT, depth_fail_op=abi.STENCIL_OP_INCREMENT_AND_WRAP,
                pass_op=abi.STENCIL_OP_DECREMENT_AND_CLAMP, compare_op=abi.COMPARE_NOT_EQUAL, compare_mask=0x0F,
                write_mask=0xFF, reference=9)
    for fmt in (abi.FORMAT_R8G8B8A8_UNORM, abi.FORMAT_B8G8R8A8_SRGB):
        draw = _scene(90 + compare, samples=4 if compare & 1 else 1, front=face, back=face, depth_compare=compare,
                      clear_depth=clear_depth, blend_enable=1, color_format=fmt)
        print(f"[stencil table] compare {compare} depth {clear_depth} format {fmt}", flush=True)
        _compare(f"compare {compare} depth {clear_depth} format {fmt}", oracle_render(draw), gpu_render(draw))


def test_tiles_of_one_wave_and_persistent_workgroups():
    """Smaller workgroups fill the table in more rounds; persistent ones again for each tile."""
    draw = _scene(99, blend_enable=1, clear_stencil=2,
                  front=dict(fail_op=3, depth_fail_op=4, pass_op=6, compare_op=4, compare_mask=0xFF, write_mask=0xFF,
                             reference=40),
                  back=dict(fail_op=5, depth_fail_op=2, pass_op=7, compare_op=1, compare_mask=0xFF, write_mask=0x7F,
                            reference=3))
    want = oracle_render(draw)
    lib, base = runtime.lib(), abi.Tuning()
    runtime.check(lib.swr_get_tuning(ctypes.byref(base)))
    try:
        for w, h, per in ((8, 8, 0xFFFFFFFF), (16, 8, 1), (16, 16, 1), (8, 8, 2)):
            print(f"[stencil table] tiles {w}x{h} workgroups {per}", flush=True)
            runtime.check(lib.swr_set_tuning(ctypes.byref(abi.Tuning(w, h, per))))
            _compare(f"tiles {w}x{h}", want, gpu_render(draw))
    finally:
        runtime.check(lib.swr_set_tuning(ctypes.byref(base)))
