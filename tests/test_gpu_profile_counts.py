"""The profile's count of fragments that passed every test, blended or not:
with one sample it is the draw's occlusion count."""
import numpy as np
import pytest

from oracle_runner import oracle_render
from swiftshader_amd import abi, runtime, scenes
from swiftshader_amd.scenes import DrawData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stencil", [0, 1])
@pytest.mark.parametrize("blend", [0, 1])
def test_passing_fragments_are_counted(blend, stencil):
    rng = np.random.default_rng(90)
    pos, _, col = scenes.screen_triangles(rng, 1500, 150, 90, area_hi=700)
    op = dict(compare_op=abi.COMPARE_GREATER_OR_EQUAL, pass_op=abi.STENCIL_OP_INCREMENT_AND_CLAMP, reference=3,
              compare_mask=0xFF, write_mask=0xFF)
    draw = DrawData(width=150, height=90, positions=pos, colors=col, shader=abi.SHADER_INTERPOLATE,
                    blend_enable=blend, has_stencil=bool(stencil), stencil_test=stencil, front=op, back=op,
                    blend=(abi.BLEND_FACTOR_SRC_ALPHA, abi.BLEND_FACTOR_ONE_MINUS_SRC_ALPHA, abi.BLEND_OP_ADD) * 2)
    want = oracle_render(draw)
    print(f"[profile counts] blend {blend} stencil {stencil}", flush=True)
    runtime.profile_read()
    runtime.profile_enable(True)
    try:
        _compare("profiled", want, gpu_render(draw))
        prof = runtime.profile_read()
    finally:
        runtime.profile_enable(False)
    assert prof["shaded"] == want[3] > 0
    assert prof["block_covers"] <= prof["block_tests"]
