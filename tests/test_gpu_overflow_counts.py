"""Occlusion counts of draws whose tiles render in two passes (the pairs that
fit the known capacity, then the primitives past it), against the oracle.

A workgroup sums its waves' counters after each pass.  The scissor leaves
some 8x8 blocks of the border tiles without work, so that their waves reach
the second pass's sum while the first one's is still being read: a count is
exact only if the passes are kept apart.
"""
import numpy as np
import pytest
import torch

from oracle_runner import oracle_render
from swiftshader_amd import abi, runtime, scenes
from swiftshader_amd.scenes import DrawData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu

BLEND = (abi.BLEND_FACTOR_SRC_ALPHA, abi.BLEND_FACTOR_ONE_MINUS_SRC_ALPHA, abi.BLEND_OP_ADD) * 2


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("blend", [0, 1])
def test_counts_of_both_passes(blend, samples):
    rng = np.random.default_rng(61 + samples)
    w, h = 200, 136
    pos, _, col = scenes.screen_triangles(rng, 3000, w, h, area_lo=30.0, area_hi=900.0)
    big = DrawData(width=w, height=h, positions=pos, colors=col, samples=samples, shader=abi.SHADER_INTERPOLATE,
                   depth_compare=abi.COMPARE_ALWAYS, blend_enable=blend, blend=BLEND, scissor=(24, 9, 155, 106))
    small = DrawData(width=16, height=16, positions=pos[:3], colors=col[:3], shader=abi.SHADER_INTERPOLATE)
    want = oracle_render(big)
    runtime.check(runtime.lib().swr_release(), "swr_release")  # forget the learnt capacity
    gpu_render(small)  # leaves a capacity of about a thousand pairs
    print(f"[overflow counts] blend {blend} x{samples}", flush=True)
    _compare("past the capacity", want, gpu_render(big))
    torch.cuda.synchronize()
    _compare("capacity grown", want, gpu_render(big))
