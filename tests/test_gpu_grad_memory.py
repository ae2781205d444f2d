"""Device memory of a plan's gradient records: one 64-byte slot (record and
sort keys) per sample, and what the last reservations of the waves of its own
gather launches can leave unused, 4 waves of at most 512 slots for each
16x16-pixel block."""
import numpy as np
import pytest
import torch

from swiftshader_amd import abi, scenes, texfit
from swiftshader_amd.scenes import TextureData

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("samples", [(1,), (4,), (1, 4)])
def test_small_plans_take_memory_for_their_own_launches(samples):
    rng = np.random.default_rng(8)
    draws, slots = [], 0
    for s in samples:
        pos, uv, col = scenes.screen_triangles(rng, 100, 64, 48, area_hi=300)
        draws.append(scenes.DrawData(width=64, height=48, positions=pos, colors=col, texcoords=uv, samples=s,
                                     shader=abi.SHADER_MODULATE, color_format=abi.FORMAT_R32G32B32A32_SFLOAT,
                                     texture=TextureData(format=abi.FORMAT_R32G32B32A32_SFLOAT, levels=[])))
        slots += 64 * 48 * s + 4 * 3 * 4 * 512
    fit = texfit.MultiViewFit(draws, torch.rand((64, 64, 4)), [torch.zeros((48, 64, 4))] * len(draws),
                              geometry_grads=False, device=DEV)
    fit.step_batched(update=False)  # loads every kernel; the plan is made anew below
    fit.plan.close()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    fit.make_plan()
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    # Besides the slots: pair lists, tables and the allocator's granularity (2 MiB for each of some 30 buffers).
    limit = 64 * slots + (64 << 20)
    print(f"[grad memory] samples {samples}: {used >> 20} MiB, at most {limit >> 20}", flush=True)
    assert used <= limit
