"""Mip chains around the size (4096 texels) from which one launch takes the rest
of the levels: the box filter bit-exact with the generator, its adjoint against
FP64 (each texel adds two float products to at most 14 levels' sums: within
32 * 2^-24 of the largest value)."""
import ctypes

import numpy as np
import pytest
import torch

from grad_cases import G
from swiftshader_amd import abi, diff, runtime, scenes

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPES = [(1, 1), (2, 1), (63, 65), (64, 64), (64, 65), (1, 4096), (1, 4097), (130, 67), (257, 128), (5000, 3)]


@pytest.mark.parametrize("u8", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_chain_is_bit_exact(shape, u8):
    rng = np.random.default_rng(shape[0] + 7 * shape[1])
    lvl0 = rng.integers(0, 256, shape + (4,), dtype=np.uint8) if u8 else rng.normal(0.5, 0.2, shape + (4,)).astype(np.float32)
    want = scenes.box_mip_chain(lvl0)
    levels = [torch.from_numpy(lvl0).to(DEV)] + [torch.zeros(w.shape, dtype=torch.uint8 if u8 else torch.float32, device=DEV)
                                                 for w in want[1:]]
    print(f"[mip tail] down {shape} u8 {u8}", flush=True)
    diff.generate_mips(levels)
    torch.cuda.synchronize()
    for a, b in zip(levels, want):
        assert np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("shape", SHAPES)
def test_adjoint(shape):
    rng = np.random.default_rng(shape[0] + 11 * shape[1])
    gs = [rng.normal(size=l.shape).astype(np.float32) for l in G.box_chain(np.zeros(shape + (4,)))]
    bufs = [torch.from_numpy(g).to(DEV) for g in gs]
    t = diff._texture_struct(bufs, abi.FORMAT_R32G32B32A32_SFLOAT)
    print(f"[mip tail] up {shape}", flush=True)
    runtime.check(runtime.lib().swr_mip_backward(ctypes.byref(t), runtime._stream_handle(None)))
    torch.cuda.synchronize()
    want = G.box_chain_adjoint([g.astype(np.float64) for g in gs])
    assert np.max(np.abs(bufs[0].cpu().numpy() - want)) <= 32 * 2.0**-24 * max(1.0, np.abs(want).max())
