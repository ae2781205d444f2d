"""The binned texel scatter of a batched backward against the per-view one.

Textures from one texel a side to sizes just around the scatter's 32-texel
tiles, wrapping and clamped, linear and point sampled, with and without
anisotropic probes, with and without vertex gradients; coordinates reach
beyond [0, 1], so footprints cross tile and level borders.

Both sides add the same float products up to order: the per-view side in
float, n of them to a texel one after the other at worst (n: fragments per
texel of the finest level, times up to 16 probes), all of one sign (the
targets are zero and everything sampled is positive).  A random walk of n
roundings stays within 4 * sqrt(n) * 2^-24 of the sum; the products
themselves, and the batched side's sums of rounded partial sums, take a few
more: 1e-6.
"""
import numpy as np
import pytest
import torch

from grad_cases import gradient_rel_error
from swiftshader_amd import abi, scenes, texfit
from swiftshader_amd.scenes import TextureData

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [  # (width, height), address mode, filter, anisotropic, samples, vertex gradients
    ((1, 1), abi.ADDRESS_REPEAT, abi.FILTER_LINEAR, False, 1, True),
    ((2, 33), abi.ADDRESS_REPEAT, abi.FILTER_LINEAR, True, 4, False),
    ((31, 32), abi.ADDRESS_CLAMP_TO_EDGE, abi.FILTER_LINEAR, False, 1, False),
    ((33, 65), abi.ADDRESS_CLAMP_TO_EDGE, abi.FILTER_LINEAR, True, 4, True),
    ((44, 45), abi.ADDRESS_REPEAT, abi.FILTER_NEAREST, False, 4, False),
    ((96, 100), abi.ADDRESS_REPEAT, abi.FILTER_LINEAR, True, 1, False),
    ((96, 3), abi.ADDRESS_CLAMP_TO_EDGE, abi.FILTER_NEAREST, False, 1, True),
]


def _levels(rng, w, h):
    levels = []
    while True:
        levels.append(rng.uniform(0.25, 1.0, (h, w, 4)).astype(np.float32))
        if w == 1 and h == 1:
            return levels
        w, h = max(1, w // 2), max(1, h // 2)


@pytest.mark.parametrize("size,mode,filt,aniso,samples,geometry", CASES)
def test_binned_scatter_matches_per_view(size, mode, filt, aniso, samples, geometry):
    rng = np.random.default_rng(size[0] * 131 + size[1])
    levels = _levels(rng, *size)
    tex = TextureData(format=abi.FORMAT_R32G32B32A32_SFLOAT, levels=levels, mag_filter=filt, min_filter=filt,
                      address_u=mode, address_v=mode, anisotropy_enable=1 if aniso else 0,
                      max_anisotropy=8.0 if aniso else 1.0)
    draws = []
    for w, h in ((96, 80), (70, 61), (128, 33)):
        pos, uv, col = scenes.screen_triangles(rng, 300, w, h, area_hi=400)
        uv = ((uv - 0.5) * 3.0).astype(np.float32)
        draws.append(scenes.DrawData(width=w, height=h, positions=pos, colors=np.abs(col).astype(np.float32) + 0.1,
                                     texcoords=uv, samples=samples, shader=abi.SHADER_MODULATE, texture=tex,
                                     color_format=abi.FORMAT_R32G32B32A32_SFLOAT))
    zeros = [torch.zeros((d.height, d.width, 4)) for d in draws]
    print(f"[gpu tap scatter] {size} mode {mode} filter {filt} aniso {aniso} x{samples} geometry {geometry}", flush=True)
    fit = texfit.MultiViewFit(draws, torch.from_numpy(levels[0]), zeros, geometry_grads=geometry, device=DEV)

    def grads():
        out = [l.detach().cpu().numpy().copy() for l in fit.d_levels]
        if geometry:
            for vb in fit.views:
                out += [vb.d_pos.cpu().numpy().copy(), vb.d_col.cpu().numpy().copy(), vb.d_uv.cpu().numpy().copy()]
        return out

    fit.step_plain(update=False)
    torch.cuda.synchronize()
    want = grads()
    fit.step_batched(update=False)
    torch.cuda.synchronize()
    got = grads()
    fragments = sum(d.width * d.height * d.samples for d in draws)
    n = max(16.0, 16.0 * fragments / (size[0] * size[1]))
    tol = 1e-6 + 4.0 * np.sqrt(n) * 2.0**-24
    for k, (a, b) in enumerate(zip(want, got)):
        texel = k < len(fit.d_levels)
        assert gradient_rel_error(b, a) < (tol if texel else 1e-5), (k, a.shape)
