"""The binned texel scatter where a probe crosses the border of its tile's
region, and where an upstream gradient is not finite, against the FP64 oracle.

A 64 x 64 quad steps 24 texels a pixel along u through a 96-texel wrapping
texture (one level, 2 probes, 6 texels either side of the centre) and one
texel a pixel along v.  Every fourth pixel's centre lies at texel 31.6, in
the first 32-texel tile, so that its right probe takes texels 37 and 38: the
last one of the tile's region, which reaches 6 texels past it, and the first
one outside.
"""
import numpy as np
import pytest
import torch

from grad_cases import G, params_of, view_of
from swiftshader_amd import abi, diff
from swiftshader_amd.batch import BatchPlan, grad_desc
from swiftshader_amd.scenes import DrawData, TextureData
from test_gpu_grad import _t, gpu_forward
from test_gpu_tap_scatter import test_binned_scatter_matches_per_view as matches_per_view

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZE, TW, TH = 64, 96, 64


def _quad():
    rng = np.random.default_rng(3)
    x = np.array([-1, 1, -1, 1, 1, -1], np.float32)
    y = np.array([-1, -1, 1, -1, 1, 1], np.float32)
    pos = np.stack([x, y, np.full(6, 0.5, np.float32), np.ones(6, np.float32)], 1)
    u = (31.6 - 12.0) / TW + (x + 1) / 2 * (SIZE * 24 / TW)
    v = (0.8 - 0.5) / TH + (y + 1) / 2 * (SIZE / TH)
    tex = TextureData(format=abi.FORMAT_R32G32B32A32_SFLOAT,
                      levels=[rng.uniform(0.25, 1.0, (TH, TW, 4)).astype(np.float32)], anisotropy_enable=1,
                      max_anisotropy=2.0, max_lod=0.0)
    return DrawData(width=SIZE, height=SIZE, positions=pos, texcoords=np.stack([u, v], 1).astype(np.float32),
                    shader=abi.SHADER_SAMPLE, texture=tex, color_format=abi.FORMAT_R32G32B32A32_SFLOAT)


def _run(d_color):
    """The batched backward's texture gradient, and the oracle's fragments and gradient function."""
    d = _quad()
    view, (pos, _, uv, levels), color, ids = gpu_forward(d)
    state = torch.zeros((1, SIZE, SIZE, 4), dtype=torch.float32, device=DEV)
    diff.backward_raw(view, pos, None, uv, levels, view.ids, torch.zeros((1, SIZE, SIZE, 4), device=DEV), state)
    target = torch.empty((1, SIZE, SIZE, 4), device=DEV)
    plan = BatchPlan([view.desc(pos, None, uv, levels, target)])
    up, got = _t(d_color), torch.zeros((TH, TW, 4), device=DEV)
    plan.set_grads([grad_desc(up, d_texture=[got])])
    plan.backward()
    torch.cuda.synchronize()
    plan.close()
    frag = G.fragments(ids, state.cpu().numpy())
    assert len(frag.t) == SIZE * SIZE and np.all(np.rint(frag.state[:, 1]) == 2) and np.all(frag.state[:, 0] == 0)

    def oracle(upstream):
        return G.gradient(view_of(d), params_of(d), frag, G.upstream(frag, upstream))["texture"]

    return got.cpu().numpy(), oracle


def test_taps_inside_a_crossing_probe_stay_in_fixed_point():
    """Upstream gradients of 1 +- 65536, of either sign for pixels that share
    their u: the sums of a texel cancel to a few units.  In fixed point each of
    the 32 products of a texel rounds by at most 2^-47 of the largest
    gradient (2^17), 2^-25 in all, and FP64 coordinates near 16 move the
    weights by some 1e-12: together below 1e-6 of a sum near 7.  In float each
    product rounds by 2^-9."""
    x = np.arange(SIZE)
    up = np.ones((1, SIZE, SIZE, 4), np.float32) * np.arange(1, 5, dtype=np.float32)
    up += np.where((x >> 2) & 1, 65536.0, -65536.0).astype(np.float32)[None, None, :, None]
    print("[tap scatter edges] cancelling gradients", flush=True)
    got, oracle = _run(up)
    want = oracle(up)
    assert np.all(want[:, 37] > 1.0) and np.all(want[:, 38] > 0.1)
    inside = np.arange(TW) != 38  # the tap outside the region: float products, added one by one
    err = np.abs(got - want)[:, inside] / np.abs(want).max()
    print(f"[tap scatter edges] column 37 {err[:, 37].max():.2e} all {err.max():.2e}", flush=True)
    assert err.max() < 1e-6


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_a_gradient_that_is_not_finite_stays_in_its_footprint(value):
    """The texels of that pixel's probes are not finite in its channel;
    everything else is the sum of the other pixels, added in float (up to 64
    adds of one sign to a texel: 64 * 2^-24 of it)."""
    up = np.ones((1, SIZE, SIZE, 4), np.float32)
    hole, only = up.copy(), np.zeros_like(up)
    hole[0, 20, 16, 2], only[0, 20, 16, 2] = 0.0, 1.0
    up[0, 20, 16, 2] = value
    print(f"[tap scatter edges] gradient {value}", flush=True)
    got, oracle = _run(up)
    want, touched = oracle(hole), oracle(only) != 0.0
    assert touched.sum() == 8 and not touched[..., [0, 1, 3]].any()
    assert not np.isfinite(got[touched]).any()
    assert np.abs(got - want)[~touched].max() < 64 * 2.0**-24 * want.max()


@pytest.mark.parametrize("mode", [abi.ADDRESS_REPEAT, abi.ADDRESS_CLAMP_TO_EDGE])
@pytest.mark.parametrize("size", [(1, 3), (3, 5), (5, 6), (7, 2), (6, 8), (8, 7), (9, 4)])
@pytest.mark.parametrize("aniso", [False, True])
def test_levels_of_fewer_than_eight_texels(size, mode, aniso):
    """Several cells of a wrapping level of fewer than 8 texels stand for one texel."""
    matches_per_view(size, mode, abi.FILTER_LINEAR, aniso, 4 if aniso else 1, size[0] == 5)
