"""The (tile, primitive) pair lists where their arithmetic changes, against the
oracle, bit for bit: triangles whose extent lies around the limit of the
32-bit block masks (16383 sixteenths of a pixel), slivers and wide ones of both
windings, and pair counts around whole blocks of the sort (4096)."""
import numpy as np
import pytest

from oracle_runner import oracle_render
from swiftshader_amd import abi
from swiftshader_amd.scenes import DrawData
from test_gpu_parity import _compare, gpu_render

pytestmark = pytest.mark.gpu


def _check(name, draw):
    print(f"[pair lists] {name}", flush=True)
    _compare(name, oracle_render(draw), gpu_render(draw))


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("extent", [1022.0, 1023.9375, 1024.0, 1025.0])
@pytest.mark.parametrize("tall", [False, True])
def test_triangles_around_the_mask_extent(extent, tall, samples):
    long, short, n = 1056, 47, 60
    rng = np.random.default_rng(int(extent * 16) + samples)
    a = rng.uniform(4.0, 1050.0 - extent, (n, 1))  # 28.4 positions of the two far vertices
    b = a + extent
    mid = rng.uniform(a, b)
    along = np.concatenate([a, b, mid], 1)
    across = rng.uniform(1.0, 46.0, (n, 3))
    across[::3] = across[::3, :1] + rng.uniform(-1.0, 1.0, (n // 3, 3))  # slivers
    along, across = np.round(along * 16) / 16, np.round(across * 16) / 16
    flip = rng.random(n) < 0.5
    along[flip], across[flip] = along[flip][:, [1, 0, 2]], across[flip][:, [1, 0, 2]]
    x, y, w, h = (across, along, short, long) if tall else (along, across, long, short)
    z = rng.uniform(0.0, 1.0, (n, 3))
    pos = np.stack([2.0 * x / w - 1.0, 2.0 * y / h - 1.0, z, np.ones_like(z)], 2).reshape(-1, 4).astype(np.float32)
    col = rng.uniform(0.0, 1.0, (3 * n, 4)).astype(np.float32)
    _check(f"extent {extent} tall {tall} x{samples}",
           DrawData(width=w, height=h, positions=pos, colors=col, samples=samples, shader=abi.SHADER_INTERPOLATE))


@pytest.mark.parametrize("pairs", [1, 4095, 4096, 4097, 12288])
def test_pair_counts_around_the_sort_blocks(pairs):
    """Triangles of one tile each."""
    side, rng = 256, np.random.default_rng(pairs)
    origin = rng.integers(0, side // 16, (pairs, 1, 2)) * 16.0
    xy = origin + rng.uniform(1.0, 15.0, (pairs, 3, 2))
    z = rng.uniform(0.0, 1.0, (pairs, 3, 1))
    pos = np.concatenate([2.0 * xy / side - 1.0, z, np.ones_like(z)], 2).reshape(-1, 4).astype(np.float32)
    col = rng.uniform(0.0, 1.0, (3 * pairs, 4)).astype(np.float32)
    _check(f"{pairs} pairs", DrawData(width=side, height=side, positions=pos, colors=col,
                                      shader=abi.SHADER_INTERPOLATE))
