"""A batched backward captured into a HIP graph follows swr_batch_plan_set_grads.

The graph is captured while only the texture's gradient is wanted; the plan's
targets then grow to the vertex attributes and shrink again.  Every replay
must equal the eager backward of the same targets.  Both sides add the same
products in an order of their own: 1e-5 of each buffer's norm, as for the
batched backward against the per-view one.
"""
import numpy as np
import pytest
import torch

from grad_cases import gradient_rel_error
from swiftshader_amd import abi, scenes, texfit
from swiftshader_amd.batch import BatchPlan, grad_desc
from swiftshader_amd.scenes import TextureData

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _fit(samples):
    """Views with the given sample counts, rendered; their upstream gradients set."""
    rng = np.random.default_rng(5)
    tex = TextureData(format=abi.FORMAT_R32G32B32A32_SFLOAT, levels=[])
    draws = []
    for k, s in enumerate(samples):
        w, h = 40 + 24 * k, 56 - 8 * k
        pos, uv, col = scenes.screen_triangles(rng, 200, w, h, area_hi=300)
        draws.append(scenes.DrawData(width=w, height=h, positions=pos, colors=col, texcoords=uv, samples=s,
                                     shader=abi.SHADER_MODULATE, texture=tex,
                                     color_format=abi.FORMAT_R32G32B32A32_SFLOAT))
    level0 = torch.from_numpy(rng.uniform(0.25, 1.0, (64, 64, 4)).astype(np.float32))
    fit = texfit.MultiViewFit(draws, level0, [torch.zeros((d.height, d.width, 4)) for d in draws],
                              geometry_grads=True, device=DEV)
    fit.forward_plain()
    fit._resolve_and_grad()
    torch.cuda.synchronize()
    return fit


@pytest.mark.parametrize("samples", [(1, 1), (4, 4), (1, 4)])
def test_replays_follow_the_gradient_targets(samples):
    fit = _fit(samples)
    plan = BatchPlan([vb.desc for vb in fit.views])

    def targets(geometry):
        return [grad_desc(vb.d_color, *((vb.d_pos, vb.d_col, vb.d_uv) if geometry and k in geometry else (None,) * 3),
                          fit.d_levels) for k, vb in enumerate(fit.views)]

    def result(run):
        fit._zero_grads()
        run()
        torch.cuda.synchronize()
        out = [l.cpu().numpy().copy() for l in fit.d_levels]
        for vb in fit.views:
            out += [t.cpu().numpy().copy() for t in (vb.d_pos, vb.d_col, vb.d_uv)]
        return out

    plan.set_grads(targets(None))
    result(plan.backward)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.backward()
    levels = len(fit.d_levels)
    # Vertex gradients of no view, of one (either group of draws), of both, of none again.
    for geometry in ((), (0,), (1,), (0, 1), ()):
        plan.set_grads(targets(geometry))
        want = result(plan.backward)
        for view in range(2):
            wanted = view in geometry
            assert all(np.any(a) == wanted for a in want[levels + 3 * view:levels + 3 * view + 3])
        for rep in range(3):
            print(f"[grad capture] samples {samples} geometry {geometry} replay {rep}", flush=True)
            got = result(graph.replay)
            for k, (a, b) in enumerate(zip(want, got)):
                assert gradient_rel_error(b, a) < 1e-5, (geometry, rep, k, a.shape)
    plan.close()
