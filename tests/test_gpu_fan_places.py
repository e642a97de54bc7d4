"""Draw-order places of clipped triangles: batches of 1024 with and without appended fan
triangles, at the batch, workgroup (4 batches) and one-launch (16 batches) edges, and a draw of
more workgroups than the down pass adds up itself."""
import numpy as np
import pytest

import oracle as O
from softwarerenderer_amd import scenes
from helpers import assert_same, run_cpu, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 1023, 1024, 1025, 4096, 4097, 16384, 16385, 40000])
@pytest.mark.parametrize("spread", [0.5, 1.6])
def test_places(gpu, cpu_oracle, n, spread):
    """The hash program folds every fragment's key and values in order."""
    sc = scenes.clip_scene(ntri=n, seed=n, width=80, height=50, spread=spread,
                           shrink=(0.02, 0.3))
    pipe = O.Pipeline(80, 50, raster_mode=O.RASTER_SPAN, cull_mode=O.CULL_NONE,
                      vs_program=O.VS_RAW, vs_counts=(1, 3, 2), ps_program=O.PS_HASH)
    assert_same(run_cpu(cpu_oracle, pipe, sc), run_gpu(pipe, sc), f"n={n} spread={spread}")


def test_more_workgroups_than_are_added_up(gpu, cpu_oracle):
    """8193 workgroups: 33,558,528 triangles of which a few hundred draw (the others are
    degenerate), spread over the whole draw."""
    import torch
    from softwarerenderer_amd import api
    n, few = 8193 * 4096, 300
    sc = scenes.clip_scene(ntri=few, seed=5, width=64, height=48, spread=1.2, shrink=(0.1, 0.5))
    at = np.unique(np.linspace(0, n - 1, few).astype(np.int64))
    idx = torch.zeros((n, 3), dtype=torch.int32, device=gpu)
    idx[torch.from_numpy(at).to(gpu)] = torch.from_numpy(
        sc.indices.reshape(-1, 3)[:at.size]).to(gpu)
    pipe = O.Pipeline(64, 48, raster_mode=O.RASTER_BLOCK, cull_mode=O.CULL_NONE,
                      vs_program=O.VS_RAW, vs_counts=(1, 3, 2), ps_program=O.PS_COVERAGE,
                      ps_z=False, ps_w=False, ps_a=0, ps_p=0)
    a = run_cpu(cpu_oracle, pipe, sc)
    out = torch.zeros((48, 64), dtype=torch.int32, device=gpu)
    r = api.Rasterizer(0)
    r.setRasterMode(api.RasterMode.Block)
    r.setScissorRect(0, 0, 64, 48)
    r.setPixelShader(api.CoverageShader(out))
    v = api.VertexProcessor(r)
    v.setViewport(0, 0, 64, 48)
    v.setCullMode(api.CullMode.None_)
    vs = api.VertexShaderBase()
    vs.Program, vs.AttribCount, vs.AVarCount, vs.PVarCount = pipe.vs_program, 1, 3, 2
    v.setVertexShader(vs)
    v.setVertexAttribPointer(0, sc.stride, torch.from_numpy(sc.vertices).to(gpu))
    v.drawElements(api.DrawMode.Triangle, idx.reshape(-1))
    r.close()
    assert int((a.t0 != 0).sum()) > 500
    assert np.array_equal(a.t0.view(np.uint32), out.cpu().numpy().view(np.uint32))
