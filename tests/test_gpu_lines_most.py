"""The most primitives a point draw takes (2^30), nearly all of them skipped by their index: the
launches that count and emit them cover every one, the last included."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def test_most_points(gpu):
    import torch
    from softwarerenderer_amd import _abi, api
    n = 1 << 30
    free, _ = torch.cuda.mem_get_info()
    if free < 40 << 30:
        pytest.skip("2^30 indices and their counts take 30 GB of device memory")
    idx = torch.full((n,), -1, dtype=torch.int32, device=gpu)
    places = [0, 1, (1 << 29) - 1, 1 << 29, n - 17, n - 16, n - 1]
    for k, i in enumerate(places):
        idx[i] = k
    v = np.zeros(len(places), O.RASTERIZER_VERTEX)
    v["x"], v["y"], v["w"] = np.arange(len(places)) + 0.5, 2.5, 1.0
    vt = torch.from_numpy(v.view(np.uint8)).to(gpu)
    buf = torch.zeros((8, 16), dtype=torch.int32, device=gpu)
    r = api.Rasterizer(0)
    try:
        r.setScissorRect(0, 0, 16, 8)
        r.setPixelShader(api.CoverageShader(buf))
        r.drawPointList(vt, idx)
        want = torch.zeros_like(buf)
        want[2, :len(places)] = 1
        assert torch.equal(buf, want)
        assert r.stats().raster_primitives == len(places)
        with pytest.raises(_abi.SwrError) as e:  # one more is refused, as before
            r.drawPointList(vt, torch.full((n + 1,), -1, dtype=torch.int32, device=gpu))
        assert e.value.code == -5
    finally:
        r.close()
        del idx
        torch.cuda.empty_cache()
