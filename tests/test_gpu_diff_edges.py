"""The antialiasing part of the backward where its lists change shape: tiles cut by the image,
groups of tiles that span views, one to four channels, one silhouette pair per several pixels
(coarse meshes) and many, against the FP64 reference with the tolerances of the other
differentiation tests."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

from test_diff_reference import make_case  # noqa: E402
from test_gpu_diff import _fp64_check, gpu_renderer  # noqa: E402


@pytest.mark.parametrize("views,size,subdiv", [(1, 16, 1), (1, 61, 1), (5, 31, 2), (9, 48, 2),
                                                (3, 95, 3)])
@pytest.mark.parametrize("channels", [1, 2, 4])
def test_edge_gradients(gpu, views, size, subdiv, channels):
    V, F, clip, _ = make_case(views=views, size=size, subdiv=subdiv, seed=size)
    attr = np.random.default_rng(size).random((V.shape[0], channels)).astype(np.float32)
    r = gpu_renderer(F, V.shape[0], views, size, channels)
    _fp64_check(r, clip, F, attr, seed=size + 1)
    r.close()


@pytest.mark.parametrize("size,n", [(16, 40), (33, 400), (61, 3000)])
@pytest.mark.parametrize("channels", [1, 3, 4])
def test_blend_of_separate_triangles(gpu, channels, size, n):
    """Separate triangles of a few pixels, every one with a silhouette all round: pixels with up
    to four blends, tiles with more blends than lanes, in two views of an image that cuts the
    tiles; the image against the FP64 reference (1e-5, as the other tests of the image)."""
    import torch
    rng = np.random.default_rng(size)
    views = 2
    c = rng.uniform(-1.1, 1.1, (views, n, 1, 2))
    p = c + rng.uniform(2.0, 9.0, (views, n, 1, 1)) / size * rng.normal(0, 1, (views, n, 3, 2))
    w = rng.uniform(0.5, 2.0, (views, n, 3, 1))
    z = rng.uniform(-0.9, 0.9, (views, n, 1, 1)) + np.zeros_like(w)
    clip = (np.concatenate([p, z, np.ones_like(w)], 3) * w).reshape(views, 3 * n, 4)
    clip = np.ascontiguousarray(clip, np.float32)
    F = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    attr = rng.random((3 * n, channels)).astype(np.float32)
    r = gpu_renderer(F, 3 * n, views, size, channels)
    img = r.forward(torch.from_numpy(clip).cuda(), torch.from_numpy(attr).cuda(), sync=True)
    img = img.cpu().numpy()
    ids, depth = r.ids.cpu().numpy().view(np.uint32), r.depth.cpu().numpy()
    ref, _, _ = O.diff_reference(clip, F, r.adj.cpu().numpy(), attr, ids, depth,
                                 np.zeros(img.shape, np.float32))
    assert (ids > 0).mean() > 0.1
    assert np.abs(img - ref).max() <= 1e-5
    r.close()
