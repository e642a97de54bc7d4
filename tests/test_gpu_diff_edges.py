"""The antialiasing part of the backward where its lists change shape: tiles cut by the image,
groups of tiles that span views, one to four channels, one silhouette pair per several pixels
(coarse meshes) and many, against the FP64 reference with the tolerances of the other
differentiation tests."""
import numpy as np
import pytest

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
