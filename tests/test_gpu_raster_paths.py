"""The raster kernel's per-program paths at the lengths and edges where they change: lists
around the group (8) and ring (64) sizes, targets that end inside a block, every bin size,
against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from softwarerenderer_amd import scenes
from helpers import assert_same, run_cpu, run_gpu

pytestmark = pytest.mark.gpu

SHAPES = [dict(), dict(raster_waves=1), dict(bin_size=16), dict(bin_size=32, waves_per_bin=2),
          dict(bin_size=16, raster_queue=1)]


def _layers(n, seed, spread):
    """n triangles over one small screen, near ones smaller, so that blocks have lists of up to
    n entries, some pixels are covered by all of them and some by none."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-spread, spread, (n, 1, 2))
    p = c + rng.uniform(0.3, 1.6, (n, 1, 1)) * rng.uniform(-1, 1, (n, 3, 2))
    v = np.concatenate([np.clip(p, -0.99, 0.99), rng.uniform(-0.9, 0.9, (n, 3, 1)),
                        rng.random((n, 3, 3))], 2)
    return scenes.Scene(v.reshape(-1, 6).astype(np.float32), np.arange(3 * n, dtype=np.int32),
                        np.eye(4, dtype=np.float32), 0, 0)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 64, 65, 200])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("prog", [O.PS_RGB, O.PS_COVERAGE])
def test_last_fragment_wins(gpu, cpu_oracle, prog, shape, n):
    from softwarerenderer_amd import api
    sc = _layers(n, 100 + n, 0.2 if n > 64 else 0.6)
    for mode in (O.RASTER_SPAN, O.RASTER_BLOCK, O.RASTER_ADAPTIVE):
        pipe = O.Pipeline(37, 21, raster_mode=mode, cull_mode=O.CULL_NONE,
                          vs_program=O.VS_POS_RGB, vs_counts=(1, 3, 0), ps_program=prog,
                          ps_z=False, ps_w=False, ps_a=3, ps_p=0)
        r = api.Rasterizer(0)
        r.setTuning(**SHAPES[shape])
        assert_same(run_cpu(cpu_oracle, pipe, sc), run_gpu(pipe, sc, rasterizer=r),
                    f"n={n} mode={mode} {SHAPES[shape]}")
        r.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 300])
@pytest.mark.parametrize("prog", [(O.PS_HASH, 3, 2), (O.PS_HASH, 16, 16),
                                  (O.PS_DEPTH_CHECKER, 3, 2), (O.PS_RGB, 3, 0)])
def test_fragments_of_a_pixel(gpu, cpu_oracle, prog, n):
    """n points: half of them in one pixel, the others over a tile that the target cuts."""
    v = scenes.window_lines(n, 7 + n, 13, 9, margin=0.0)[:n]
    v["x"][::2], v["y"][::2] = 9.5, 8.25
    v["x"][1::2] = np.random.default_rng(n).uniform(0, 13, n // 2)
    v["y"][1::2] = np.random.default_rng(n + 1).uniform(0, 9, n // 2)
    pipe = O.Pipeline(13, 9, ps_program=prog[0], ps_z=prog[0] != O.PS_RGB,
                      ps_w=prog[0] != O.PS_RGB, ps_a=prog[1], ps_p=prog[2])
    idx = np.arange(n, dtype=np.int32)
    assert_same(run_cpu(cpu_oracle, pipe, vertices=v, indices=idx, prim="point"),
                run_gpu(pipe, vertices=v, indices=idx, prim="point"), f"n={n} {prog}")


GROUPS = SHAPES + [dict(raster_group=1), dict(raster_group=2, bin_size=16),
                   dict(raster_group=4, bin_size=32)]


@pytest.mark.parametrize("n", [1, 3, 8, 9, 70])
@pytest.mark.parametrize("shape", range(len(GROUPS)))
@pytest.mark.parametrize("prog", [(O.PS_HASH, 4, 4), (O.PS_HASH, 16, 16), (O.PS_HASH, 0, 0),
                                  (O.PS_DEPTH_CHECKER, 3, 2), (O.PS_VISIBILITY, 0, 0)])
def test_chained_planes(gpu, cpu_oracle, prog, shape, n):
    """Every interpolant of every fragment (hash), and the nearest fragment, for lists of n
    primitives in blocks that the target's right and lower edges cut."""
    from softwarerenderer_amd import api
    rng = np.random.default_rng(n)
    lay = _layers(n, 300 + n, 0.5)
    w = rng.uniform(0.5, 2.0, (3 * n, 1))
    na, np_ = max(prog[1], 1), max(prog[2], 1)
    v = np.concatenate([lay.vertices[:, :3] * w, w, rng.random((3 * n, na + np_))], 1)
    sc = scenes.Scene(v.astype(np.float32), lay.indices, np.eye(4, dtype=np.float32), 0, 0)
    for mode in (O.RASTER_SPAN, O.RASTER_BLOCK, O.RASTER_ADAPTIVE):
        pipe = O.Pipeline(37, 21, raster_mode=mode, cull_mode=O.CULL_NONE, vs_program=O.VS_RAW,
                          vs_counts=(1, na, np_), ps_program=prog[0], ps_z=True,
                          ps_w=prog[0] != O.PS_VISIBILITY, ps_a=prog[1], ps_p=prog[2])
        r = api.Rasterizer(0)
        r.setTuning(**GROUPS[shape])
        assert_same(run_cpu(cpu_oracle, pipe, sc), run_gpu(pipe, sc, rasterizer=r),
                    f"n={n} mode={mode} {GROUPS[shape]} {prog}")
        r.close()


@pytest.mark.parametrize("n", [1, 5, 64, 65, 150])
@pytest.mark.parametrize("prog", [(O.PS_LOG, 3, 2), (O.PS_LOG, 16, 16), (O.PS_DEPTH_CHECKER, 3, 2)])
def test_lines_of_all_lengths(gpu, cpu_oracle, prog, n):
    """Lines of 0 to some 2,000 steps side by side, many of them partly off the target: their
    pieces (32 steps) start where the step-by-step walk would be."""
    w, h = 700, 45
    v = scenes.window_lines(n, 11 + n, w, h, long_frac=0.0)
    rng = np.random.default_rng(n)
    steps = np.resize([0, 1, 63, 64, 65, 128, 129, 700, 2000, 333], n)
    x0 = rng.uniform(-300, 500, n)
    v["x"][0::2], v["x"][1::2] = x0, x0 + steps * rng.choice([-1, 1], n)
    v["y"][0::2] = rng.uniform(0, h, n)
    v["y"][1::2] = v["y"][0::2] + rng.uniform(-1, 1, n) * np.minimum(steps, 60)
    pipe = O.Pipeline(w, h, ps_program=prog[0], ps_z=True, ps_w=True, ps_a=prog[1], ps_p=prog[2])
    idx = np.arange(2 * n, dtype=np.int32)
    cap = 200_000 if prog[0] == O.PS_LOG else 0
    assert_same(run_cpu(cpu_oracle, pipe, vertices=v, indices=idx, prim="line", log_capacity=cap),
                run_gpu(pipe, vertices=v, indices=idx, prim="line", log_capacity=cap),
                f"n={n} {prog}")


@pytest.mark.parametrize("scissor", [(0, 0, 70, 45), (-400, -9, 480, 60), (5, 3, 50, 40)])
@pytest.mark.parametrize("shape", [2, 3, 4])
@pytest.mark.parametrize("prog", [(O.PS_DEPTH_CHECKER, 3, 2), (O.PS_VISIBILITY, 0, 0)])
def test_hidden_primitives(gpu, cpu_oracle, prog, shape, scissor):
    """Long lists of larger bins, where what lies behind a block's pixels is dropped: sloped
    planes crossing each other, and the same planes again one unit in the last place nearer or
    farther, in front, behind and in random order."""
    from softwarerenderer_amd import api
    n = 500
    lay = _layers(n, 500 + shape, 0.5).vertices.reshape(n, 3, 6)
    lay[:, :, 0:2] = np.clip(lay[:, :, 0:2] * 3, -0.99, 0.99)
    same = lay.copy()
    same[:, :, 2] = np.nextafter(same[:, :, 2], np.float32(-1) ** np.arange(n)[:, None] * 2,
                                 dtype=np.float32)
    v = np.concatenate([lay, same])
    order = np.argsort(v[:, :, 2].max(1), kind="stable")
    for mode in (O.RASTER_SPAN, O.RASTER_BLOCK, O.RASTER_ADAPTIVE):
        for name, o in (("near first", order), ("far first", order[::-1]),
                        ("mixed", np.random.default_rng(mode).permutation(2 * n))):
            t = v[o].reshape(-1, 6)
            w = np.ones((t.shape[0], 1), np.float32)
            t = np.concatenate([t[:, :3], w, t[:, 3:], t[:, :2]], 1).astype(np.float32)
            sc = scenes.Scene(t, np.arange(6 * n, dtype=np.int32), np.eye(4, dtype=np.float32),
                              0, 0)
            pipe = O.Pipeline(70, 45, raster_mode=mode, cull_mode=O.CULL_NONE, scissor=scissor,
                              vs_program=O.VS_RAW, vs_counts=(1, 3, 2), ps_program=prog[0],
                              ps_w=prog[0] != O.PS_VISIBILITY, ps_a=prog[1], ps_p=prog[2])
            r = api.Rasterizer(0)
            r.setTuning(**SHAPES[shape])
            a, b = run_cpu(cpu_oracle, pipe, sc), run_gpu(pipe, sc, rasterizer=r)
            r.close()
            assert int((a.t0 != 0).sum()) > 500
            assert_same(a, b, f"{name} mode={mode} {prog} {SHAPES[shape]}")
