"""Lines with values that stay zero along their length, against the oracle bit for bit: lines on
the axes x = 0 and y = 0, zero z, colours and texture coordinates of either sign, and lines of
up to SWR_MAX_LINE_STEPS steps.  Pieces of a line start with the chain of its first step
(chain_add), whose cost must not grow with the piece's place in the line."""
import numpy as np
import pytest

import oracle as O
from helpers import assert_same, run_cpu, run_gpu

pytestmark = pytest.mark.gpu

PROGS = [O.PS_LOG, O.PS_HASH, O.PS_DEPTH_CHECKER]


def _lines(points):
    """[n, 2, 2] window-space endpoints -> vertices whose z, colour and uv are zero but for red."""
    v = np.zeros(2 * len(points), O.RASTERIZER_VERTEX)
    v["x"], v["y"] = np.asarray(points, np.float32).reshape(-1, 2).T
    v["w"] = 1.0
    v["avar"][:, 0] = np.linspace(0.0, 1.0, v.size)
    v["avar"][::4, 1] = -0.0
    v["pvar"][::3] = -0.0
    return v, np.arange(v.size, dtype=np.int32)


@pytest.mark.parametrize("prog", PROGS)
@pytest.mark.parametrize("shape", [(16, 9000), (9000, 16)])
def test_axis_lines(gpu, cpu_oracle, prog, shape):
    w, h = shape
    n = 8900.0
    pts = [[(0, 1), (0, n)], [(0, n), (0, 1)], [(3.5, 2), (3.5, n)]] if h > w else \
        [[(1, 0), (n, 0)], [(n, 0), (1, 0)], [(2, 3.5), (n, 3.5)]]
    pts += [[(0, 0), (12, 12)], [(12.5, 3.25), (0, 0)]]
    v, idx = _lines(pts)
    pipe = O.Pipeline(w, h, scissor=(0, 0, w, h), ps_program=prog)
    cap = 60_000 if prog == O.PS_LOG else 0
    a = run_cpu(cpu_oracle, pipe, vertices=v, indices=idx, prim="line", log_capacity=cap)
    b = run_gpu(pipe, vertices=v, indices=idx, prim="line", log_capacity=cap)
    if prog == O.PS_LOG:
        assert int(a.log_count[0]) > 3 * 8_000
    assert_same(a, b, f"axis lines {shape} prog={prog}")


@pytest.mark.parametrize("steps", [1 << 14, 1 << 20])
def test_longest_lines(gpu, cpu_oracle, steps):
    """Most of each line lies off the target; every step counts."""
    n = float(steps)
    v, idx = _lines([[(0, 0), (0, n)], [(0, n), (0, 0)], [(0, 0), (n, 0)], [(5.25, 3), (5.25, n)],
                     [(-n / 2, 20), (n / 2, 20)]])
    pipe = O.Pipeline(40, 64, scissor=(0, 0, 40, 64), ps_program=O.PS_HASH)
    a = run_cpu(cpu_oracle, pipe, vertices=v, indices=idx, prim="line")
    b = run_gpu(pipe, vertices=v, indices=idx, prim="line")
    assert int(a.t1.sum()) > 200
    assert_same(a, b, f"lines of {steps} steps")
