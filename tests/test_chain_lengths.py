"""chain_add (softwarerenderer_amd/csrc/swr_chain.h) where its start or step is zero, subnormal,
huge, infinite or NaN, compiled for the host: the same bits as the addition loop, and a cost
that does not grow with the number of additions.  Lines are walked in pieces that each start
with a chain from the line's first step, so a chain of one addition per step makes a line's
cost the square of its length."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("chain") / "chain_lengths")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__host__=",
                    "-D__device__=", "-I" + os.path.join(ROOT, "softwarerenderer_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "chain_lengths.cpp"), "-o", out],
                   check=True)
    return out


def test_every_start_matches_the_addition_loop(exe):
    out = subprocess.run([exe, "values"], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert "mismatches 0" in out.stdout


def test_cost_does_not_grow_with_the_length(exe):
    # 126,760 chains of 2^30 additions: 1.4e14 of them one by one, many hours
    out = subprocess.run([exe, "cost"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0
