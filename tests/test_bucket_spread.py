"""How the binning sort deals tiles to its buckets (softwarerenderer_amd/csrc/swr_buckets.h),
compiled for the host.  A bucket is one workgroup's work, so a mesh that lies in a column, a
strip or a diagonal of the screen must not fall into a few of them: dealt by the id's low 8 bits,
a column of a 2048-pixel target is one bucket's (256 times its share)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_that_lie_together_lie_in_different_buckets(tmp_path):
    exe = str(tmp_path / "bucket_spread")
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__host__=", "-D__device__=",
                    "-I" + os.path.join(ROOT, "softwarerenderer_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "bucket_spread.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe, "16"], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
