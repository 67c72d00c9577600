"""Batches of more MBs than one grid has room for: the inter stage's launch holds 1.5 (MBAFF: 2)
blocks per MB since it derives the boundary strengths too, so 2^32 threads are 44.7 million MBs,
1,380 pictures of 3840x2160."""
import os
import subprocess

from h264_video_decoder_demo_amd import build as hbuild

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_launch_fits_a_grid(tmp_path):
    exe = str(tmp_path / "launch_check")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(hbuild.ROOT, "include"), "-I", hbuild.CSRC,
                    os.path.join(HERE, "launch_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout
