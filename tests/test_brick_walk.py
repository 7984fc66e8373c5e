"""CPU check of the readout's walk over a brick's particles.

tests/cpu/brick_walk_check.cpp replays it with the kernel's own index code
(flowpm_amd/csrc/brick_index.h) on grids of whole and of partial bricks, and
fails on any offset that is not the particle's or lies outside the brick.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_readout_walk_stays_in_its_brick(tmp_path):
  exe = str(tmp_path / "walk")
  subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined",
                  "-fno-sanitize-recover=all",
                  os.path.join(HERE, "cpu", "brick_walk_check.cpp"), "-o",
                  exe], check=True)
  r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
  print(r.stdout)
  assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
