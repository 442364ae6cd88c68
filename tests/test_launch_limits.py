"""The host-side limits of kernel launches, compiled for the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# (256: FLIP G2P; 512: the density splat, whose split takes ~200 GB of grid to reach)
@pytest.mark.parametrize("threads", [64, 256, 448, 512, 1024])
def test_lanes_of_a_launch_stay_below_2_to_the_32(tmp_path, threads):
    src = tmp_path / "limit.cpp"
    src.write_text('#include "launch.hpp"\n#include <cstdio>\n'
                   'int main() { std::printf("%%lld", (long long)msbg::max_groups(%d)); }\n' % threads)
    exe = str(tmp_path / "limit")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "msbg-rs_amd", "csrc"), str(src), "-o", exe],
                   check=True)
    most = int(subprocess.run([exe], check=True, capture_output=True, text=True).stdout)
    assert most * threads < 2 ** 32 <= (most + 1) * threads
