"""The operand loads of the LDS-staged FP64 / FP32 tiles stay inside their
blocks: the kernels' own address arithmetic (csrc/tile_loads.hpp) replayed on
the host for every thread and K step, at odd and even block sizes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_big_tile_loads_stay_inside_the_block(tmp_path):
    exe = str(tmp_path / "loads_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(ROOT, "vmps_amd", "csrc"),
                    os.path.join(ROOT, "tests", "loads", "loads_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
