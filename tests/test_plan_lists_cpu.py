"""Work lists of the LDS-staged stage C tiles: those the library builds cover
every K step of every tile once, and a wrong entry is refused before it reaches
the device; a plan's tuning key tells plans of different rules apart
(tests/plan/plan_check.cpp, against the built library)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "vmps_amd")


def build(name, tmp_path):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-I" + os.path.join(LIB, "csrc"),
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "plan", name + ".cpp"), "-o", exe,
                    "-L" + LIB, "-lvmps_hxv", "-Wl,-rpath," + LIB], check=True)
    return exe


def test_work_items_and_signatures(tmp_path):
    r = subprocess.run([build("plan_check", tmp_path)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
