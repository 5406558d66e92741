"""The way to the fronts after a workspace's peel was set or tuned
(pagmo2_amd/csrc/fnds_route.hpp), on the CPU (tests/cpp/test_fnds_route.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_choice_of_the_way():
    out = os.path.join(HERE, "cpp", "bin", "test_fnds_route")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "pagmo2_amd", "csrc"),
                           os.path.join(HERE, "cpp", "test_fnds_route.cpp"), "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
