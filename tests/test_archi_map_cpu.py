"""The archipelago tuner's candidates (pagmo2_amd/csrc/archi_map.hpp), on the CPU
(tests/cpp/test_archi_map.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_the_default_is_a_candidate():
    out = os.path.join(HERE, "cpp", "bin", "test_archi_map")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "pagmo2_amd", "csrc"), "-I",
                           os.path.join(ROOT, "include"), os.path.join(HERE, "cpp", "test_archi_map.cpp"), "-o",
                           out + ".tmp"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
