"""The memoised multiples of a jump distance, the first calls that go without a table of
them and the velocity shares that jumps reach (pagmo2_amd/csrc/mt_jump_host.hpp), on the
CPU (tests/cpp/test_mt_multiples.cpp, test_mt_first_calls.cpp, test_velocity_shares.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def run(name):
    out = os.path.join(HERE, "cpp", "bin", name)
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "pagmo2_amd", "csrc"),
                           os.path.join(HERE, "cpp", name + ".cpp"), "-o", out + ".tmp", "-pthread"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_every_multiple_is_memoised():
    run("test_mt_multiples")


def test_first_calls_make_no_table():
    run("test_mt_first_calls")


def test_velocity_shares_are_bounded():
    run("test_velocity_shares")
