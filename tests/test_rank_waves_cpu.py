"""k_order, k_rank, k_far, k_fronts, k_slots and k_masks (pagmo2_amd/csrc/fnds_chain.hip)
give the ranks, fronts and dominators under any order of their wavefronts, also where most points have no dominator:
the kernels' own text on the CPU (tests/cpp/test_rank_waves.cpp)."""
import os
import subprocess

from test_chain_waves_cpu import BIN, HERE, write_kernels


def test_ranks_under_any_order_of_the_wavefronts():
    os.makedirs(BIN, exist_ok=True)
    write_kernels()
    out = os.path.join(BIN, "test_rank_waves")
    subprocess.check_call(["g++", "-std=c++20", "-O1", "-U_FORTIFY_SOURCE", "-w", os.path.join(HERE, "cpp", "test_rank_waves.cpp"),
                           "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
