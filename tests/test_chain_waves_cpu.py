"""k_chain (pagmo2_amd/csrc/fnds_chain.hip) gives the same order whichever of its
wavefronts is ahead between two barriers: the kernel's own text, run on the CPU
(tests/cpp/test_chain_waves.cpp, wave_emu.hpp)."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
BIN = os.path.join(HERE, "cpp", "bin")


def kernels():
    """The unnamed namespace of the source, its LDS objects as plain memory."""
    with open(os.path.join(ROOT, "pagmo2_amd", "csrc", "fnds_chain.hip")) as f:
        text = f.read()
    text = text[text.index("namespace\n{"):text.index("} // namespace\n") + len("} // namespace\n")]
    text = re.sub(r"extern __shared__ (?:__align__\(\d+\) )?(\w+) (\w+)\[\];",
                  r"\1 *\2 = reinterpret_cast<\1 *>(wave_emu::dynamic_lds);", text)
    return re.sub(r"(?<!_)__shared__\b", "static", text)


def write_kernels():
    inc = os.path.join(BIN, "fnds_chain_kernels.inc")
    with open(f"{inc}.{os.getpid()}", "w") as f:
        f.write(kernels())
    os.replace(f"{inc}.{os.getpid()}", inc)


def test_positions_under_any_order_of_the_wavefronts():
    os.makedirs(BIN, exist_ok=True)
    write_kernels()
    out = os.path.join(BIN, "test_chain_waves")
    subprocess.check_call(["g++", "-std=c++20", "-O1", "-U_FORTIFY_SOURCE", "-w", os.path.join(HERE, "cpp", "test_chain_waves.cpp"),
                           "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
