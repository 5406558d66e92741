"""The archipelago's move with several elements in flight per thread (step_move,
pagmo2_amd/csrc/pso.hip) stays inside its item's arrays and moves each element as the
plain form does: its own text on the CPU between pages without access
(tests/cpp/test_step_move.cpp, wave_emu.hpp)."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
BIN = os.path.join(HERE, "cpp", "bin")


def definition(text, head):
    """The definition whose first line holds `head`, its template line included."""
    at = text.index(head)
    start = text.rindex("\n", 0, at) + 1
    before = text[text.rindex("\n", 0, start - 1) + 1:start]
    if before.startswith("template"):
        start -= len(before)
    return text[start:text.index("\n}", at) + 2] + (";\n" if head.startswith("struct") else "\n")


def test_move_stays_in_its_item():
    with open(os.path.join(ROOT, "pagmo2_amd", "csrc", "pso.hip")) as f:
        text = f.read()
    parts = [definition(text, h) for h in
             ("struct island_desc {", "struct tile {", "bool le_f(", "uint32_t best_neighbour(", "double pso_clamp_move(",
              "double pso_move(", "const uint4 *gen_words4(", "struct step_args {", "struct step_rows {",
              "void step_row(")]
    parts.append("inline void step_move_general(const island_desc &, const tile &, const step_args &, step_rows &) {}\n")
    parts.append(definition(text, "bool step_move("))
    os.makedirs(BIN, exist_ok=True)
    with open(os.path.join(BIN, "step_move.inc"), "w") as f:
        f.write(re.sub(r"#pragma unroll[^\n]*", "", "\n".join(parts)))
    out = os.path.join(BIN, "test_step_move")
    subprocess.check_call(["g++", "-std=c++20", "-O1", "-ffp-contract=off", "-U_FORTIFY_SOURCE", "-w",
                           os.path.join(HERE, "cpp", "test_step_move.cpp"), "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout + r.stderr)
