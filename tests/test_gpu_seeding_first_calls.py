"""The first draws of a program, while no table of jumps exists, and those after it was
made give the same words: std::mt19937's (numpy's RandomState is the same generator)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import numpy as np, torch
import pagmo2_amd as P
for n in (131074, 262144, 300002, 1048578, 2097152, 2097154):
    for call in range(max(3, 2 + 2097152 // n)):
        out = torch.zeros(n, dtype=torch.int32, device="cuda:0")
        P.mt19937_generate(call + 7, n, out)
        got = out.cpu().numpy().view(np.uint32)
        want = np.frombuffer(np.random.RandomState(call + 7).bytes(4 * n), dtype="<u4")
        assert np.array_equal(got, want), (n, call)
print("words ok")
"""


def test_words():
    r = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "words ok" in r.stdout, r.stdout + r.stderr
