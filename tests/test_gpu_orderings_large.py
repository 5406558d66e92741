"""sort_population_mo and select_best_N_mo where one front is larger than a workgroup
sorts (4096 members, 2048 of at most 4096 points) beside others that are not, in every position, and where none
is although the points are many.  Bit for bit with the oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def layers(sizes, seed):
    """Fronts of the given sizes: points on anti-diagonals, each beyond the one before."""
    rng = np.random.default_rng(seed)
    out = []
    for L, c in enumerate(sizes):
        x = rng.uniform(0, 1, c)
        out.append(np.stack([x + 2.0 * L, 1 - x + 2.0 * L], axis=1))
    objs = np.concatenate(out)
    return objs[rng.permutation(len(objs))]


def check(objs, Ns):
    n = len(objs)
    d = torch.from_numpy(np.ascontiguousarray(objs)).to("cuda:0")
    ws = P.Fnds()
    out = torch.empty(n, dtype=torch.int64, device="cuda:0")
    ws.sort_population_mo(d, out)
    assert np.array_equal(out.cpu().numpy().astype(np.uint64), O.sort_population_mo(objs, stable=True))
    for N in (N for N in Ns if N < n):
        got = torch.empty(N, dtype=torch.int64, device="cuda:0")
        assert ws.select_best_N_mo(d, N, got) == N
        assert np.array_equal(got.cpu().numpy().astype(np.uint64), O.select_best_N_mo(objs, N, stable=True)), N
    ws.close()


@pytest.mark.parametrize("sizes", [(4097, 20), (20, 4097), (300, 4200, 700), (4096, 4096), (700, 700, 4096), (1, 4097),
                                   (2048, 2048), (2049, 2047), (30, 2049), (2048, 2049), (1, 4095), (2049,)])
def test_layers(sizes):
    ends = np.cumsum(sizes)
    check(layers(sizes, len(sizes)), sorted({1, *(int(e) for e in ends[:-1]), *(int(e) - 1 for e in ends),
                                             int(ends[0]) + 1}))


@pytest.mark.parametrize("n,m", [(5000, 4), (5000, 7), (9000, 7), (9000, 12)])
def test_many_objectives(n, m):
    objs = np.random.default_rng(m).uniform(0, 1, (n, m))
    objs[: n // 9] = objs[n // 2: n // 2 + n // 9]
    check(objs, (1, n // 3, n - 1))
