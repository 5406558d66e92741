"""fast_non_dominated_sorting of populations that are one front or a few large ones, as
late generations are: fronts beyond 1024 and 4096 members of every density.  Bit for
bit with the oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
KEYS = ("dom_count", "rank", "front_offsets", "front_items", "dom_offsets", "dom_items")


def population(kind, n, m, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0, 1, (n, m))
    x /= x.sum(1, keepdims=True)
    if kind == "two dense":
        x += (np.arange(n) * 2 // n)[:, None] * 2.0
    elif kind == "sparse tail":  # a few dominators each
        x += rng.exponential(0.0125, n)[:, None]
    elif kind == "dense tail":
        x += rng.exponential(0.1, n)[:, None]
    elif kind == "one beyond":  # every member of the second front has one dominator
        x[: n // 2] += 1e-12
        x[: n // 2] = x[n // 2: n // 2 + n // 2] + 1e-9
    return x[rng.permutation(n)]


@pytest.mark.parametrize("kind", ["one", "two dense", "sparse tail", "dense tail", "one beyond"])
@pytest.mark.parametrize("n,m", [(4097, 2), (9001, 3), (16384, 2)])
def test_fronts(kind, n, m):
    objs = population(kind, n, m, n)
    ws = P.Fnds()
    ws.run(torch.from_numpy(np.ascontiguousarray(objs)).to("cuda:0"))
    got = ws.to_host(n)
    ws.close()
    ref = O.fnds(objs)
    for k in KEYS:
        assert np.array_equal(got[k], ref[k]), k
