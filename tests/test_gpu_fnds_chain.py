"""The ranks and orders of fast_non_dominated_sorting without a peel, at the
sizes where its parts change hands: blocks of 64 points, spans of 32 blocks,
fronts of 64, 128 and 1024 members, bins of 64; and the orderings of fronts
within and beyond one workgroup's sort.  Bit for bit with the oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
KEYS = ("dom_count", "rank", "front_offsets", "front_items", "dom_offsets", "dom_items")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64)).to("cuda:0")


def check(objs):
    ws = P.Fnds()
    ws.run(dev(objs))
    got = ws.to_host(len(objs))
    ws.close()
    ref = O.fnds(objs)
    for k in KEYS:
        assert np.array_equal(got[k], ref[k]), k


def layers(sizes, seed, delta):
    """Fronts of the given sizes for small deltas: points on anti-diagonals
    x + y = L, L growing by delta; larger deltas leave fewer dominators."""
    rng = np.random.default_rng(seed)
    out = []
    for L, c in enumerate(sizes):
        x = np.sort(rng.uniform(0, 1, c))
        out.append(np.stack([x + L * delta, 1 - x + L * delta], axis=1))
    objs = np.concatenate(out)
    return objs[rng.permutation(len(objs))]


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 128, 129, 191, 193, 2047, 2048, 2049, 4097])
@pytest.mark.parametrize("m", [1, 2, 3])
def test_sizes(n, m):
    check(np.random.default_rng(n + m).uniform(0, 1, (n, m)))


@pytest.mark.parametrize("sizes", [(64, 64, 64), (65, 64, 65), (1, 128, 1, 128), (129, 128, 129), (64, 65, 128, 129),
                                   (3, 1024, 1024, 2), (1025, 1024, 1025), (2, 3000, 2500), (1023, 700, 40, 90)])
@pytest.mark.parametrize("delta", [2.0, 0.01, 0.0005])
def test_front_sizes(sizes, delta):
    check(layers(sizes, sum(sizes), delta))


@pytest.mark.parametrize("kind", ["chain", "one front", "equal", "few values", "special", "one over all"])
@pytest.mark.parametrize("n", [100, 2300])
def test_shapes(kind, n):
    rng = np.random.default_rng(n)
    if kind == "chain":
        objs = np.repeat(rng.permutation(n)[:, None], 3, axis=1).astype(float)
    elif kind == "one front":
        x = rng.uniform(0, 1, n)
        objs = np.stack([x, -x], axis=1)
    elif kind == "equal":
        objs = np.full((n, 2), 0.5)
    elif kind == "few values":
        objs = rng.integers(0, 6, (n, 3)).astype(float)
    elif kind == "special":
        objs = rng.choice([np.nan, np.inf, -np.inf, -0.0, 0.0, 1.0, 5e-324, -1.0], (n, 3))
    else:  # every member of front 1 has the same last dominator
        x = rng.uniform(0, 1, n)
        objs = np.stack([x, -x], axis=1)
        objs[n // 3] = (-2.0, -2.0)
    check(objs)


@pytest.mark.parametrize("n,m", [(16384, 1), (16384, 2), (16385, 2)])
def test_largest(n, m):
    check(np.random.default_rng(m).uniform(0, 1, (n, m)))


def test_equal_to_the_peel():
    objs = dev(np.random.default_rng(4).uniform(0, 1, (12000, 3)))
    ws = P.Fnds()
    ws.run(objs)
    a = ws.to_host(12000)
    ws.set_peel_blocks(20)
    ws.run(objs)
    b = ws.to_host(12000)
    ws.close()
    for k in KEYS:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("n,m,N", [(300, 2, 1), (300, 3, 150), (5000, 2, 2500), (5000, 3, 4999)])
def test_results_after_a_selection(n, m, N):
    """select_best_N_mo orders only the fronts it needs; the workspace still
    gives every output of the sort afterwards."""
    objs = np.random.default_rng(N).uniform(0, 1, (n, m))
    objs[: n // 10] = objs[n // 2: n // 2 + n // 10]
    ws = P.Fnds()
    out = torch.empty(N, dtype=torch.int64, device="cuda:0")
    assert ws.select_best_N_mo(dev(objs), N, out) == N
    assert np.array_equal(out.cpu().numpy().astype(np.uint64), O.select_best_N_mo(objs, N, stable=True))
    got = ws.to_host(n)
    ws.close()
    ref = O.fnds(objs)
    for k in KEYS:
        assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("sizes", [(4096, 10), (4097, 10), (5, 4500, 300), (700, 700, 700), (1, 1, 2, 1)])
def test_orderings(sizes):
    """Fronts of 4096 members and less are ordered by one workgroup each, larger
    ones by radix sorts."""
    objs = layers(sizes, 3, 0.02)
    objs = np.concatenate([objs, objs[: len(objs) // 8]])  # duplicates
    n = len(objs)
    d = dev(objs)
    ws = P.Fnds()
    out = torch.empty(n, dtype=torch.int64, device="cuda:0")
    ws.sort_population_mo(d, out)
    assert np.array_equal(out.cpu().numpy().astype(np.uint64), O.sort_population_mo(objs, stable=True))
    for N in (1, n // 3, n - 1):
        got = torch.empty(N, dtype=torch.int64, device="cuda:0")
        if ws.select_best_N_mo(d, N, got) == 0:
            continue
        assert np.array_equal(got.cpu().numpy().astype(np.uint64), O.select_best_N_mo(objs, N, stable=True)), N
    ws.close()


@pytest.mark.parametrize("n", [2, 3, 4095, 4096, 4097])
@pytest.mark.parametrize("m", [2, 4])
def test_crowding(n, m):
    pts = np.random.default_rng(n).integers(0, max(2, n // 2), (n, m)).astype(float)
    ws = P.Fnds()
    out = torch.empty(n, dtype=torch.float64, device="cuda:0")
    ws.crowding_distance(dev(pts), out)
    ws.close()
    ref = O.crowding_distance(pts, stable=True)
    assert np.array_equal(out.cpu().numpy(), ref, equal_nan=True)
    assert np.array_equal(P.crowding_distance_host(pts), ref, equal_nan=True)


@pytest.mark.parametrize("n,m", [(2, 2), (65, 1), (700, 3), (16385, 2)])
@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("only", [KEYS, ("dom_items",), ("rank", "front_offsets")])
def test_copies_to_device(n, m, shift, only):
    """pgh_fnds_copy into device memory (words in place, and an address that only a
    copy can take), any subset of the outputs, twice, and to the host afterwards."""
    objs = np.random.default_rng(n).uniform(0, 1, (n, m))
    ws = P.Fnds()
    ws.run(dev(objs))
    n_fronts, n_dom = ws.sizes()
    count = dict(dom_count=n, rank=n, front_offsets=n_fronts + 1, front_items=n, dom_offsets=n + 1, dom_items=n_dom)
    for _ in range(2):
        out = {k: torch.full((8 * count[k] + 16,), 255, dtype=torch.uint8, device="cuda:0") for k in only}
        P.check(P.lib().pgh_fnds_copy(ws.h, *(out[k].data_ptr() + shift if k in out else None for k in KEYS), 0))
        torch.cuda.synchronize()
        ref = ws.to_host(n)
        for k, t in out.items():
            got = t.cpu().numpy()
            assert np.array_equal(got[shift:shift + 8 * count[k]].view(np.uint64), ref[k]), k
            assert (got[:shift] == 255).all() and (got[shift + 8 * count[k]:] == 255).all(), k
    ws.close()
    if n < 1000:
        want = O.fnds(objs)
        for k in KEYS:
            assert np.array_equal(ref[k], want[k]), k
