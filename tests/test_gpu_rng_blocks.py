"""std::mt19937 on the device at the edges of its blocks (624 words), phases
(2496 words), shares (2^14 words and more) and splits (from 2^17 words, at most
512 shares), and pso_gen's velocity draws made by many workgroups: bit for bit
with the oracle's sequential generator."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda:0"


@pytest.mark.parametrize("n", [2, 623, 624, 625, 1248, 2495, 2496, 2497, 4992, 4993, (1 << 17) - 1, 1 << 17,
                               (1 << 17) + 1, 9 * (1 << 14) - 1, 9 * (1 << 14) + 1, 33 * (1 << 14) + 625,
                               512 * (1 << 14), 512 * (1 << 14) + 1])
def test_words(n):
    out = torch.full((n + 8,), -1, dtype=torch.int32, device=DEV)
    P.mt19937_generate(77, n, out[3:])  # 4-byte aligned output
    torch.cuda.synchronize()
    h = out.cpu().numpy()
    assert np.array_equal(h[3:3 + n].view(np.uint32), O.mt19937_u32(77, n))
    assert (h[:3] == -1).all() and (h[3 + n:] == -1).all()


@pytest.mark.parametrize("skip", [1, 623, 624, 625, 2497, 5000])
@pytest.mark.parametrize("n", [1, 624, 3001])
def test_words_after_skip(skip, n):
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    P.mt19937_generate(5, n, out, skip=skip)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), O.mt19937_u32(5, n, skip=skip))


@pytest.mark.parametrize("kind,dim,n", [(P.ROSENBROCK, 2, 1), (P.ACKLEY, 1, 313), (P.LENNARD_JONES, 3, 416),
                                        (P.LENNARD_JONES, 7, 4370), (P.LENNARD_JONES, 40, 5000),
                                        (P.GRIEWANK, 99, 663), (P.SCHWEFEL, 13, 5042)])
def test_population(kind, dim, n):
    nx, _ = P.dims(kind, dim)
    out = torch.empty((n, nx), dtype=torch.float64, device=DEV)
    P.batch_random_dv(kind, dim, n, 9, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), O.batch_random_dv(kind, dim, n, 9))


@pytest.mark.parametrize("mode", [P.ARCHI_BATCHED, P.ARCHI_PER_ISLAND])
def test_velocities_of_large_islands(mode):
    """Islands whose velocity draws are split (more than 2^17 words), beside
    small ones, one whose generations draw fewer words than its velocities,
    one that keeps its velocities and one of no generations."""
    spec = [(P.LENNARD_JONES, 13, 2001, {}), (P.ROSENBROCK, 10, 30, {}), (P.ROSENBROCK, 40, 4096, {}),
            (P.ROSENBROCK, 700, 100, dict(variant=4)), (P.ROSENBROCK, 64, 1025, dict(memory=True)),
            (P.ROSENBROCK, 33, 2500, dict(gen=0))]
    isl = []
    for k, (kind, dim, pop, more) in enumerate(spec):
        X0, F0 = O.population_init(kind, dim, pop, 300 + k)
        isl.append(dict(kind=kind, dim=dim, X0=X0, F0=F0, algo=P.pso_params(**{"gen": 2, "seed": 40 + k, **more})))
    a = P.Archipelago(isl)
    for _ in range(2):
        a.evolve(mode)
    for k, (kind, dim, pop, more) in enumerate(spec):
        d = isl[k]
        args = {"gen": 2, **more}
        xo, fo = O.pso_gen_evolve(kind, dim, d["X0"], d["F0"], args.pop("gen"), 40 + k, calls=2, **args)
        xg, fg = a.get(k)
        assert np.array_equal(xg, xo), k
        if kind == P.ROSENBROCK:
            assert np.array_equal(fg, fo.reshape(-1)), k
    a.close()
