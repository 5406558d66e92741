"""One generation of an archipelago (k_step) at the edges of its items: rows that
fill a round of the move, miss one element of it or take several; rosenbrock items
staged in LDS and too long for it; Lennard-Jones individuals from 3 atoms on; each
with the default update rule and with the others.
"""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P
from parity_bars import assert_fitness

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def island(kind, dim, pop, gens, variant=5, topo=2):
    X0, F0 = O.population_init(kind, dim, pop, 7)
    return dict(kind=kind, dim=dim, X0=X0, F0=F0,
                algo=P.pso_params(gen=gens, seed=13, variant=variant, neighb_type=topo))


def evolve(islands, mode, mapping=None):
    a = P.Archipelago(islands, trace=True)
    if mapping:
        a.set_mapping(*mapping)
    a.evolve(mode)
    out = [(a.get(k), a.trace(k)) for k in range(len(islands))]
    a.close()
    return out


@pytest.mark.parametrize("variant,topo", [(5, 2), (1, 2), (6, 3)])
@pytest.mark.parametrize("dim,pop", [
    (2, 33), (32, 32),        # less than a round; exactly one
    (128, 33), (129, 17),     # 32 rows of 4096 elements; 16 rows of 2064
    (255, 9), (256, 17), (257, 16),
    (512, 9), (513, 8),       # 8 rows: 4096 elements are staged, 4104 are not
    (4100, 3),
])
def test_rosenbrock_items_against_oracle(dim, pop, variant, topo):
    """Rosenbrock trajectories are the oracle's bit for bit."""
    X0, F0 = O.population_init(P.ROSENBROCK, dim, pop, 7)
    kw = dict(variant=variant, neighb_type=topo)
    Xo, Fo = O.pso_gen_evolve(P.ROSENBROCK, dim, X0, F0, 4, 13, **kw)
    for mode in (0, 1):
        (X, F), _ = evolve([island(P.ROSENBROCK, dim, pop, 4, variant, topo)], mode)[0]
        assert np.array_equal(X, Xo) and np.array_equal(F, Fo)


@pytest.mark.parametrize("mapping", [None, (0, 0, 1), (1, 0, 0), (1, 4096, 3)])
@pytest.mark.parametrize("variant,topo", [(5, 2), (2, 1)])
def test_fitness_of_the_final_positions(variant, topo, mapping):
    """Every item evaluates the rows that it moved: a row's final fitness is its
    best over the generations and the batch evaluator's (at the kind's bar) at its
    final position; every mapping and the island-by-island launches give one result."""
    cases = [(P.LENNARD_JONES, 3, 300), (P.LENNARD_JONES, 4, 37), (P.LENNARD_JONES, 75, 20), (P.RASTRIGIN, 1, 300),
             (P.ACKLEY, 31, 65), (P.SCHWEFEL, 257, 9), (P.GRIEWANK, 1025, 5), (P.ROSENBROCK, 513, 9)]
    islands = [island(k, d, p, 5, variant, topo) for k, d, p in cases]
    got = evolve(islands, 0, mapping)
    for (kind, dim, _), isl, ((X, F), trace), ((Xp, Fp), tp) in zip(cases, islands, got, evolve(islands, 1)):
        assert np.array_equal(X, Xp) and np.array_equal(F, Fp) and np.array_equal(trace, tp)
        best = np.minimum(np.ravel(isl["F0"]), np.asarray(trace).reshape(5, -1).min(axis=0))
        assert np.array_equal(np.ravel(F), best)
        assert_fitness(kind, X, F, P.bfe_eval_host(kind, dim, X), (kind, dim))


@pytest.mark.parametrize("kind,dim,pop,param", [
    (P.ROSENBROCK, 2, 5, 4),      # fewer elements than threads
    (P.ROSENBROCK, 8, 64, 4),     # 512 elements: one each
    (P.ROSENBROCK, 27, 19, 4),    # 513
    (P.ROSENBROCK, 16, 64, 2),    # 1024: one round, two neighbours
    (P.ROSENBROCK, 25, 41, 6),    # 1025: a second round, six neighbours
    (P.ROSENBROCK, 600, 3, 2),    # rows longer than the workgroup
    (P.ROSENBROCK, 16, 256, 4),   # the largest tile held in LDS
    (P.ROSENBROCK, 17, 256, 4),   # not held
    (P.RASTRIGIN, 1, 16, 2), (P.GRIEWANK, 65, 4, 2), (P.SCHWEFEL, 33, 16, 4), (P.ACKLEY, 300, 5, 4),
    (P.LENNARD_JONES, 3, 9, 4), (P.LENNARD_JONES, 75, 4, 2),
    (P.ACKLEY, 1200, 4, 2), (P.RASTRIGIN, 5001, 3, 2), (P.LENNARD_JONES, 300, 4, 2),  # not held
])
def test_one_shot_tiles(kind, dim, pop, param):
    """pgh_pso_gen_evolve_host of a single tile equals the archipelago's launches bit
    for bit (and the oracle's, for rosenbrock) over two batches of words."""
    X0, F0 = O.population_init(kind, dim, pop, 3)
    prm = dict(gen=35, seed=21, neighb_param=param)
    Xh, Fh = P.pso_gen_evolve_host(kind, dim, X0, F0, P.pso_params(**prm))
    (Xa, Fa), _ = evolve([dict(kind=kind, dim=dim, X0=X0, F0=F0, algo=P.pso_params(**prm))], 1)[0]
    assert np.array_equal(Xh, Xa) and np.array_equal(np.ravel(Fh), np.ravel(Fa))
    if kind == P.ROSENBROCK:
        Xo, Fo = O.pso_gen_evolve(kind, dim, X0, F0, 35, 21, neighb_param=param)
        assert np.array_equal(Xh, Xo) and np.array_equal(Fh, Fo)


@pytest.mark.parametrize("pop", [5, 1800, 1819, 1820, 1821, 2048, 2100])
@pytest.mark.parametrize("islands", [1, 2])
def test_populations_in_and_out(pop, islands):
    """Populations on both sides of 128 KiB (8 elements and a fitness a row) arrive
    and come back unchanged before an evolve call and as the oracle's after one."""
    isl = []
    for k in range(islands):
        X0, F0 = O.population_init(P.ROSENBROCK, 8, pop, 3 + k)
        isl.append(dict(kind=P.ROSENBROCK, dim=8, X0=X0, F0=F0, algo=P.pso_params(gen=2, seed=9)))
    a = P.Archipelago(isl)
    for k, d in enumerate(isl):
        X, F = a.get(k)
        assert np.array_equal(X, d["X0"]) and np.array_equal(F, np.ravel(d["F0"]))
    a.evolve()
    for k, d in enumerate(isl):
        X, F = a.get(k)
        Xo, Fo = O.pso_gen_evolve(P.ROSENBROCK, 8, d["X0"], d["F0"], 2, 9)
        assert np.array_equal(X, Xo) and np.array_equal(F, np.ravel(Fo))
    a.close()
