"""An archipelago with more velocity draws than two shares of 2^15 words per CU: an
island whose shares are larger, and a small one beside it.  Bit for bit with the oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu


def test_velocities_of_a_large_island():
    sizes = [(33001, 521), (30, 11), (700, 190)]  # 34.4 M words, 660 and 266000
    isl, start = [], []
    for k, (pop, dim) in enumerate(sizes):
        X = np.random.default_rng(k).uniform(-5.0, 10.0, (pop, dim))
        F = P.bfe_eval_host(P.ROSENBROCK, dim, X).reshape(-1)
        start.append((X, F))
        isl.append(dict(kind=P.ROSENBROCK, dim=dim, X0=X, F0=F, algo=P.pso_params(gen=1, seed=k + 5)))
    a = P.Archipelago(isl)
    a.evolve()
    for k, (pop, dim) in enumerate(sizes):
        X, F = start[k]
        ref = O.pso_gen_evolve(O.ROSENBROCK, dim, X, F, 1, k + 5)
        x, f = a.get(k)
        assert np.array_equal(x, ref[0]) and np.array_equal(f.reshape(-1), ref[1]), k
    a.close()
