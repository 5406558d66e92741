"""Velocities of islands with the smallest velocity limits: U(minv, maxv) rounds as
std::uniform_real_distribution does also where the width is near the subnormals.
Positions at the origin show every bit of them.  Bit for bit with the oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

MAX_VEL = [1e-285, 1e-290, 1e-300, 1e-310, 5e-324]


def origin(pop, dim):
    return np.zeros((pop, dim)), np.zeros(pop)


@pytest.mark.parametrize("max_vel", MAX_VEL)
@pytest.mark.parametrize("pop,dim,gen", [(10, 6, 2), (40, 33, 1)])
def test_one_shot(pop, dim, gen, max_vel):
    X, F = origin(pop, dim)
    got = P.pso_gen_evolve_host(P.RASTRIGIN, dim, X, F, P.pso_params(gen=gen, seed=3, max_vel=max_vel))
    ref = O.pso_gen_evolve(O.RASTRIGIN, dim, X, F, gen, 3, max_vel=max_vel)
    assert np.any(ref[0] != 0.0)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1].reshape(-1), ref[1])


@pytest.mark.parametrize("max_vel", MAX_VEL)
def test_archipelago(max_vel):
    """An island whose velocities are one share of the draws, and one whose are
    several (more than 2^17 words)."""
    sizes = [(12, 7), (1100, 65)]
    isl = []
    for k, (pop, dim) in enumerate(sizes):
        X, F = origin(pop, dim)
        isl.append(dict(kind=P.RASTRIGIN, dim=dim, X0=X, F0=F,
                        algo=P.pso_params(gen=2, seed=k + 5, max_vel=max_vel)))
    a = P.Archipelago(isl)
    a.evolve()
    for k, (pop, dim) in enumerate(sizes):
        X, F = origin(pop, dim)
        ref = O.pso_gen_evolve(O.RASTRIGIN, dim, X, F, 2, k + 5, max_vel=max_vel)
        x, f = a.get(k)
        assert np.array_equal(x, ref[0]) and np.array_equal(f.reshape(-1), ref[1]), k
    a.close()
