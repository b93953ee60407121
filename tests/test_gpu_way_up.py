"""The way up to the level above the coarsest as one matrix of its residual
(Mu).  Its sums hold the coarsest level's call, whose matrix is FP64: so is Mu,
in the FP32 cycles too, which round their vectors only."""
import dataclasses

import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_brick import graded

pytestmark = pytest.mark.gpu


def context(shape, mixed, tdepv=1):
    from citcom_amd.hip import Citcom
    p = dataclasses.replace(graded(*shape), tdepv=tdepv)
    c = Citcom(p, mixed=mixed)
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    return p, c


# levels of 45 to 1089 nodes above the coarsest; three levels (mixed forms with
# three have no exact level), and four whose second is past the exact level's limit
@pytest.mark.parametrize("mixed", [1, 2])
@pytest.mark.parametrize("shape", [(1, 1, 2, 3), (2, 2, 3, 3), (3, 3, 4, 3), (4, 4, 4, 3), (5, 5, 4, 3), (5, 5, 4, 4)])
def test_way_up_of_the_fp32_cycles_keeps_fp64(shape, mixed):
    """FP32 residual in: the FP64 sums over the FP64 matrix, rounded once."""
    p, c = context(shape, mixed)
    r = c.apply("strip", 1, np.random.default_rng(8).normal(size=3 * c.nno(1)))
    r = r.astype(np.float32).astype(np.float64)
    exact, got = c.apply("up", 1, None, r), c.apply("up_f32", 1, None, r)
    c.close()
    assert np.isfinite(exact).all() and np.abs(exact).max() > 0
    assert np.array_equal(got, exact.astype(np.float32).astype(np.float64)), shape


# three levels, at most 500 nodes above the coarsest, viscosity of the deck's law
@pytest.mark.parametrize("shape", [(1, 1, 2, 3), (2, 2, 3, 3), (3, 3, 4, 3), (2, 2, 2, 4)])
def test_way_up_with_varying_viscosity(shape):
    """One FP64 multigrid call with the maps and with the sweeps, which differ by
    the FP32 rounding of the sweeps' increments: 6e-8 of a level's correction a
    sweep, some dozen calls a cycle, 1e-6 of the result."""
    p, c = context(shape, 0)
    assert p.tdepv
    F = c.apply("strip", c.levmax, np.random.default_rng(8).normal(size=3 * c.nno()))
    got = []
    for small in (1, 0):
        c.set_option("small_levels", small)
        d, _, cycles = c.solve_del2_u(F, 0.95 * np.sqrt((F * F).mean()))
        got.append(d)
        assert cycles == 1
    c.close()
    e = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
    assert e < 1e-6, (shape, e)
