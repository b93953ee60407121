"""Arrays of an operator uploaded between two solves without a rebuild.  The
transfers and the sweeps read them as they are; a matrix of the level was formed
at the last rebuild and is left out until the next, except the maps of at most
1500 unknowns, which have always stood for the last rebuild's arrays."""
import dataclasses

import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_brick import graded

pytestmark = pytest.mark.gpu


def context(shape, mixed):
    from citcom_amd.hip import Citcom
    p = dataclasses.replace(graded(*shape), tdepv=0)
    c = Citcom(p, mixed=mixed)
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    return c


def solve(c, F):
    d, _, cycles = c.solve_del2_u(F, 0.95 * np.sqrt((F * F).mean()))
    assert cycles == 1
    return d


def check(c, F, which, arr, lev, mixed, counts=True):
    """one call with `arr` uploaded after the rebuild, against the sweeps and
    transfers alone (up to the maps' rounding: 1e-6 plain, 1e-5 in the FP32
    cycles), and the old call's bits after the next rebuild of the old array"""
    before, old = solve(c, F), c.download(which, lev)
    c.upload(which, arr, lev)
    at_once = solve(c, F)
    c.set_option("small_levels", 0)
    sweeps = solve(c, F)
    c.set_option("small_levels", 1)
    c.upload(which, old, lev)
    c.construct_stiffness_B_matrix()
    assert np.array_equal(solve(c, F), before)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    print("[gpu-test]", which, mixed, f"{rel(at_once, sweeps):.1e} {rel(before, sweeps):.1e}", flush=True)
    assert rel(at_once, sweeps) < (1e-5 if mixed else 1e-6)
    assert not counts or rel(before, sweeps) > 1e-3


# 147, 729 and 1089 nodes above the coarsest of three levels
@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("shape", [(3, 3, 1, 3), (4, 4, 4, 3), (5, 5, 4, 3)])
def test_uploaded_transfer_weights_count_at_once(shape, mixed):
    """The coarsest level's mass matrix scales its restriction."""
    c = context(shape, mixed)
    rng = np.random.default_rng(8)
    F = c.apply("strip", c.levmax, rng.normal(size=3 * c.nno()))
    mass = c.download("MASS", 0)
    check(c, F, "MASS", mass * rng.uniform(0.5, 1.5, mass.size).astype(np.float32), 0, mixed)
    c.close()


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("shape,lev", [((4, 4, 4, 3), 1), ((5, 5, 4, 3), 1), ((1, 1, 1, 5), 2)])
def test_uploaded_diagonal_counts_at_once_on_larger_maps(shape, lev, mixed):
    """BI of a level of more than 500 nodes, or of 125 nodes two above the
    coarsest, halved: the plain form's sweeps read it (the FP32 cycles a copy
    made at the rebuild, which is left as it was)."""
    c = context(shape, mixed)
    rng = np.random.default_rng(8)
    F = c.apply("strip", c.levmax, rng.normal(size=3 * c.nno()))
    check(c, F, "BI", 0.5 * c.download("BI", lev), lev, mixed, counts=not mixed)
    c.close()
