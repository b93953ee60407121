"""Joined colour passes (k_gs_rect: four colours of a plane's strip in one
launch) against one launch per colour: the same bits on every level, from zero
and from a guess, at the edges of the strips, segments and shapes."""
import numpy as np
import pytest

from citcom_amd import deck

pytestmark = pytest.mark.gpu

# (mgunitx, mgunity, mgunitz, levels): even coarsest node counts, one strip,
# remainders of the strips, lines cut into segments (narrow: past 17 nodes,
# wide: past 41), both shapes, the largest level of the rule
BOXES = [(3, 1, 1, 3), (2, 2, 5, 3), (5, 3, 2, 3), (1, 2, 9, 4), (1, 1, 5, 5), (4, 4, 4, 4), (5, 2, 3, 4), (2, 3, 11, 4)]


def box(mx, my, mz, levels):
    keys = deck.workload("tiny_tdep")
    f = 1 << (levels - 1)
    keys["levels"] = levels
    for ax, m in zip("xyz", (mx, my, mz)):
        keys["mgunit" + ax], keys["dimen" + ax] = m, m / mz
        keys[2 * ax], keys["n" + ax] = f"0,{m / mz}", f"1,{m * f + 1}"
    return deck.problem_from_deck({k: str(v) for k, v in keys.items()})


@pytest.mark.parametrize("shape", BOXES)
def test_joined_colour_passes_same_bits(shape):
    from citcom_amd.hip import Citcom
    p = box(*shape)
    c = Citcom(p)
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    rng = np.random.default_rng(8)
    for lev in range(p.levels):
        n = 3 * c.nno(lev)
        F, d0 = rng.normal(size=n), rng.normal(size=n)
        got = {}
        for small in (1, 0):
            c.set_option("small_levels", small)
            got[small] = [c.apply(op, lev, d0, F, sweeps=s) for op, s in (("gs0", 1), ("gs0", 2), ("gs1", 1), ("gs1", 3))]
        for a, b in zip(got[1], got[0]):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), (shape, lev)
    c.close()
