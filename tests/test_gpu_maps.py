"""The smoother calls of small levels as matrices (k_map_columns, k_map_apply,
the way up as one matrix) against the sweeps: one multigrid call each.  The two
differ by the FP32 rounding of the sweeps' increments, 6e-8 of a level's
correction a sweep, and the dozen calls of a cycle: 1e-6 of the result; the
FP32 cycles add their own rounding, 1e-5."""
import dataclasses

import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_brick import graded

pytestmark = pytest.mark.gpu

# (mgunitx, mgunity, mgunitz, levels): rows of at most 8 terms a lane, of one
# batch more (9, 20, 21, 36), of the largest level, two batches; two levels of maps; a level
# just past the rule; three levels (no exact level in the mixed forms)
BOXES = [(1, 1, 1, 4), (2, 2, 3, 3), (2, 3, 3, 3), (2, 4, 4, 3), (3, 3, 4, 3), (4, 4, 4, 3), (3, 4, 5, 3), (1, 1, 1, 5),
         (4, 4, 5, 3), (5, 5, 4, 3), (5, 5, 5, 3), (4, 5, 4, 4), (2, 1, 3, 5)]


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("shape", BOXES)
def test_maps_against_sweeps(shape, mixed):
    from citcom_amd.hip import Citcom
    p = dataclasses.replace(graded(*shape), tdepv=0)   # the plain form's larger maps: constant viscosity
    c = Citcom(p, mixed=mixed)
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    F = np.random.default_rng(8).normal(size=3 * c.nno())
    F = c.apply("strip", c.levmax, F)
    got = []
    for small in (1, 0):
        c.set_option("small_levels", small)
        d, _, cycles = c.solve_del2_u(F, 0.95 * np.sqrt((F * F).mean()))
        got.append(d)
        assert cycles == 1
    c.close()
    e = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
    assert e < (1e-5 if mixed else 1e-6), (shape, mixed, e)
