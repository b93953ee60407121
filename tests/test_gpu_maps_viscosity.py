"""Which FP64 cycles take the smoother's larger maps (levels of 500 to 1100
nodes): those of a viscosity that is one value.  A finest-level viscosity
uploaded from the host counts by what it holds, in a context whose own law is
constant: such a context then runs the sweeps, as one whose law varies does."""
import dataclasses

import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_brick import graded

pytestmark = pytest.mark.gpu

SHAPES = [(3, 4, 5, 3), (5, 5, 4, 3), (4, 5, 4, 4)]   # 693, 1089, 891 nodes above the coarsest


def context(shape, tdepv):
    from citcom_amd.hip import Citcom
    p = dataclasses.replace(graded(*shape), tdepv=tdepv)
    c = Citcom(p)
    c.initialize(deck.seeded_temperature(p, seed=5))
    return c


def solved(c, F):
    """the operators from the viscosity the context holds, one multigrid call"""
    c.construct_stiffness_B_matrix()
    d, _, cycles = c.solve_del2_u(F, 0.95 * np.sqrt((F * F).mean()))
    assert cycles == 1
    return d


@pytest.mark.parametrize("shape", SHAPES)
def test_uploaded_viscosity_keeps_the_sweeps(shape):
    a, b = context(shape, 0), context(shape, 1)
    rng = np.random.default_rng(8)
    F = a.apply("strip", a.levmax, rng.normal(size=3 * a.nno()))
    evi = (10.0 ** rng.uniform(-2, 2, 8 * a.nel())).astype(np.float32)
    a.get_system_viscosity()
    law, value = solved(a, F), a.download("EVI")
    assert (value == value[0]).all()
    for lev in (-1, a.levmax):
        got = []
        for c in (a, b):
            c.upload("EVI", evi, lev)
            got.append(solved(c, F))
        assert np.array_equal(*got), shape
        # one value uploaded, and the law's own: the maps again
        a.upload("EVI", value, lev)
        assert np.array_equal(solved(a, F), law), shape
        a.upload("EVI", evi, lev)
        a.get_system_viscosity()
        assert np.array_equal(solved(a, F), law), shape
    a.close()
    b.close()
