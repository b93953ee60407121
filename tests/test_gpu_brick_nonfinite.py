"""Compact geometry (brick elements): an element whose centre derivatives are not
finite spoils the rows of its own nodes and no others, as the arrays do.  The
compact form counts the elements past the mesh as zero times another element's
numbers, so that it has to hold finite ones."""
import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_brick import graded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_only_the_elements_own_rows(value):
    from citcom_amd.hip import Citcom
    p = graded(3, 2, 3, 2)
    assert p.aug_lagr
    c = Citcom(p)
    c.initialize(deck.seeded_temperature(p, seed=6))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    good = c.download("K").reshape(c.nno(), -1)
    geo = c.download("GNX").reshape(-1, 216)
    # element 0, z derivatives at the centre (get_elt_g's), with the signs of a brick's corners
    geo[0, 208:216] = np.copysign(np.float32(value), geo[0, 208:216])
    c.upload("GNX", geo)
    c.construct_stiffness_B_matrix()
    K = c.download("K").reshape(c.nno(), -1)
    c.close()
    nox, _, noz = p.dims()
    n = np.arange(c.nno())
    own = (n % noz < 2) & (n // noz % nox < 2) & (n // (noz * nox) < 2)
    assert not np.isfinite(K[own]).all()
    assert np.array_equal(K[~own], good[~own])
