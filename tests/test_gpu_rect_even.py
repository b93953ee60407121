"""Joined colour passes (k_gs_rect) on levels with an even number of planes,
whose last plane is one of the odd planes' launch and has no plane beyond it:
the bits of one launch per colour."""
import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_rect import box

pytestmark = pytest.mark.gpu


# two levels, the coarser one (8x6x6, 4x8x10, 13x4x8 nodes along x, y, z) too
# large for the one-workgroup smoother
@pytest.mark.parametrize("shape", [(7, 5, 5, 2), (3, 7, 9, 2), (12, 3, 7, 2)])
def test_even_planes_same_bits(shape):
    from citcom_amd.hip import Citcom
    p = box(*shape)
    c = Citcom(p)
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    rng = np.random.default_rng(8)
    assert p.dims(0)[1] % 2 == 0
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
