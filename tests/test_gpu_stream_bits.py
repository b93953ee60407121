"""Coefficients read past the caches (large levels; here, by the option, any)
against plain reads: the same bits from the colour pass and the product of large
levels, with FP64 and FP32 vectors on FP32 coefficients and FP32 vectors on FP16
ones."""
import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_rect import box

pytestmark = pytest.mark.gpu


# finest levels of more than 20000 nodes, below which the product has another
# kernel: 33x33x33, 41x33x25 and, past both limits by its size, 81x81x65 nodes
@pytest.mark.parametrize("mixed", [0, 1, 2])
@pytest.mark.parametrize("shape", [(4, 4, 4, 4), (5, 4, 3, 4), (5, 5, 4, 5)])
def test_same_bits(shape, mixed):
    from citcom_amd.hip import Citcom
    p = box(*shape)
    c = Citcom(p, mixed=mixed)
    c.set_option("box_gs", 0)
    c.set_option("small_levels", 0)   # one launch per colour
    c.initialize(deck.seeded_temperature(p, seed=5))
    c.get_system_viscosity()
    c.construct_stiffness_B_matrix()
    rng = np.random.default_rng(8)
    for lev in (c.levmax - 1, c.levmax):
        n = 3 * c.nno(lev)
        F, d0 = rng.normal(size=n), rng.normal(size=n)
        got = {}
        for stream in (-1, 0, 1):
            c.set_option("stream", stream)
            got[stream] = [a for sfx in (("", "_f32") if mixed else ("",))
                           for a in (*c.apply("gs1" + sfx, lev, d0, F, sweeps=1), c.apply("matvec" + sfx, lev, d0))]
        for a, b, s in zip(*got.values()):
            assert np.isfinite(a).all() and np.abs(a).max() > 0
            assert np.array_equal(a, b) and np.array_equal(a, s), (shape, lev)
    c.close()


def test_option_values():
    from citcom_amd.hip import ChipError, Citcom
    c = Citcom(box(1, 1, 1, 2))
    for bad in (-2, 2):
        with pytest.raises(ChipError):
            c.set_option("stream", bad)
    c.close()
