"""Levels whose coefficients are read past the caches (more than 256 MB: the
colour passes; more than 400 MB: the product): the same values, checked on a
level past both limits against the product and one colour sweep in NumPy."""
import numpy as np
import pytest

from citcom_amd import deck
from test_gpu_rect import box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 5, 4, 5), (6, 6, 5, 5)])   # 81x81x65 nodes, 415 MB; 97x97x81, 741 MB
def test_streamed_levels_agree_with_cached_ones(shape):
    """A sweep from zero of a right-hand side that is zero outside the lower
    half in y is, away from the cut, the sweep of the half box's level, whose
    coefficients stay below the limits (same spacing, constant viscosity)."""
    from citcom_amd.hip import Citcom
    mx, my, mz, levels = shape
    rng = np.random.default_rng(3)
    out = []
    for m in (my, 2):
        p = box(mx, m, mz, levels)
        p.tdepv = 0
        c = Citcom(p)
        c.initialize(deck.seeded_temperature(p, seed=5))
        c.get_system_viscosity()
        c.construct_stiffness_B_matrix()
        nox, noy, noz = p.dims(levels - 1)
        if not out:
            F = rng.normal(size=(noy, nox, noz, 3))
        f = F[:noy] if noy < F.shape[0] else F
        d, ad = c.apply("gs0", levels - 1, None, f.ravel(), sweeps=1)
        mv = c.apply("matvec", levels - 1, f.ravel())
        c.close()
        out.append([a.reshape(noy, nox, noz, 3) for a in (d, mv)])
    for a, b in zip(*out):
        n = b.shape[0] - 4
        assert np.isfinite(a).all()
        # the two boxes' FP32 coordinates along y may round differently: a few
        # 1e-7 of the spacing, 1e-5 after differences of a coefficient's terms
        assert np.abs(a[:n] - b[:n]).max() <= 1e-4 * np.abs(b).max()
