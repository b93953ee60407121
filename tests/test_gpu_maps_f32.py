"""Smoother calls of the FP32 cycles as matrices rounded to FP32 (FP64 sums)
against the same call in FP32 sweeps: both are measured from the call in FP64
(tests/box_model.py with one box for the level), and the matrices are no
further from it."""
import numpy as np
import pytest

from box_model import sweep_model
from test_gpu_way_up import context

pytestmark = pytest.mark.gpu


# levels of 441 to 1089 nodes above the coarsest of three, contrast of the deck's law
@pytest.mark.parametrize("shape", [(3, 3, 4, 3), (3, 4, 5, 3), (4, 4, 4, 3), (5, 5, 4, 3)])
def test_maps_no_further_from_fp64_than_sweeps(shape):
    p, c = context(shape, 1)
    nox, noy, noz = p.dims(1)
    K, BI = c.download("K", 1), c.download("BI", 1)
    f32 = lambda v: v.astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(3)
    F, d0 = (f32(rng.normal(size=3 * c.nno(1))) for _ in range(2))
    for guess in (0, 1):
        exact = d0 if guess else np.zeros_like(F)
        for _ in range(p.down_heavy):
            exact = sweep_model(K, BI, F, exact, (noz, nox, noy), boxes=False)
        err = {}
        for name, d in (("map", c.apply(f"map{guess}_f32", 1, d0, F)),
                        ("sweeps", c.apply(f"gs{guess}_f32", 1, d0, F, sweeps=p.down_heavy)[0]),
                        ("map64", c.apply(f"map{guess}", 1, d0, F)),
                        ("sweeps64", c.apply(f"gs{guess}", 1, d0, F, sweeps=p.down_heavy)[0])):
            err[name] = np.linalg.norm(d - exact) / np.linalg.norm(exact)
        print("[gpu-test]", shape, guess, {k: f"{v:.2e}" for k, v in err.items()}, flush=True)
        assert err["map"] <= err["sweeps"], (shape, guess, err)
    c.close()
