"""The FP64 matrices of the smoother calls on levels of 500 to 1100 nodes (Ma,
Mb) and of the way up (Mu) are those calls in FP64: their columns carry no
increment rounded to FP32, so that a call is as near to FP64 as its sums, where
the sweeps it stands for are 2e-8 to 3e-8 away.  81 products a row, a dozen
updates of a node a call, rows of at most 3300 terms: 1e-13 of the result."""
import numpy as np
import pytest

from box_model import sweep_model
from test_gpu_way_up import context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 4, 5, 3), (4, 4, 4, 3), (5, 5, 4, 3)])   # 693, 729, 1089 nodes
def test_wide_maps_are_the_calls_in_fp64(shape):
    p, c = context(shape, 0, tdepv=0)
    nox, noy, noz = p.dims(1)
    K, BI = c.download("K", 1), c.download("BI", 1)
    rng = np.random.default_rng(3)
    F, d0 = (rng.normal(size=3 * c.nno(1)) for _ in range(2))
    for guess in (0, 1):
        exact = d0 if guess else np.zeros_like(F)
        for _ in range(p.down_heavy):
            exact = sweep_model(K, BI, F, exact, (noz, nox, noy), boxes=False)
        err = np.abs(c.apply(f"map{guess}", 1, d0, F) - exact).max() / np.abs(exact).max()
        print("[gpu-test]", shape, guess, f"{err:.2e}", flush=True)
        assert err < 1e-13, (shape, guess, err)
    c.close()


SMALL = [(1, 1, 2, 3), (2, 2, 3, 3), (3, 3, 4, 3)]   # 45 to 441 nodes


@pytest.mark.parametrize("shape,tdepv", [(s, t) for s in SMALL for t in (0, 1)] + [((4, 4, 4, 3), 0), ((5, 5, 4, 3), 0)])
def test_way_up_is_the_call_in_fp64(shape, tdepv):
    """Mu r against the restriction, the coarsest level's matrix, the
    prolongation and the sweeps in FP64 (levels past 500 nodes: constant viscosity)."""
    p, c = context(shape, 0, tdepv=tdepv)
    nox, noy, noz = p.dims(1)
    K, BI = c.download("K", 1), c.download("BI", 1)
    r = c.apply("strip", 1, np.random.default_rng(3).normal(size=3 * c.nno(1)))
    v = c.apply("coarse", 0, None, c.apply("strip", 0, c.apply("project", 1, r)))
    exact = c.apply("strip", 1, c.apply("interp", 1, v))
    for _ in range(p.up_heavy):
        exact = sweep_model(K, BI, r, exact, (noz, nox, noy), boxes=False)
    err = np.abs(c.apply("up", 1, None, r) - exact).max() / np.abs(exact).max()
    print("[gpu-test]", shape, tdepv, f"{err:.2e}", flush=True)
    c.close()
    assert err < 1e-13, (shape, err)
