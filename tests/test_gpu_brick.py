"""Kernels that read an element's geometry in its compact form (brick elements
of one coordinate array per axis) against the same ones on the arrays: the
same bits.  A changed entry of one element, read by the gradient operator
only, sends the whole level to the arrays; the entry put back, it returns."""
import dataclasses

import numpy as np
import pytest

from citcom_amd import deck

pytestmark = pytest.mark.gpu

# (mgunitx, mgunity, mgunitz, levels): two and three element layers, ragged
# tiles, more columns than one workgroup of the layer sums, more layers than a wave
BOXES = [(1, 1, 1, 2), (3, 2, 3, 2), (3, 5, 2, 3), (9, 2, 2, 3), (1, 3, 9, 4)]


def graded(mx, my, mz, levels):
    keys = deck.workload("tiny_tdep")
    f = 1 << (levels - 1)
    keys["levels"] = levels
    for ax, m in zip("xyz", (mx, my, mz)):
        keys["mgunit" + ax], keys["dimen" + ax] = m, m / mz
        keys[2 * ax], keys["n" + ax] = f"0,{m / mz}", f"1,{m * f + 1}"
    p = deck.problem_from_deck({k: str(v) for k, v in keys.items()})
    rng = np.random.default_rng(3)
    co = []
    for c in p.coords:
        h = rng.uniform(0.5, 1.5, len(c) - 1).cumsum()
        co.append(np.concatenate([[0.0], h / h[-1] * c[-1]]).astype(np.float32))
    return dataclasses.replace(p, coords=tuple(co))


@pytest.mark.parametrize("shape", BOXES)
def test_compact_geometry_same_bits(shape):
    from citcom_amd.hip import Citcom
    p = graded(*shape)
    rng = np.random.default_rng(4)
    c = Citcom(p)
    T = deck.seeded_temperature(p, seed=6)
    Tdot, V = rng.normal(size=c.nno()).astype(np.float32), (200 * rng.normal(size=3 * c.nno())).astype(np.float32)
    geo = c.download("GNX")
    other = geo.reshape(-1, 216).copy()
    other[-1, 192 + 8 * 2 + 6] *= np.float32(1.25)

    def run():
        c.initialize(T)
        c.get_system_viscosity()
        c.construct_stiffness_B_matrix()
        out = {"K": c.download("K").reshape(c.nno(), -1), "BI": c.download("BI").reshape(c.nno(), -1),
               "EG": c.download("EG").reshape(c.nel(), -1)}
        for k, a in (("T", T), ("Tdot", Tdot), ("V", V)):
            c.upload(k, a)
        out["nu"] = np.array(c.heat_flux())
        out["dt"] = np.array(c.PG_timestep()["timestep"])
        for k in ("T", "Tdot", "buoyancy"):
            out[k] = c.download(k)
        return out

    compact = run()
    c.upload("GNX", other)
    arrays = run()
    c.upload("GNX", geo)
    again = run()
    noz, nox = p.dims()[2], p.dims()[0]
    n = np.arange(c.nno())
    far = (n % noz < noz - 2) | (n // noz % nox < nox - 2)   # not in a block with the changed element
    assert not np.array_equal(arrays["EG"], compact["EG"])
    assert np.isfinite(compact["nu"]).all() and np.isfinite(compact["T"]).all()
    for k, a in compact.items():
        assert np.array_equal(again[k], a), k
        if k == "EG":
            assert np.array_equal(arrays[k][:-1], a[:-1]), k
        elif k in ("K", "BI"):
            assert np.array_equal(arrays[k][far], a[far]), k
        else:
            assert np.array_equal(arrays[k], a), k
    c.close()
