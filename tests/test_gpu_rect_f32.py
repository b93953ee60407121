"""Joined colour passes (k_gs_rect) of the FP32 cycles, with FP32 and with FP16
(BI-scaled) coefficients, against one launch per colour: the same bits on every
level, from zero and from a guess, in both workgroup shapes."""
import numpy as np
import pytest

from citcom_amd import deck
import rect_model as rm
from test_gpu_rect import BOXES, box

SHAPES = BOXES + [(5, 5, 5, 4), (7, 5, 5, 2)]


def shape_of(nz, nx, ny):
    """the workgroup shape a level gets: at most two narrow workgroups to a CU, or one wide one"""
    for shape, most in (("narrow", 512), ("wide", 256)):
        p = rm.part(shape, nz, nx, ny)
        if p and (ny + 1) // 2 * p["nstrip"] * p["ns"] <= most:
            return shape


def test_shapes_reach_every_kernel():
    """FP32 coefficients: every level; FP16 ones (mixed = 2): the two finest, two above the coarsest."""
    seen = {4: set(), 2: set()}
    for s in SHAPES:
        p = box(*s)
        for lev in range(p.levels):
            nox, noy, noz = p.dims(lev)
            shape = shape_of(noz, nox, noy)
            seen[4].add(shape)
            if lev >= max(2, p.levels - 2):
                seen[2].add(shape)
    assert seen[4] >= {"narrow", "wide"} and seen[2] >= {"narrow", "wide"}, seen


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_joined_colour_passes_of_the_fp32_cycles_same_bits(shape, mixed):
    from citcom_amd.hip import Citcom
    p = box(*shape)
    c = Citcom(p, mixed=mixed)
    c.set_option("box_gs", 0)   # the levels the boxes would take are smoothed by colour passes
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
            got[small] = [c.apply(op, lev, d0, F, sweeps=s)
                          for op, s in (("gs0_f32", 1), ("gs0_f32", 2), ("gs1_f32", 1), ("gs1_f32", 3))]
        for a, b in zip(got[1], got[0]):
            assert np.isfinite(a[0]).all() and np.abs(a[0]).max() > 0
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), (shape, lev)
    c.close()
