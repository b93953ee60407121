"""The joined colour passes' partition (tests/rect_model.py), on the CPU: what a
workgroup reads and writes stays in its staged region and its limits, every
node is written once per sweep, and a sweep made of these launches gives the
8-colour sweep's bits."""
import numpy as np
import pytest

import rect_model as rm

# (nz, nx, ny): the levels of the workloads here, thin and long boxes, even
# node counts (coarsest levels), the limits of the shapes
GRIDS = [(2, 2, 2), (3, 5, 5), (4, 4, 2), (5, 5, 5), (9, 9, 9), (3, 3, 17), (17, 17, 17), (9, 17, 17), (33, 17, 9),
         (20, 4, 4), (21, 5, 3), (41, 21, 5), (42, 6, 4), (43, 5, 3), (11, 21, 13), (61, 9, 5), (65, 9, 5), (81, 13, 5),
         (129, 5, 5), (130, 6, 4), (257, 3, 3), (3, 131, 3), (2, 257, 2), (33, 33, 33), (17, 33, 33)]
LARGE = [(33, 65, 65), (65, 129, 129), (41, 81, 49), (129, 257, 257)]


@pytest.mark.parametrize("nz,nx,ny", GRIDS + LARGE)
@pytest.mark.parametrize("shape", sorted(rm.SHAPES))
def test_workgroups_within_limits(shape, nz, nx, ny):
    p = rm.part(shape, nz, nx, ny)
    assert p is not None       # every level has a partition of every shape
    for jpar, n in rm.launches(p, ny):
        seen = {}
        for b in range(n) if n <= 3000 else list(range(200)) + list(range(n - 200, n)):
            j, colours, (kr0, kr1, ir0, ir1), own_k, own_i = rm.workgroup(p, nz, nx, ny, jpar, b)
            assert j < ny and kr0 % 2 == 0
            updated = set()
            for kp, ip, nodes in colours:
                assert len(nodes) <= p["nodes"]
                for k, i in nodes:
                    assert k % 2 == kp and i % 2 == ip and 0 <= k < nz and 0 <= i < nx
                    assert kr0 < k < kr1 and ir0 < i < ir1     # its neighbours are staged
                    updated.add((k, i))
            for i in own_i:
                for k in own_k:
                    assert (k, i) in updated
                    assert seen.setdefault((j, k, i), b) == b   # nobody else writes it
        if n <= 3000:
            assert len(seen) == len(range(jpar, ny, 2)) * nz * nx


def sweep(d, K, F):
    """8-colour sweep of a scalar 27-point operator"""
    d = d.copy()
    ny, nx, nz = d.shape
    for c in range(8):
        new = d.copy()
        for j in range(c >> 2, ny, 2):
            for i in range((c >> 1) & 1, nx, 2):
                for k in range(c & 1, nz, 2):
                    new[j, i, k] = update(d, K, F, j, i, k)
        d = new
    return d


def update(d, K, F, j, i, k):
    ny, nx, nz = F.shape
    s = 0.0
    for t in range(27):
        kk, ii, jj = k + t % 3 - 1, i + (t // 3) % 3 - 1, j + t // 9 - 1
        if 0 <= kk < nz and 0 <= ii < nx and 0 <= jj < ny:
            s += K[j, i, k, t] * d[jj, ii, kk]
    return d[j, i, k] + (F[j, i, k] - s) * 0.9


def joined_sweep(p, din, K, F):
    ny, nx, nz = din.shape
    dout = np.full_like(din, np.nan)
    for jpar, n in rm.launches(p, ny):
        # what the workgroups of one launch see: nothing another one writes
        view = np.where((np.arange(ny) % 2 == jpar)[:, None, None], din, dout if jpar else din).copy()
        for b in range(n):
            j, colours, (kr0, kr1, ir0, ir1), own_k, own_i = rm.workgroup(p, nz, nx, ny, jpar, b)
            local = np.full_like(view, np.nan)      # what is not staged is not there
            s = np.s_[max(j - 1, 0):j + 2, max(ir0, 0):ir1 + 1, max(kr0, 0):kr1 + 1]
            local[s] = view[s]
            for _, _, nodes in colours:
                new = [update(local, K, F, j, i, k) for k, i in nodes]
                for (k, i), v in zip(nodes, new):
                    local[j, i, k] = v
            dout[j, own_i[0]:own_i[-1] + 1, own_k[0]:own_k[-1] + 1] = \
                local[j, own_i[0]:own_i[-1] + 1, own_k[0]:own_k[-1] + 1]
    return dout


@pytest.mark.parametrize("nz,nx,ny", [(2, 2, 2), (4, 4, 2), (5, 5, 5), (3, 9, 5), (9, 7, 3), (4, 3, 6), (21, 4, 3)])
@pytest.mark.parametrize("shape", ["narrow", "wide", "cut"])
def test_same_bits_as_eight_colours(shape, nz, nx, ny):
    p = rm.part("narrow" if shape == "cut" else shape, nz, nx, ny)
    if shape == "cut":      # short segments, as on large levels
        p.update({"Wz": 2, "ns": max(1, -(-(nz - 1) // 2))})
    rng = np.random.default_rng(nz * 100 + nx * 10 + ny)
    K, F, d = rng.normal(size=(ny, nx, nz, 27)), rng.normal(size=(ny, nx, nz)), rng.normal(size=(ny, nx, nz))
    assert np.array_equal(joined_sweep(p, d, K, F), sweep(d, K, F))
