"""The face tables of the moving-mesh update on both sides of the size at
which their kernel changes (131072 seeds: lanes per cell below, a thread per
cell above).

A batch of two boxes counts as one mesh of both, so it takes the upper form
where each box alone takes the lower one; a box's states must be the same to
the bit either way (each face is solved once, by the same cell, and summed in
the same order).
"""
import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd.generators import batch_points, kelvin_helmholtz_state, sod_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,boundary,k", [(2, 67000, "periodic", 16), (2, 70001, "reflective", 20),
                                              (3, 68003, "reflective", 32), (3, 45000, "periodic", 24)])
def test_two_boxes_equal_single_runs(ctx, dim, n, boundary, k):
    sizes = np.array([n, n - 37])
    pts = batch_points(sizes, dim, 900 + dim)
    st = kelvin_helmholtz_state(pts) if boundary == "periodic" else sod_state(pts, 1.4)
    kw = dict(boundary=boundary, buff=0.04 if dim == 2 else 0.1, k=k, gamma=1.4, cfl=0.3, flux="physical", move_mesh=True)
    B = api.Batch(ctx, sizes, pts, *st, **kw)
    B.step()
    B.step()
    got = B.get()
    B.free()
    off = 0
    for m in sizes:
        sl = slice(off, off + m)
        s = api.Simulation(ctx, pts[sl], *(a[sl] for a in st), **kw)
        s.step()
        s.step()
        for a, b in zip(got, s.get()):
            assert np.array_equal(a[sl], b)
        s.free()
        off += m
