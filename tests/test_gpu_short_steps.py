"""Bookkeeping kernels of a build at the sizes where their shape changes.

The scan of grid-cell counts takes one block up to 16384 cells and tiles above;
a collect of restarting seeds takes blocks of 2048 seeds; a chain that leaves
no seed uncertified, overflowed or failed skips the passes after it, and one
that does must not.  Topology must equal the oracle's, whole numbers throughout.
"""
import numpy as np
import pytest

from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import uniform_points

pytestmark = pytest.mark.gpu

SUCCESS = 4
KEYS = ("status", "kcert", "face_counts", "face_ptr", "neighbor_cell", "face_normal")


def _same(ctx, pts, **kw):
    g = api.Mesh(ctx, pts, **kw)
    ref = O.Mesh(pts, kw["boundary"], **{a: b for a, b in kw.items() if a != "boundary"})
    out = g.copy_out()
    for key in KEYS:
        assert np.array_equal(out[key], ref.get(key)), key
    assert g.n_failed == int((out["status"] != SUCCESS).sum())
    assert g.num_faces == int(out["face_counts"].sum())
    return g


# 2D grids of up to 130 cells a side (16384 cells: 128), rows so short that
# nearly every seed restarts (the collect's list is about as long as its input)
@pytest.mark.parametrize("n", [800, 2047, 2048, 2049, 4097, 50600, 51000, 51700, 53000])
@pytest.mark.parametrize("k,restart", [(6, True), (24, True), (12, False)])
def test_collect_and_scan_edges(ctx, n, k, restart):
    _same(ctx, uniform_points(n, 2, n), boundary="reflective", k=k, restart=restart)


@pytest.mark.parametrize("k_max", [16, 32])
def test_chains_that_leave_work(ctx, k_max):
    """A cap on the rows leaves uncertified seeds to the completion pass, and a
    shell of neighbours around one seed overflows the fast kernel's slots."""
    u = uniform_points(400, 3, 5) - 0.5
    shell = 0.5 + 0.05 * u / np.linalg.norm(u, axis=1)[:, None]
    base = uniform_points(6000, 3, 6)
    base = base[np.linalg.norm(base - 0.5, axis=1) > 0.1]
    pts = np.concatenate([base, shell[:40], [[0.5, 0.5, 0.5]]])
    g = _same(ctx, pts, boundary="reflective", k=16, restart=True, k_max=k_max)
    assert g.n_ball > 0 or g.n_restarted > 0
