"""Windows of the clip's row walk: row entries that cannot cut the cell are
passed over without a conflict test, 16 entries at a time.

Integer results (statuses, certified k, topology) must equal the oracle's, which
tests every entry: rows around multiples of the window, restarts that start
inside a window, rows without restarts, and sets where a conflict
determinant is near its eps though its plane is far (nearly degenerate
lattices, clusters far below the box's scale), where passing over would lose
the needs_exact_predicates flag.
"""
import numpy as np
import pytest

from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import jittered_lattice, uniform_points

pytestmark = pytest.mark.gpu

KEYS = ("status", "kcert", "face_counts", "face_ptr", "neighbor_cell", "face_normal")


def _same(ctx, pts, **kw):
    g = api.Mesh(ctx, pts, **kw)
    ref = O.Mesh(pts, kw["boundary"], **{a: b for a, b in kw.items() if a != "boundary"})
    out = g.copy_out()
    for key in KEYS:
        assert np.array_equal(out[key], ref.get(key)), key
    return out


@pytest.mark.parametrize("restart", [True, False])
@pytest.mark.parametrize("dim,k", [(2, 7), (2, 15), (2, 17), (3, 15), (3, 16), (3, 17), (3, 31), (3, 33), (3, 49)])
def test_rows_around_the_window(ctx, dim, k, restart):
    _same(ctx, uniform_points(3000 if dim == 2 else 14000, dim, 100 + k), boundary="reflective", k=k, restart=restart)


@pytest.mark.parametrize("dim,amp", [(2, 1e-13), (2, 1e-9), (3, 1e-13), (3, 1e-11), (3, 1e-9), (3, 1e-6)])
def test_nearly_degenerate_lattices(ctx, dim, amp):
    pts = jittered_lattice(40 if dim == 2 else 24, dim, 3, amp=amp)
    _same(ctx, pts, boundary="reflective", k=32, restart=True)


@pytest.mark.parametrize("scale", [1e-4, 1e-6, 1e-7])
def test_clusters_far_below_the_box(ctx, scale):
    pts = np.concatenate([scale * (uniform_points(4000, 3, 5) - 0.5) + 0.5, uniform_points(12000, 3, 6)])
    _same(ctx, pts, boundary="reflective", k=32, restart=True, k_max=128)


@pytest.mark.parametrize("faces", [12, 15, 16, 17, 20, 21, 30, 60])
def test_2d_cells_of_many_faces(ctx, faces):
    """Rings of points around a seed: cells around the 16 vertex slots and 24
    planes (20 besides the box) of the fast 2D kernel, and beyond them (60 and
    the box's 4 fill max_p: the next row entry overflows the cell)."""
    a = 2 * np.pi * (np.arange(faces) + 0.25) / faces
    rings = [np.concatenate([[[cx, cy]], np.stack([cx + 0.04 * np.cos(a), cy + 0.04 * np.sin(a)], 1)])
             for cx, cy in ((0.31, 0.42), (0.68, 0.27), (0.5, 0.8))]
    base = uniform_points(3000, 2, 91)
    keep = np.all([np.hypot(*(base - r[0]).T) > 0.09 for r in rings], axis=0)
    pts = np.concatenate([base[keep]] + rings)
    for k in (16, 32):
        out = _same(ctx, pts, boundary="reflective", k=k, restart=True)
        assert faces == 60 or out["face_counts"].max() >= faces
