"""Neighbour rows of seeds in and beside crowded grid cells.

The ball a query searches first is sized from the sub-cells around it, from
the cells that are not crowded, or (rows that continue a saved one) from the
neighbours it knows; the rows must equal the oracle's whatever the guess:
clusters far below a cell, at its size and above, clusters on the box's edge,
empty sub-cells and coincident points inside a crowded cell, and rows longer
than a cluster.
"""
import numpy as np
import pytest

from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import uniform_points

pytestmark = pytest.mark.gpu


def _clusters(dim, scale, seed):
    rng = np.random.default_rng(seed)
    base = uniform_points(3000 if dim == 2 else 14000, dim, seed)
    at = [np.full(dim, 0.5), np.full(dim, 0.013), np.r_[0.999, np.full(dim - 1, 0.31)]]
    return np.clip(np.concatenate([base] + [c + scale * rng.standard_normal((700, dim)) for c in at]), 0.0, 0.999999)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("scale", [1e-1, 2e-2, 3e-3, 1e-5])
def test_rows_equal_the_oracle(ctx, dim, scale):
    pts = _clusters(dim, scale, 11)
    p = np.concatenate([pts, pts[-40:], pts[-40:-20]])
    kp = api.KnnProblem(ctx, p)
    for k in (16, 32, 64, 200):
        kp.solve(k)
        assert np.array_equal(kp.get_knearest(), O.knn(p, k)[3]), k
    kp.free()


@pytest.mark.parametrize("dim,k", [(2, 16), (3, 24)])
@pytest.mark.parametrize("scale", [2e-2, 3e-3])
def test_restarted_rows(ctx, dim, k, scale):
    pts = _clusters(dim, scale, 12)
    pts = pts[np.all((pts > 0.0) & (pts < 0.999999), axis=1)]  # none moved onto a plane
    g = api.Mesh(ctx, pts, boundary="reflective", k=k, restart=True, k_max=256)
    ref = O.Mesh(pts, "reflective", k=k, restart=True, k_max=256)
    out = g.copy_out()
    for key in ("status", "kcert", "face_counts", "face_ptr", "neighbor_cell"):
        assert np.array_equal(out[key], ref.get(key)), key
    assert g.n_restarted > 0
