"""Learned k without restarts, or with restarts that end below the buckets: a
seed is clipped by the row of its bucket and no longer one, whichever kernel
clips it.

2D rings of points give cells that outgrow the fast kernel's 16 vertices; a
classifier that puts every seed into one bucket must leave the statuses and
cells of the fixed k of that bucket (the oracle's)."""
import numpy as np
import pytest

from oracle import learned_k as L
from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import sod_state, uniform_points

pytestmark = pytest.mark.gpu

BUCKETS = (16, 24, 32, 48, 64, 96)


def _rings(jitter=0.0, gap=0.09):
    """jitter: of the rings' radii (points on one circle are degenerate, which
    a run refuses); gap: radius around a ring without other points."""
    rng, rings = np.random.default_rng(92), []
    for faces, cx, cy in ((17, 0.31, 0.42), (22, 0.68, 0.27), (40, 0.5, 0.8)):
        a = 2 * np.pi * (np.arange(faces) + 0.25) / faces
        r = 0.04 * (1 + jitter * rng.random(faces))
        rings.append(np.concatenate([[[cx, cy]], np.stack([cx + r * np.cos(a), cy + r * np.sin(a)], 1)]))
    base = uniform_points(3000, 2, 91)
    keep = np.all([np.hypot(*(base - r[0]).T) > gap for r in rings], axis=0)
    return np.concatenate([base[keep]] + rings)


def _model(ctx, c):
    """Every seed in bucket c."""
    P = np.zeros(L.NPARAM, dtype=np.float32)
    P[5632 + c] = 30.0
    km = api.KModel(ctx)
    km.params = P
    km.set_cost(0.0)
    return km


@pytest.mark.parametrize("c", range(6))
def test_rows_of_the_bucket(ctx, c):
    pts, km = _rings(), _model(ctx, c)
    g = api.Mesh(ctx, pts, boundary="reflective", k=16, restart=False, kmodel=km)
    k = BUCKETS[int(np.argmax(g.n_class))]
    assert g.n_class.max() == g.n_seeds
    ref = O.Mesh(pts, "reflective", k=k, restart=False)
    out = g.copy_out()
    for key in ("status", "kcert", "face_counts", "neighbor_cell"):
        assert np.array_equal(out[key], ref.get(key)), (k, key)
    km.free()
    g.free()


@pytest.mark.parametrize("c", [1, 2])
def test_completion_after_the_bucket(ctx, c):
    """Restarts that may not go beyond 16 neighbours: what a bucket's row leaves
    uncertified is completed from the vertices (kcert k_max + 1)."""
    pts, km = _rings(1e-3), _model(ctx, c)
    g = api.Mesh(ctx, pts, boundary="reflective", k=16, k_max=16, restart=True, kmodel=km)
    k = BUCKETS[int(np.argmax(g.n_class))]
    ref = O.Mesh(pts, "reflective", k=k, k_max=k, restart=True)
    out, kcert = g.copy_out(), ref.get("kcert").copy()
    assert np.any(kcert == k + 1)
    kcert[kcert == k + 1] = 17
    assert np.array_equal(out["kcert"], kcert)
    for key in ("status", "face_counts", "neighbor_cell"):
        assert np.array_equal(out[key], ref.get(key)), key
    km.free()
    g.free()


def test_batch_equals_single_run(ctx):
    pts, km = _rings(1e-3, 0.06), _model(ctx, 5)
    st = sod_state(pts, 1.4)
    kw = dict(boundary="reflective", k=200, gamma=1.4, cfl=0.3, move_mesh="static", restart=False)
    assert api.Mesh(ctx, pts, boundary="reflective", k=200).copy_out()["face_counts"].max() > 20
    s = api.Simulation(ctx, pts, *st, **kw)
    B = api.Batch(ctx, [len(pts)], pts, *st, **kw)
    for o in (s, B):
        o.set_kmodel(km)
        for _ in range(3):
            o.step()
    for a, b in zip(s.get(), B.get()):
        assert np.array_equal(a, b)
    s.free()
    B.free()
