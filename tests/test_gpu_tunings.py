"""Tunings of a batch choose kernels, never results.

The KNN's line between heap and wave rows at, below and above the row length
(short 2D rows, 3D rows, and rows long enough for the heap's half-filled
blocks), for all the batch's passes, the 3D clip shapes, and caps on the
resident blocks below and above the kernels' occupancy, which make the first
passes persistent blocks or a block per query or group (with rows so short
that nearly every cell goes on from its saved state, and without restarts):
states equal to the bit, and equal to the boxes run alone.
"""
import itertools

import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd.generators import batch_points, kelvin_helmholtz_state, sod_state

pytestmark = pytest.mark.gpu


def _case(dim, k):
    sizes = np.array([3000, 4500] if dim == 2 else [13500, 15000])
    pts = batch_points(sizes, dim, 600 + k)
    st = kelvin_helmholtz_state(pts) if dim == 2 else sod_state(pts, 1.4)
    kw = dict(boundary="periodic" if dim == 2 else "reflective", buff=0.1, k=k, gamma=1.4, cfl=0.3, move_mesh=True)
    return sizes, pts, st, kw


def _run(ctx, sizes, pts, st, kw, **tuning):
    B = api.Batch(ctx, sizes, pts, *st, **kw)
    B.set_tuning(**tuning)
    B.step()
    B.step()
    out = B.get()
    B.free()
    return out


def _alone(ctx, sizes, pts, st, kw):
    outs, off = [], 0
    for n in sizes:
        s = api.Simulation(ctx, pts[off:off + n], *(a[off:off + n] for a in st), **kw)
        s.step()
        s.step()
        outs.append(s.get())
        s.free()
        off += n
    return [np.concatenate(a) for a in zip(*outs)]


@pytest.mark.parametrize("dim,k", [(2, 8), (2, 16), (3, 24), (3, 70), (2, 210), (3, 256)])
def test_knn_line(ctx, dim, k):
    case = _case(dim, k)
    ref = _alone(ctx, *case)
    for wmk, graph in itertools.product((1, 20, k, k + 1, 300), (True, False)):
        for a, b in zip(_run(ctx, *case, knn_wave_min_k=wmk, use_graph=graph), ref):
            assert np.array_equal(a, b), (wmk, graph)


def test_clip_shapes_3d(ctx):
    case = _case(3, 32)
    ref = _alone(ctx, *case)
    for lanes, slots in itertools.product((8, 16), (48, 64)):
        for a, b in zip(_run(ctx, *case, clip_lanes=lanes, clip_slots=slots), ref):
            assert np.array_equal(a, b), (lanes, slots)


@pytest.mark.parametrize("dim,k,restart", [(2, 10, True), (2, 16, True), (2, 64, False), (3, 24, True)])
def test_caps_on_resident_blocks(ctx, dim, k, restart):
    sizes, pts, st, kw = _case(dim, k)
    kw["restart"] = restart
    ref = _alone(ctx, sizes, pts, st, kw)
    for cap, graph in itertools.product((1, 2, 8, 64), (True, False)):
        for a, b in zip(_run(ctx, sizes, pts, st, kw, blocks_per_cu=cap, use_graph=graph), ref):
            assert np.array_equal(a, b), (cap, graph)


def test_autotune_leaves_what_it_cannot_time(ctx):
    """2D clips have one shape, so the setting stays as it was; every candidate's
    step still gives the same states."""
    sizes, pts, st, kw = _case(2, 16)
    ref = _alone(ctx, sizes, pts, st, kw)
    for lanes, slots in ((8, 48), (16, 48)):
        B = api.Batch(ctx, sizes, pts, *st, **kw)
        B.set_tuning(clip_lanes=lanes, clip_slots=slots)
        best, _ = B.autotune(reps=1)
        assert (best["clip_lanes"], best["clip_slots"]) == (lanes, slots)
        assert B.tuning == best
        B.step()
        B.step()
        for a, b in zip(B.get(), ref):
            assert np.array_equal(a, b)
        B.free()
