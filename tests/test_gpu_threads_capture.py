"""Threads with their own contexts: some capture and replay batched steps while
others build meshes, whose buffers come from blocks that freed ones left (a
wait for the device among them).  Everyone gets what a serial run gets."""
import threading

import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd.generators import batch_points, kelvin_helmholtz_state, uniform_points

pytestmark = pytest.mark.gpu


def _batch(ctx, i):
    sizes = np.array([1500 + 100 * i, 2600])
    pts = batch_points(sizes, 2, 700 + i)
    B = api.Batch(ctx, sizes, pts, *kelvin_helmholtz_state(pts), boundary="periodic", buff=0.1, k=16, gamma=1.4, cfl=0.3)
    for _ in range(3):
        B.step()
    out = B.get()
    B.free()
    return out


def _mesh(ctx, i):
    m = api.Mesh(ctx, uniform_points(4000 + 500 * i, 2, 800 + i), boundary="periodic", buff=0.1, k=16)
    out = m.copy_out()
    m.free()
    return [out[k] for k in ("status", "face_counts", "neighbor_cell", "face_area", "volumes")]


def test_captures_beside_builds(ctx):
    jobs = [lambda c, i=i: (_batch if i % 2 else _mesh)(c, i) for i in range(6)]
    alone = [j(ctx) for j in jobs]
    got = {}

    def work(t):
        c = api.Context(0)
        got[t] = [(t + r) % 6 for r in range(12)], [jobs[(t + r) % 6](c) for r in range(12)]
        c.close()

    th = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join(60)
        assert not t.is_alive()
    for t in range(4):
        for i, out in zip(*got[t]):
            for a, b in zip(out, alone[i]):
                assert np.array_equal(a, b), (t, i)
