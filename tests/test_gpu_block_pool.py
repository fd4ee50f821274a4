"""Device blocks that freed buffers leave for later ones: contexts, threads and
streams that share them get the results they get alone, and what is held is
bounded and given back."""
import subprocess
import sys
import threading

import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd.generators import sod_state, uniform_points

pytestmark = pytest.mark.gpu

KEYS = ("status", "face_counts", "neighbor_cell", "face_area", "volumes")


def _mesh(ctx, dim, n, seed):
    m = api.Mesh(ctx, uniform_points(n, dim, seed), boundary="periodic", buff=0.1, k=16 if dim == 2 else 24)
    out = m.copy_out()
    m.free()
    return [out[k] for k in KEYS]


def _sim(ctx, n, seed):
    p = uniform_points(n, 2, seed)
    s = api.Simulation(ctx, p, *sod_state(p, 1.4), boundary="reflective", k=16, gamma=1.4, cfl=0.3, move_mesh=True)
    for _ in range(3):
        s.step()
    out = s.get()
    s.free()
    return out


def test_threads_with_their_own_streams(ctx):
    jobs = [lambda c, i=i: _mesh(c, 2 + i % 2, 5000 + 700 * i + (11000 if i % 2 else 0), i) if i % 3
            else _sim(c, 4000 + 300 * i, i) for i in range(8)]
    alone = [j(ctx) for j in jobs]
    got = {}

    def work(t):
        c = api.Context(0)
        got[t] = [[jobs[(t + r) % 8](c) for r in range(8)] for _ in range(2)]
        c.close()

    th = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join(60)
        assert not t.is_alive()
    for t in range(4):
        for rep in got[t]:
            for r, out in enumerate(rep):
                for a, b in zip(out, alone[(t + r) % 8]):
                    assert np.array_equal(a, b), (t, r)


CHILD = """
import torch
from proteusgpu_amd import api
from proteusgpu_amd.generators import uniform_points
ctx = api.Context(0)
used = lambda: torch.cuda.mem_get_info(0)[1] - torch.cuda.mem_get_info(0)[0]
p = uniform_points(700000, 3, 1)
u0 = used()
ms = [api.Mesh(ctx, p, boundary="reflective", k=32) for _ in range(3)]
u1 = used()
for m in ms:
    m.free()
u2 = used()
ctx.close()
u3 = used()
print(u0, u1, u2, u3)
"""


def test_held_blocks_are_bounded_and_given_back():
    r = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    u0, u1, u2, u3 = (int(x) for x in r.stdout.split())
    gib = 1 << 30
    assert u1 - u0 > 9 * gib          # more than the bound was in use
    assert u2 - u0 < 8 * gib + gib // 4
    assert u3 - u0 < gib // 4
