"""Memory that freed objects left behind is bounded in blocks as well, and given
back on request, while the context and its other objects go on."""
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import numpy as np
import torch
from proteusgpu_amd import api
from proteusgpu_amd.generators import uniform_points
ctx = api.Context(0)
used = lambda: torch.cuda.mem_get_info(0)[1] - torch.cuda.mem_get_info(0)[0]
p = uniform_points(300000, 3, 1)
small = api.Mesh(ctx, p[:30000], boundary="reflective", k=32)
before = small.copy_out()
ctx.trim()
u0 = used()
api.Mesh(ctx, p, boundary="reflective", k=32).free()
u1 = used()
ctx.trim()
u2 = used()
api.Mesh(ctx, p, boundary="reflective", k=32).free()
after = small.copy_out()
assert all(np.array_equal(before[k], after[k]) for k in before)
print(u0, u1, u2)
"""


def test_trim():
    r = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    u0, u1, u2 = (int(x) for x in r.stdout.split())
    mib = 1 << 20
    assert u1 - u0 > 500 * mib and u2 - u0 < 64 * mib


MANY = """
import numpy as np
import torch
from proteusgpu_amd import api
ctx = api.Context(0)
used = lambda: torch.cuda.mem_get_info(0)[1] - torch.cuda.mem_get_info(0)[0]
x = np.zeros((16384, 16), np.float32)
models = [api.KModel(ctx) for _ in range(5000)]
u0 = used()
for km in models:
    km.predict(x)
u1 = used()
for km in models:
    km.free()
u2 = used()
print(u0, u1, u2)
"""


def test_many_small_blocks():
    """5000 models of 1 MiB and four small blocks each: most blocks go."""
    r = subprocess.run([sys.executable, "-c", MANY], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    u0, u1, u2 = (int(x) for x in r.stdout.split())
    gib = 1 << 30
    assert u1 - u0 > 4 * gib and u2 - u0 < 2 * gib
