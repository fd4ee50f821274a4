"""Batches made in device memory that freed buffers left behind.

The blocks are filled beforehand, in the size class of a batch's per-seed
32-bit tables, with a word that would pass there for a saved cell of 8 row
entries.  The first pass of a rebuild (fixed and learned k) must not look at
what its tables held: every box equals, to the bit, the same box run alone.
Periodic boxes move, so that later rebuilds also hold more seeds than earlier
ones wrote entries for.
"""
import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd.generators import batch_points, kelvin_helmholtz_state, sod_state

pytestmark = pytest.mark.gpu


def _leave(ctx, nbytes, word, copies=40):
    """Freed blocks of nbytes (rounded up to 64) full of word."""
    x = np.full((-(-nbytes // 64), 16), word, np.uint32).view(np.float32)
    models = [api.KModel(ctx) for _ in range(copies)]
    for km in models:
        km.predict(x)
    for km in models:
        km.free()


@pytest.mark.parametrize("dim,boundary,sizes,k", [(3, "reflective", (13000, 15001), 32), (3, "periodic", (14000,), 24),
                                                  (2, "periodic", (1500, 4001), 16)])
@pytest.mark.parametrize("learned", [False, True])
def test_first_pass_ignores_what_its_memory_held(ctx, dim, boundary, sizes, k, learned):
    sizes, buff = np.array(sizes), 0.1 if dim == 2 else 0.12
    pts = batch_points(sizes, dim, 500 + dim)
    st = kelvin_helmholtz_state(pts) if boundary == "periodic" else sod_state(pts, 1.4)
    kw = dict(boundary=boundary, buff=buff, k=k, gamma=1.4, cfl=0.3, flux="physical", move_mesh=True)
    ref, off = [], 0
    for n in sizes:
        s = api.Simulation(ctx, pts[off:off + n], *(a[off:off + n] for a in st), **kw)
        for _ in range(3):
            s.step()
        ref.append(s.get())
        s.free()
        off += n
    km = api.KModel(ctx, seed=2)
    # lanes and slots per lane of the default clip shape, and a row length
    tag = (16 << 24 | 4 << 16 if dim == 3 else 8 << 24 | 2 << 16) | 8
    like = api.Batch(ctx, sizes, pts, *st, **kw)  # lives on, so that its blocks are not the ones taken
    cap = like.info()["seed_capacity"]
    print(f"dim={dim} {boundary} sizes={sizes.tolist()} k={k} learned={learned} capacity={cap}", flush=True)
    _leave(ctx, 4 * cap, tag)
    B = api.Batch(ctx, sizes, pts, *st, **kw)
    if learned:
        B.set_kmodel(km)
    for _ in range(3):
        B.step()
    for a, b in zip(B.get(), zip(*ref)):
        assert np.array_equal(a, np.concatenate(b))
    B.free()
    like.free()


def test_no_step_no_dt(ctx):
    """The CFL steps of a batch that has not stepped are 0, whatever its memory held."""
    sizes = np.array([1500, 1700, 1600])
    pts = batch_points(sizes, 2, 520)
    _leave(ctx, 64, 0x3ff01234)
    B = api.Batch(ctx, sizes, pts, *kelvin_helmholtz_state(pts), boundary="periodic", buff=0.1, k=16)
    assert np.array_equal(B.dt(), np.zeros(3))
    B.step()
    assert np.all(B.dt() > 0)
    B.free()
