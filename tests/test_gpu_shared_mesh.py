"""One finalised mesh, several host threads, each with its own context and its
own state: the mesh is only read, so every state ends as in a serial run.  A
state is only read by its CFL step, which two contexts may ask for at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from proteusgpu_amd import api
from proteusgpu_amd._native import check, lib
from proteusgpu_amd.generators import sod_state, uniform_points

pytestmark = pytest.mark.gpu


def _setup(ctx, dim, n, boundary):
    pts = uniform_points(n, dim, 31)
    return api.Mesh(ctx, pts, boundary=boundary, buff=0.1, k=16 if dim == 2 else 32), sod_state(pts, 1.4)


def _threads(work, count):
    """work(i, context) for i < count at once; their results."""
    got = {}

    def run(i):
        c = api.Context(0)
        got[i] = work(i, c)
        c.close()

    th = [threading.Thread(target=run, args=(i,)) for i in range(count)]
    for t in th:
        t.start()
    for t in th:
        t.join(60)
        assert not t.is_alive()
    return [got[i] for i in range(count)]


def _advance(ctx, mesh, state, steps):
    st = api.HydroState(ctx, mesh, *state)
    dt = []
    for _ in range(steps):
        dt.append(st.dt_cfl(1.4, 0.3))
        st.step(1.4, dt[-1], "physical")
    out = st.copy_out()
    st.free()
    return [np.array(dt), *out]


SETUPS = pytest.mark.parametrize("dim,n,boundary", [(2, 40000, "periodic"), (3, 60000, "reflective")])


@SETUPS
def test_states_on_one_mesh(ctx, dim, n, boundary):
    mesh, (rho, vel, E) = _setup(ctx, dim, n, boundary)
    states = [(rho * f, vel + 0.1 * f, E * f) for f in (1.0, 1.3, 0.7, 2.1)]
    serial = [_advance(ctx, mesh, s, 20) for s in states]
    got = _threads(lambda i, c: _advance(c, mesh, states[i], 20), len(states))
    for i, ref in enumerate(serial):
        for a, b in zip(got[i], ref):
            assert np.array_equal(a, b), i
    mesh.free()


@SETUPS
def test_one_state_two_contexts(ctx, dim, n, boundary):
    mesh, state = _setup(ctx, dim, n, boundary)
    st = api.HydroState(ctx, mesh, *state)
    want = [st.dt_cfl(1.4, cfl) for cfl in (0.3, 0.4)]

    def ask(i, c):
        dt, seen = C.c_double(), set()
        for _ in range(200):
            check(lib().pg_dt_cfl(c.h, mesh.h, st.h, 1.4, (0.3, 0.4)[i], C.byref(dt)))
            seen.add(dt.value)
        return seen

    assert _threads(ask, 2) == [{w} for w in want]
    st.free()
    mesh.free()
