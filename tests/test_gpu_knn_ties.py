"""Neighbour rows whose distances tie, or lie closer together than the row
search's quantized keys tell apart: lattices (every shell ties, within the row,
across 64 ranks and across its end, where members may have left the kept keys),
lattices displaced below a quantum, and coincident points, more of them than
the 64 candidates a tie with the last rank may have.  Rows must equal the
oracle's order by (distance, input index), by the problem interface and by the
allocation-free one (which has no sub-grids), and restarts must continue them.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from proteusgpu_amd import _native, api
from proteusgpu_amd.generators import jittered_lattice, uniform_points

pytestmark = pytest.mark.gpu

KS = (8, 12, 16, 20, 32, 48, 63, 64, 65, 100, 127, 128, 129, 192, 200, 256)


def _rows_noalloc(ctx, pts, k):
    n, dim = pts.shape
    d = torch.from_numpy(np.ascontiguousarray(pts)).cuda()
    s, p = torch.empty_like(d), torch.empty(n, dtype=torch.int32, device="cuda")
    r = torch.empty((n, k), dtype=torch.int32, device="cuda")
    _native.check(_native.lib().pg_knn_solve_noalloc(ctx.h, dim, d.data_ptr(), n, k, s.data_ptr(), p.data_ptr(),
                                                     r.data_ptr(), None))
    ctx.sync()
    return r.cpu().numpy().view(np.uint32)


def _check(ctx, pts, ks=KS):
    kp = api.KnnProblem(ctx, pts)
    for k in ks:
        ref = O.knn(pts, k)[3]
        kp.solve(k)
        assert np.array_equal(kp.get_knearest(), ref), k
        assert np.array_equal(_rows_noalloc(ctx, pts, k), ref), k
    kp.free()


@pytest.mark.parametrize("dim,m", [(2, 48), (2, 61), (3, 24), (3, 25)])
@pytest.mark.parametrize("amp", [0.0, 1e-12, 1e-8])
def test_lattices(ctx, dim, m, amp):
    _check(ctx, jittered_lattice(m, dim, 1, amp=amp))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("copies", [3, 30, 70, 100])
def test_coincident_points(ctx, dim, copies):
    p = uniform_points(2500 if dim == 2 else 13000, dim, 75)
    _check(ctx, np.concatenate([p] + [p[:5]] * copies), (8, 16, 32, 64, 100, 200))


def test_lattice_of_pairs(ctx):
    """Every lattice point twice: runs of twice a shell's length."""
    p = jittered_lattice(19, 3, 1, amp=0.0)
    _check(ctx, np.concatenate([p, p]), (16, 33, 64, 128, 256))


@pytest.mark.parametrize("dim,amp,k", [(2, 1e-6, 8), (3, 1e-6, 16), (3, 1e-5, 14)])
def test_restarted_rows(ctx, dim, amp, k):
    pts = jittered_lattice(40 if dim == 2 else 24, dim, 3, amp=amp)
    g = api.Mesh(ctx, pts, boundary="reflective", k=k, restart=True)
    ref = O.Mesh(pts, "reflective", k=k, restart=True)
    out = g.copy_out()
    for key in ("status", "kcert", "face_counts", "neighbor_cell"):
        assert np.array_equal(out[key], ref.get(key)), key
    assert g.n_restarted > 0
