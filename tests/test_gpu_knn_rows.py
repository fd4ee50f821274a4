"""The neighbour search by rows of grid cells.

Neighbour lists must equal the oracle's: row lengths around the kept 64 keys
per slot, equal distances (lattices, whose shells tie inside and across the
row's end), distances on the edge of a ring of cells (a lattice commensurate
with the grid), coincident points, a density that varies across the query's
block (the ball guess is off), and points outside the unit box, which the
grid keeps in its border cells.
"""
import numpy as np
import pytest

from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import jittered_lattice, uniform_points

pytestmark = pytest.mark.gpu


def _check(ctx, pts, ks):
    kp = api.KnnProblem(ctx, pts)
    for k in ks:
        kp.solve(k)
        assert np.array_equal(kp.get_knearest(), O.knn(pts, k)[3]), k
    kp.free()


@pytest.mark.parametrize("dim", [2, 3])
def test_row_lengths(ctx, dim):
    _check(ctx, uniform_points(5000 if dim == 2 else 16000, dim, 71), (1, 16, 20, 31, 63, 64, 65, 127, 128, 129, 200, 256))


@pytest.mark.parametrize("dim,m", [(2, 50), (3, 24), (3, 27)])
def test_ties(ctx, dim, m):
    _check(ctx, jittered_lattice(m, dim, 1, amp=0.0), (16, 20, 32, 33, 64, 100))


@pytest.mark.parametrize("dim", [2, 3])
def test_coincident_points(ctx, dim):
    p = uniform_points(4000 if dim == 2 else 14000, dim, 72)
    _check(ctx, np.concatenate([p, p[:500], p[:300], p[:40]]), (20, 32, 64))


@pytest.mark.parametrize("dim", [2, 3])
def test_uneven_density(ctx, dim):
    p = uniform_points(6000 if dim == 2 else 20000, dim, 73)
    p[:, 0] = p[:, 0] ** 2.5
    _check(ctx, p, (20, 32, 64, 96))


@pytest.mark.parametrize("dim", [2, 3])
def test_points_outside_the_box(ctx, dim):
    p = uniform_points(4000 if dim == 2 else 14000, dim, 74)
    _check(ctx, 1.1 * p - 0.05, (20, 32, 64))
