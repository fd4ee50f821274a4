"""Neighbour lists of more queries than one launch of a wave per query can
hold (2^26), by the wave kernel and by the heap, against torch in 64 bits for
queries on both sides of the launches' ends; and the cell order that such a
set is sorted into, whose kernel takes 2^24 cells per launch."""
import numpy as np
import pytest
import torch

from proteusgpu_amd import api

pytestmark = pytest.mark.gpu

N = (1 << 26) + 4099


@pytest.fixture(scope="module")
def problem(ctx):
    kp = api.KnnProblem(ctx, np.random.default_rng(3).random((N, 2)))
    print(f"n={N} N_grid={kp.N_grid}", flush=True)
    yield kp, torch.from_numpy(kp.get_points()).cuda()
    kp.free()


def test_points_of_a_cell_in_input_order(problem):
    kp, pts = problem
    m = kp.N_grid
    assert m * m > (1 << 24)
    perm = torch.from_numpy(kp.get_permutation().astype(np.int64)).cuda()
    c = torch.clamp(torch.floor(pts * m).long(), 0, m - 1)
    cell = c[:, 0] + m * c[:, 1]
    assert bool(torch.all((cell[1:] > cell[:-1]) | ((cell[1:] == cell[:-1]) & (perm[1:] > perm[:-1]))))


@pytest.mark.parametrize("k", [12, 16])
def test_rows(problem, k):
    kp, pts = problem
    kp.solve(k)
    rows = kp.get_knearest()
    print(f"k={k} solved", flush=True)
    rng = np.random.default_rng(k)
    q = np.r_[0, 1, 5000, (1 << 25) + np.arange(-2, 3), (1 << 26) + np.arange(-2, 3), N - 2, N - 1, rng.integers(0, N, 20)]
    for i in q:
        d = pts - pts[i]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]
        near = torch.topk(d2, k + 1, largest=False, sorted=True).indices.cpu().numpy()
        assert near[0] == i and np.array_equal(rows[i], near[1:]), i
