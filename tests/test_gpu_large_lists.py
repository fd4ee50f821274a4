"""Neighbour lists of more queries than one launch of a wave per query can
hold (2^26), by the wave kernel and by the heap, against torch in 64 bits for
queries on both sides of the launches' ends."""
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
