"""What a build reports of sets whose cells mostly fail (exact lattices: a
degenerate predicate at nearly every seed), over block edges of the collect:
failures counted as the oracle counts them."""
import numpy as np
import pytest

from oracle import oracle as O
from proteusgpu_amd import api
from proteusgpu_amd.generators import jittered_lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,m,k", [(2, 45, 16), (2, 46, 16), (3, 24, 32), (3, 26, 24)])
@pytest.mark.parametrize("restart", [True, False])
def test_lattices(ctx, dim, m, k, restart):
    pts = jittered_lattice(m, dim, 1, amp=0.0)
    g = api.Mesh(ctx, pts, boundary="reflective", k=k, restart=restart)
    ref = O.Mesh(pts, "reflective", k=k, restart=restart)
    status = g.copy_out()["status"]
    assert np.array_equal(status, ref.get("status"))
    assert g.n_failed == int((status != 4).sum()) == ref.n_failed
