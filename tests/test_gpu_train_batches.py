"""Gradients of batches around the groups of 16 and blocks of 64 seeds.

The reduction over blocks is in block order whatever the split, so a batch's
gradient is checked against the oracle's FP64 pass with the tolerance of
test_gpu_learned_k.py's full batch (bfloat16 rounding flips: 2e-2 of each
block's norm), and repeated calls give equal bits.
"""
import numpy as np
import pytest

from oracle import learned_k as L
from proteusgpu_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 15, 16, 17, 63, 64, 65, 2047, 2049, 4200])
def test_gradient_of_a_batch(ctx, B):
    rng = np.random.default_rng(100 + B)
    X = np.abs(rng.standard_normal((B, 16))).astype(np.float32)
    y = rng.integers(0, 6, B).astype(np.int32)
    P = (0.3 * rng.standard_normal(L.NPARAM)).astype(np.float32)
    km = api.KModel(ctx)
    km.params = P
    loss, g = km.grad(X, y)
    loss_o, go = L.loss_grad(P, X, y, bf16_ops=True)
    assert abs(loss - loss_o) <= 1e-3 * abs(loss_o)
    gd, od = L.unpack(g), L.unpack(go)
    for name, _ in L.SHAPES:
        assert np.linalg.norm(gd[name] - od[name]) <= 2e-2 * np.linalg.norm(od[name]), name
    loss2, g2 = km.grad(X, y)
    assert loss2 == loss and np.array_equal(g2, g)
    km.free()
