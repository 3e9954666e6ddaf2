"""Kernels and dispatch rules at the sizes where they can go wrong: tile edges,
remainders, the smallest and the largest of a rule's range. Each against the
restatements under oracle/ or plain numpy in 64 bits."""
import numpy as np
import pytest

from oracle import mlp_ref


@pytest.mark.gpu
@pytest.mark.parametrize("in_features,hidden,n", [(1, 1, 1), (3, 17, 5), (14, 64, 32), (14, 64, 33), (16, 16, 31),
                                                  (15, 15, 64), (31, 48, 2051), (14, 200, 700), (5, 700, 40)])
def test_mlp_contractions_at_tile_edges(in_features, hidden, n):
    """Result tiles of 16, four samples per MFMA, slices of the samples (one,
    several, a short last one; one when the tiles alone fill the chip) against
    float64, at the bar of the network's other tests."""
    from hisvsim_amd.costmodel import MLP
    rng = np.random.default_rng(n)
    m = MLP(in_features, hidden, seed=3)
    p = m.params().astype(np.float64)
    X = rng.normal(size=(n, in_features)).astype(np.float32)
    y = rng.normal(size=n).astype(np.float32)
    want, _ = mlp_ref.forward(p, X, in_features, hidden)
    assert np.abs(m.predict(X) - want).max() <= 1e-4 * max(1.0, np.abs(want).max())
    loss, g = m.gradient(X, y)
    rl, rg = mlp_ref.loss_and_grad(p, X, y, in_features, hidden)
    assert abs(loss - rl) <= 1e-4 * rl
    assert np.abs(g - rg).max() <= 1e-4 * max(1.0, np.abs(rg).max())
    m.close()
