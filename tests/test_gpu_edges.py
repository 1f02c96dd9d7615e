"""Kernels at the edges of their tiles: remainders, the smallest sizes, and sizes past one tile
or one launch's blocks, each against the FP64 oracle or plain numpy."""
import numpy as np
import pytest

from masterthesislucas_amd import tsne
from masterthesislucas_amd.learned import N_OUT, FarFieldMLP, flatten, unflatten
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("terms", [3, 7])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 100, 256 * 32 + 5])
def test_training_gradient_edges(gpu, n, terms):
    """Samples in tiles of 32, at most 256 tiles at a time: one sample, around one tile, a ragged
    last tile, and a block that takes two tiles. Gradient blocks to 1e-4 of their norm, as FP32
    activations with FP32 sums (n products of about 1e-7 relative error each) allow."""
    rng = np.random.default_rng(100 + n)
    p = {"W1": rng.normal(0, 0.4, (10, 64)), "b1": rng.normal(0, 0.1, 64),
         "W2": rng.normal(0, 0.15, (64, 64)), "b2": rng.normal(0, 0.1, 64),
         "W3": rng.normal(0, 0.15, (64, N_OUT)), "b3": rng.normal(0, 0.1, N_OUT)}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    X = rng.normal(0, 1, (n, 13)).astype(np.float32)
    a = rng.uniform(0, 2 * np.pi, n)
    X[:, 10], X[:, 11] = np.cos(a), np.sin(a)
    X[:, 12] = rng.uniform(0.05, 1.0, n)
    T = rng.normal(0, 0.5, (n, 2)).astype(np.float32)
    net = FarFieldMLP(max_samples=max(n, 16))
    net.terms = terms
    net.set_params(flatten(p))
    loss, g = net.loss_grad(X, T)
    ref_loss, ref_g = O.learned_loss_grad(X.astype(np.float64), T.astype(np.float64),
                                          {k: v.astype(np.float64) for k, v in p.items()},
                                          terms=terms)
    assert abs(loss - ref_loss) < 1e-5 * ref_loss
    gg = unflatten(g)
    for k in ref_g:
        num = np.linalg.norm(gg[k].astype(np.float64) - ref_g[k])
        assert num < 1e-4 * np.linalg.norm(ref_g[k]) + 1e-9, k
    # the data-set loss that training reports (forward only) is the same loss
    net.set_dataset(X, T)
    assert abs(net.train(0) - ref_loss) < 1e-5 * ref_loss
    net.close()
