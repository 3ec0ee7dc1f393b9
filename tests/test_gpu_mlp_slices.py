"""Gradients of the warm-start perceptron around the edges of the batch slices
that the weight-gradient products split over workgroups: slices of 128 rows up
to a batch of 8192, longer ones (at most 64) beyond, partial last slices, and a
batch below one 32-row step of a tile.  Oracle and bounds as in test_gpu_mlp.py:
8-bit mantissas through four layers each way give a few percent per layer."""
import numpy as np
import pytest

from oracle import mlp as omlp
import solfec
from solfec import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [31, 128, 129, 8192, 8193, 20011])
def test_gradient_at_slice_edges(n):
    print(f"[mlp slices] n={n}", flush=True)
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 18)).astype(np.float32)
    Y = np.stack([np.sin(X[:, 0]), X[:, 1] * X[:, 2], np.tanh(X[:, 3])], 1).astype(np.float32)
    p = learned.init_params(1)
    W = learned.unpack(p)
    for k in (1, 3, 5, 7):
        W[k][:] = rng.normal(scale=0.1, size=W[k].shape)
    norm = learned.norm_from_data(X, Y)
    dev = solfec.Device(0)
    dev.mlp_set(p, norm)
    loss, g = dev.mlp_grad(X, Y)
    dev.close()
    rloss, rg = omlp.loss_and_grad(p.astype(np.float64), norm.astype(np.float64), X.astype(np.float64),
                                   Y.astype(np.float64))
    assert abs(loss - rloss) <= 3e-2 * rloss
    offs = np.cumsum([0] + [int(np.prod(s)) for s in omlp.SHAPES])
    for k in range(8):
        a, b = g[offs[k]:offs[k + 1]].astype(np.float64), rg[offs[k]:offs[k + 1]]
        assert np.linalg.norm(a - b) / np.linalg.norm(b) < 0.1, k
        assert a @ b / (np.linalg.norm(a) * np.linalg.norm(b)) > 0.99, k
