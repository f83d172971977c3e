"""The surrogate's GEMM kernels at the edges of their tiles: the three tilings
(16 x 16 blocks straight from memory, 64 x 64 and 128 x 128 through LDS) give the
same bits for the same rows, and gradients of odd shapes match the oracle network
within the bars of test_gpu_mlp.py (outputs 5e-3, gradients 2e-2 relative
Frobenius: bf16 activations that round to the neighbouring value)."""
import numpy as np
import pytest

import leo2d_amd as L
from oracle import mlp_oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("d_in,hidden,out", [(72, 256, 1024), (64, 200, 500), (33, 72, 130)])
def test_same_bits_in_every_tile(d_in, hidden, out):
    rng = np.random.default_rng(d_in)
    x = rng.standard_normal((4096, d_in)).astype(np.float32)
    net = L.Mlp(0, d_in, hidden, 2, out, seed=1)
    y = net.forward(x)
    ref, _ = O.forward(net.params(), net.dims, x[:64])
    assert _rel(y[:64], ref) <= 5e-3
    for rows in (1, 31, 33, 64, 129, 700, 2048):
        assert np.array_equal(net.forward(x[:rows]), y[:rows]), rows
    net.close()


@pytest.mark.parametrize("d_in,hidden,layers,out,n", [(1, 8, 1, 1, 1), (7, 13, 2, 5, 9), (72, 40, 1, 17, 33),
                                                      (64, 96, 3, 100, 257), (72, 256, 1, 64, 8192)])
def test_gradients_of_odd_shapes(d_in, hidden, layers, out, n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, d_in)).astype(np.float32)
    t = (0.3 * rng.standard_normal((n, out))).astype(np.float32)
    net = L.Mlp(0, d_in, hidden, layers, out, seed=2)
    loss, g = net.gradients(x, t)
    oloss, og = O.loss_and_grad(net.params(), net.dims, x, t)
    assert abs(loss - oloss) <= 1e-3 * oloss
    off = 0
    for a, b in zip(net.dims, net.dims[1:]):
        for size in (a * b, b):
            assert _rel(g[off:off + size], og[off:off + size]) <= 2e-2
            off += size
    # a smaller batch after a larger one reads nothing the larger one left
    k = max(1, n // 3)
    loss2, g2 = net.gradients(x[:k], t[:k])
    fresh = L.Mlp(0, d_in, hidden, layers, out, seed=2)
    loss3, g3 = fresh.gradients(x[:k], t[:k])
    assert loss2 == loss3 and np.array_equal(g2, g3)
    net.close()
    fresh.close()
