"""The gradient pass of the network (64 rows per block, 16 per wave): batches that fill one wave, one
block and more against the oracle, and batches beyond one round of blocks against the mean of
their halves."""
import numpy as np
import pytest

import pyoracle as po
from helpers import rel_linf
from lbmpond_amd import Pond
from test_mlp_oracle import make

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": (0, 8640), "b1": (8640, 8704), "W2": (8704, 12800), "b2": (12800, 12864), "W3": (12864, 13120),
          "b3": (13120, 13124)}


def grad(p, X, T):
    with Pond("D3Q27", (4, 4, 4), "weno5c", "split", use_mlp=True) as pond:
        pond.mlp_set_params(p, np.ones(9, np.float32))
        return pond.mlp_grad(X, T)


@pytest.mark.parametrize("B", [16, 32, 64, 80, 336])
def test_small_batches_match_oracle(gpu, B):
    p, X, T = make(20 + B, B=B)
    g, loss = grad(p, X, T)
    gr, lr = po.mlp_grad(p, X, T, bf16=True)
    # the bounds the gradients are held to at 256 rows (test_mlp_gpu.py): a BF16 rounding that falls the
    # other way moves one term by 2^-8
    assert abs(loss - lr) <= 1e-4 * lr
    for name, (a, b) in BLOCKS.items():
        assert rel_linf(g[a:b], gr[a:b]) < 1e-2, name


@pytest.mark.parametrize("B", [2048, 32768, 65536])
def test_large_batch_is_the_mean_of_its_halves(gpu, B):
    """Halving B scales every output gradient by two, which no rounding sees: only the order of the
    FP32 sums differs, an error of 2^-24 sqrt(B/2) of the sum for terms of random sign."""
    p, X, T = make(7, B=B)
    g, loss = grad(p, X, T)
    h = [grad(p, X[k * (B // 2):(k + 1) * (B // 2)], T[k * (B // 2):(k + 1) * (B // 2)]) for k in (0, 1)]
    mean = 0.5 * (h[0][0].astype(np.float64) + h[1][0])
    assert abs(loss - 0.5 * (h[0][1] + h[1][1])) <= 2e-5 * loss
    for name, (a, b) in BLOCKS.items():
        assert rel_linf(g[a:b], mean[a:b]) <= 2e-5, name
