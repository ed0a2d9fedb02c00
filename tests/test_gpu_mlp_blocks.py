"""The training kernel's block partials and their reduction at block-count edges.

Tiles of 32 samples go to up to four blocks a CU, and 16 wavefronts add the blocks' gradients: fewer blocks than
wavefronts, one past a multiple of 16, and more tiles than blocks.  Bounds as for the gradient's other sizes
(bfloat16 roundings that an ulp of tanh flips).
"""
import numpy as np
import pytest

from oracle import mlp as M
from picopic_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15 * 32, 17 * 32 - 5, 40001])
def test_gradient_over_blocks(n):
    rng = np.random.default_rng(n)
    c = capi.Context((8e-4, 8e-4), (8, 8), (1, 1), 1e-12, [(-1, 1, False, 64), (1, 1836, False, 64)])
    p = M.init(7)
    c.mlp_set_params(p)
    X = rng.normal(size=(n, 6)).astype(np.float32)
    T = np.tanh(X[:, :4] * 0.7).astype(np.float32)
    print("blocks", n, flush=True)
    g, loss = c.mlp_grad(X, T)
    g_ref, loss_ref = M.grad(p, X, T, True)
    assert abs(loss - loss_ref) <= 1e-3 * loss_ref
    assert np.abs(g - g_ref).max() <= 2e-2 * np.abs(g_ref).max()
    g2, loss2 = c.mlp_grad(X, T)
    assert np.array_equal(g, g2) and loss == loss2
