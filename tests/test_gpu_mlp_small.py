"""Products of few tiles (gemm_small_kernel) and both sides of the rule that picks it (128 tiles of
64 x 64): edges of its 32 x 32 tiles and of its rounds of K (32 per step, 256
per load of all waves, 1024 per chunk) for the four operand layouts,
against a float64 product of the rounded operands (bound: FP32 accumulation,
K 2^-23 |A| |B|); and the network's gradient where its layers take different
forms, so that the row tiles of their column sums differ."""
import numpy as np
import pytest

from pdhcg_amd import warmstart
from tests import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(32, 32, 240), (48, 16, 272), (16, 48, 1040), (80, 112, 3008),
                                   (1024, 512, 48), (1024, 528, 48), (1040, 1008, 144)])
def test_products(ta, tb, M, N, K):
    rng = np.random.default_rng(M + 3 * N + 5 * K + 100 * ta + 10 * tb)
    A = rng.standard_normal((K, M) if ta else (M, K)).astype(np.float32)
    B = rng.standard_normal((N, K) if tb else (K, N)).astype(np.float32)
    Ar, Br = mlp_ref.bf16(A), mlp_ref.bf16(B)
    opA, opB = (Ar.T if ta else Ar), (Br.T if tb else Br)
    got = warmstart.mfma_gemm(A, B, bool(ta), bool(tb)).astype(np.float64)
    assert np.all(np.abs(got - opA @ opB) <= K * 2.0 ** -23 * (np.abs(opA) @ np.abs(opB)) + 1e-30)


@pytest.mark.parametrize("dims,rows", [((16, 1024, 40), 1024), ((5, 256, 2056), 272)])
def test_gradient_with_layers_in_both_forms(dims, rows):
    net = warmstart.MLP(*dims, seed=3)
    rng = np.random.default_rng(3)
    p = (rng.standard_normal(net.num_params) * 0.05).astype(np.float32)
    net.set_params(p)
    X = rng.standard_normal((rows, dims[0])).astype(np.float32)
    T = rng.standard_normal((rows, dims[2])).astype(np.float32)
    loss, g = net.loss_grad(X, T)
    rl, rg = mlp_ref.loss_grad(p, dims, X, T, bf16_products=True)
    net.close()
    # the bounds of the gradient test at smaller sizes
    assert abs(loss - rl) <= 1e-4 * rl
    assert np.linalg.norm(g - rg) <= 2e-3 * np.linalg.norm(rg)
