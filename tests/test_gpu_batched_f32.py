"""fp32 products of batches in 64 x 64 tiles at any alignment (gemm_split_batched.h): the ends of tiles in every layout, slices of the contraction, triangular
structures against the general path's rule, and attention through them."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, kernels_of, stable_seed

pytestmark = pytest.mark.gpu

# one to four rows behind a tile (fewer than a vector), one before it, K of one stage, no whole stage, and long enough for slices
SHAPES = [(65, 66, 16), (67, 129, 33), (68, 63, 17), (4, 5, 31), (64, 64, 1999), (97, 131, 700), (128, 192, 515)]


@pytest.mark.parametrize("lhs,rhs", [(2, 1), (1, 1), (2, 2), (1, 2)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products(gpu, lhs, rhs, M, N, K):
    rng = np.random.default_rng(stable_seed("batched f32", lhs, rhs, M, N, K))
    a = rng.normal(size=(M, K, 3) if lhs == 2 else (K, M, 3)).astype(np.float32)
    b = rng.normal(size=(K, N, 3) if rhs == 1 else (N, K, 3)).astype(np.float32)
    da, db, out = dev(gpu, a, "f32"), dev(gpu, b, "f32"), []
    kernels = kernels_of(gpu, lambda: out.append(gpu.batched_matmul(da, db, lhs, rhs)))
    assert set(kernels) == {"split_batched_kernel+slices" if K > 500 else "split_batched_kernel"}
    got = out[0].to_numpy()
    assert_close(got, O.batched_matmul(f64(a), f64(b), lhs, rhs), "f32", f"{M} x {N} x {K} {lhs} {rhs}")
    np.testing.assert_array_equal(got, gpu.batched_matmul(dev(gpu, a, "f32"), dev(gpu, b, "f32"), lhs, rhs).to_numpy())


# queries and keys that end one, two and three behind a tile, within one and after many; few heads (slices) and many; a short last block of the diagonal
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("E,H,L", [(20, 2, 65), (33, 1, 130), (48, 3, 195), (16, 2, 257), (64, 2, 1030), (128, 1, 640), (8, 40, 67)])
def test_attention(gpu, causal, E, H, L):
    rng = np.random.default_rng(stable_seed("attention f32", E, H, L))
    q, k, v, d = (rng.normal(size=(E, H, L, 2)).astype(np.float32) for _ in range(4))
    dq, dk, dv, dd = (dev(gpu, t, "f32") for t in (q, k, v, d))
    out, grads = [], []
    kernels = kernels_of(gpu, lambda: out.extend(gpu.pullback(gpu.scaled_dot_product_attention, dq, dk, dv, 1, 3, None, None, True if causal else None)))
    (y, w), back = out
    kernels_back = kernels_of(gpu, lambda: grads.extend(g.to_numpy() for g in back(dd)))
    # 8 features are less than a stage: the products that contract over them stay on the general tiles
    assert "batched_gemm_kernel<f32>" not in kernels_back and ("batched_gemm_kernel<f32>" in kernels) == (E < 16)
    assert ("split_batched_kernel+softmax_rule" if E >= 16 else "batched_gemm_kernel+softmax_rule") in kernels_back
    for products in (kernels, kernels_back):
        assert ("split_batched_kernel+slices" in products) == (L > 200)
    Q, K, V, D = (np.moveaxis(f64(t), (3, 1, 2, 0), (0, 1, 2, 3)) for t in (q, k, v, d))       # (B, H, L, E)
    z = Q @ np.swapaxes(K, 2, 3) / np.sqrt(E)
    if causal:
        z = np.where(np.arange(L)[:, None] >= np.arange(L)[None, :], z, -np.inf)
    P = np.exp(z - z.max(-1, keepdims=True))
    P /= P.sum(-1, keepdims=True)
    dP = D @ np.swapaxes(V, 2, 3)
    dz = P * (dP - (P * dP).sum(-1, keepdims=True)) / np.sqrt(E)
    back4 = lambda t: np.moveaxis(t, (0, 1, 2, 3), (3, 1, 2, 0))
    assert_close(y.to_numpy(), back4(P @ V), "f32", "y")
    assert_close(w.to_numpy(), np.moveaxis(P, (0, 1, 2, 3), (3, 2, 1, 0)), "f32", "weights")
    for name, g, want in zip("qkv", grads, (dz @ K, np.swapaxes(dz, 2, 3) @ Q, np.swapaxes(P, 2, 3) @ D)):
        assert_close(g, back4(want), "f32", "d" + name)
