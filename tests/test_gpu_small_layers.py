"""Small dense layers (gemm_small.hip): fp32 products in tiles of 32 whose contraction is divided among the waves of a workgroup, and the
pullback in one launch, against the fp64 oracle at the edges of tiles and of the eight waves' shares of k."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, rms, stable_seed

pytestmark = pytest.mark.gpu

# below, at and above a tile; K of one step per wave, of fewer steps than waves, of a group and a step more, ragged last steps
PRODUCTS = [(4, 5, 32), (31, 33, 64), (32, 32, 65), (33, 130, 71), (64, 9, 255), (257, 63, 256), (96, 100, 521), (1, 500, 40)]
LAYERS = [(8, 1, 8), (8, 40, 9), (31, 33, 32), (32, 32, 33), (33, 65, 64), (65, 31, 257), (100, 9, 70), (257, 64, 12)]     # M, K, N


@pytest.mark.parametrize("transA", [False, True])
@pytest.mark.parametrize("transB", [False, True])
def test_products(gpu, transA, transB):
    rng = np.random.default_rng(stable_seed("small", transA, transB))
    took = 0
    for (M, N, K) in PRODUCTS:
        A, B, bias = rng.normal(size=(K, M) if transA else (M, K)), rng.normal(size=(N, K) if transB else (K, N)), rng.normal(size=M)
        A, B, bias = host_inputs("f32", A, B, bias)
        dA, dB, db = (dev(gpu, v, "f32") for v in (A, B, bias))
        out = []
        took += "small_gemm_kernel" in kernels_of(gpu, lambda: out.append(gpu.matmul(dA, dB, db, transA, transB)))
        want = (f64(A).T if transA else f64(A)) @ (f64(B).T if transB else f64(B)) + f64(bias)[:, None]
        assert_close(out[0].to_numpy(), want, "f32", f"small matmul {M}x{N}x{K} tA={transA} tB={transB}")
        np.testing.assert_array_equal(out[0].to_numpy(), gpu.matmul(dA, dB, db, transA, transB).to_numpy())
    assert took >= 5                                    # the others are products of few rows or columns


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "relu", "tanh", "sigmoid", "swish", "gelu", "softplus", "logsigmoid", "lisht"])
def test_pullbacks(gpu, dtype, act):
    rng = np.random.default_rng(stable_seed("small layer", dtype, act))
    for (M, K, N) in LAYERS:
        # Pre-activations are multiples of 1/8 below 32, which bf16 holds: with others one that lies at a tie is stored a step (2^-8 of it) off,
        # and with |x act''(x)| up to 0.6, |delta| and |x| up to 4 that alone is 0.04 of a gradient over 12 columns, past the tolerance.
        W, x, b, delta = host_inputs(dtype, rng.integers(-2, 3, size=(M, K)) / 4, rng.integers(-2, 3, size=(K, N)) / 2, rng.integers(-2, 3, size=M) / 8,
                                     rng.normal(size=(M, N)))
        y, back = gpu.pullback(gpu.fused_dense_bias_activation, act, *(dev(gpu, a, dtype) for a in (W, x, b)))
        d, grads = dev(gpu, delta, dtype), []
        assert set(kernels_of(gpu, lambda: grads.extend(back(d)))) == {"small_layer_bwd_kernel"}
        z = O.matmuladd(f64(W), f64(x), f64(b))
        yy, pre = O.fused_dense_bias_activation(act, f64(W), f64(x), f64(b)), z
        if dtype == "bf16":                             # y, the pre-activation and dz have the precision of storage
            yy = f64(O.round_to_bf16(yy.astype(np.float32)))
            pre = f64(O.round_to_bf16(z.astype(np.float32)))
        dz = O.grad_activation(f64(delta), yy, act, pre)
        wdb = dz.sum(axis=1)
        if dtype == "bf16":
            dz = f64(O.round_to_bf16(dz.astype(np.float32)))
        tag = f"{dtype} {act} {M}x{K}x{N}"
        assert_close(grads[0].to_numpy(), dz @ f64(x).T, dtype, tag + " dW", scale=np.sqrt(N) * rms(dz) * rms(x))
        assert_close(grads[1].to_numpy(), f64(W).T @ dz, dtype, tag + " dx", scale=np.sqrt(M) * rms(dz) * rms(W))
        assert_close(grads[2].to_numpy(), wdb, dtype, tag + " db", scale=np.sqrt(N) * rms(dz))


def test_what_is_repeated_counts_as_zero(gpu):
    """The last eight k are moved back: an infinity among those that are done counts once, in dW (k = n) and in dx (k = m)."""
    M, K, N = 37, 5, 43
    W, x, delta = np.ones((M, K)), np.ones((K, N)), np.ones((M, N))
    delta[30, 36] = np.inf
    args = tuple(dev(gpu, a, "f32") for a in (W, x, np.zeros(M)))
    _, back = gpu.pullback(gpu.fused_dense_bias_activation, "identity", *args)
    gW, gx, gb = (g.to_numpy() for g in back(dev(gpu, delta, "f32")))
    wW, wx, wb = np.full((M, K), float(N)), np.full((K, N), float(M)), np.full(M, float(N))
    wW[30], wx[:, 36], wb[30] = np.inf, np.inf, np.inf
    np.testing.assert_array_equal(gW, wW)
    np.testing.assert_array_equal(gx, wx)
    np.testing.assert_array_equal(gb, wb)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_larger_layers_keep_their_kernels(gpu, dtype):
    """Past the line the pass over delta and the pair of products run, and agree with the oracle."""
    M, K, N = 464, 1296, 250
    rng = np.random.default_rng(stable_seed("past", dtype))
    W, x, b, delta = host_inputs(dtype, rng.normal(size=(M, K)) / np.sqrt(K), rng.normal(size=(K, N)), rng.normal(size=M), rng.normal(size=(M, N)))
    _, back = gpu.pullback(gpu.fused_dense_bias_activation, "identity", *(dev(gpu, a, dtype) for a in (W, x, b)))
    d, grads = dev(gpu, delta, dtype), []
    assert "small_layer_bwd_kernel" not in kernels_of(gpu, lambda: grads.extend(back(d)))
    assert_close(grads[0].to_numpy(), f64(delta) @ f64(x).T, dtype, "dW", scale=np.sqrt(N) * rms(delta) * rms(x))
    assert_close(grads[1].to_numpy(), f64(W).T @ f64(delta), dtype, "dx", scale=np.sqrt(M) * rms(delta) * rms(W))
