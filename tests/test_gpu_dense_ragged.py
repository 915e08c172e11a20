"""Products with few tiles, ragged operands or few columns (gemm_split.h, gemm_skinny.hip) against the fp64 oracle: every
layout at the edges of tiles, stages and slices, the fused layer whose two gradient products share a launch, and the layer
that a handful of tokens pass through."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, rms, stable_seed

pytestmark = pytest.mark.gpu

# below / at / above a tile of 64 and of 128, rows of fewer than two vectors, K of one stage, of a stage and a bit, of
# several slices with a ragged last one
SHAPES = [(8, 9, 32), (64, 64, 33), (65, 63, 64), (9, 130, 95), (129, 64, 4099), (130, 131, 1023), (517, 301, 70), (640, 1030, 45)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("transA", [False, True])
@pytest.mark.parametrize("transB", [False, True])
def test_ragged_products(gpu, dtype, transA, transB):
    rng = np.random.default_rng(stable_seed("ragged", dtype, transA, transB))
    for (M, N, K) in SHAPES:
        A = rng.normal(size=(K, M) if transA else (M, K))
        B = rng.normal(size=(N, K) if transB else (K, N))
        A, B, bias = host_inputs(dtype, A, B, rng.normal(size=M))
        want = (f64(A).T if transA else f64(A)) @ (f64(B).T if transB else f64(B)) + f64(bias)[:, None]
        got = gpu.matmul(dev(gpu, A, dtype), dev(gpu, B, dtype), dev(gpu, bias, dtype), transA, transB).to_numpy()
        again = gpu.matmul(dev(gpu, A, dtype), dev(gpu, B, dtype), dev(gpu, bias, dtype), transA, transB).to_numpy()
        assert_close(got, want, dtype, f"{dtype} ragged matmul {M}x{N}x{K} tA={transA} tB={transB}")
        np.testing.assert_array_equal(got, again)          # slices are added in a fixed order


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_zeroed_overlap_is_not_multiplied(gpu, dtype):
    """The last stage repeats k that are done: they count as zero in both operands, so an infinity there must not turn
    into a NaN and must count once."""
    M, N, K = 70, 66, 45
    A, B = np.ones((M, K)), np.ones((K, N))
    A[3, 20] = np.inf                                       # k = 20 lies in the part of the last stage that is repeated
    for transA in (False, True):
        got = gpu.matmul(dev(gpu, A.T if transA else A, dtype), dev(gpu, B, dtype), None, transA, False).to_numpy()
        want = np.full((M, N), float(K))
        want[3] = np.inf
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "tanh", "gelu"])
def test_fused_layer_with_gradients_in_one_launch(gpu, dtype, act):
    rng = np.random.default_rng(stable_seed("pair", dtype, act))
    for (M, K, N) in [(64, 32, 32), (65, 47, 33), (200, 300, 70), (130, 64, 515)]:
        W, x, b, delta = host_inputs(dtype, rng.normal(size=(M, K)) / np.sqrt(K), rng.normal(size=(K, N)), 0.1 * rng.normal(size=M),
                                     rng.normal(size=(M, N)))
        y, back = gpu.pullback(gpu.fused_dense_bias_activation, act, *(dev(gpu, a, dtype) for a in (W, x, b)))
        gW, gx, gb = back(dev(gpu, delta, dtype))
        wy, wdW, wdx, wdb = O.fused_dense_pullback(act, f64(W), f64(x), f64(b), f64(delta))
        dz = O.grad_activation(f64(delta), wy, act, O.matmuladd(f64(W), f64(x), f64(b)))
        if dtype == "bf16":                                 # y, the pre-activation and dz are stored in bf16 in between
            pre = f64(O.round_to_bf16(O.matmuladd(f64(W), f64(x), f64(b)).astype(np.float32)))
            dz = O.grad_activation(f64(delta), f64(O.round_to_bf16(wy.astype(np.float32))), act, pre)
            wdb = dz.sum(axis=1)
            dz = f64(O.round_to_bf16(dz.astype(np.float32)))
            wdW, wdx = dz @ f64(x).T, f64(W).T @ dz
        tag = f"{dtype} {act} {M}x{K}x{N}"
        assert_close(y.to_numpy(), wy, dtype, tag + " y")
        assert_close(gW.to_numpy(), wdW, dtype, tag + " dW", scale=np.sqrt(N) * rms(dz) * rms(x))
        assert_close(gx.to_numpy(), wdx, dtype, tag + " dx", scale=np.sqrt(M) * rms(dz) * rms(W))
        assert_close(gb.to_numpy(), wdb, dtype, tag + " db")


def test_gradients_of_a_layer_with_more_tiles_than_counters(gpu):
    """dW has 70000 tiles and one slice, dx one tile and sixteen slices: only dx takes arrival counters.  All values are
    -1, 0 or 1 and every sum stays below M < 2^24, so fp32 holds each partial sum exactly, whatever the order (rounded
    inputs would need a bound for sums of 4.5 million terms)."""
    M, K, N = 70000 * 64, 8, 16
    rng = np.random.default_rng(stable_seed("tall"))
    W, x, delta = (rng.integers(-1, 2, size=s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    args = tuple(dev(gpu, a, "f32") for a in (W, x, np.zeros(M, np.float32)))
    _, back = gpu.pullback(gpu.fused_dense_bias_activation, "identity", *args)
    gW, gx, gb = back(dev(gpu, delta, "f32"))
    np.testing.assert_array_equal(gW.to_numpy(), f64(delta) @ f64(x).T)
    np.testing.assert_array_equal(gx.to_numpy(), f64(W).T @ f64(delta))
    np.testing.assert_array_equal(gb.to_numpy(), f64(delta).sum(axis=1))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "gelu"])
def test_few_columns(gpu, dtype, act):
    rng = np.random.default_rng(stable_seed("skinny", dtype, act))
    for (M, N, K) in [(128, 1, 1), (131, 16, 31), (256, 2, 32), (300, 5, 1000), (2055, 3, 4097), (64, 15, 517)]:
        W, x, b = host_inputs(dtype, rng.normal(size=(M, K)) / np.sqrt(K), rng.normal(size=(K, N)), rng.normal(size=M))
        args = tuple(dev(gpu, a, dtype) for a in (W, x, b))
        want = O.fused_dense_pullback(act, f64(W), f64(x), f64(b), np.zeros((M, N)))[0]
        got = gpu.fused_dense_bias_activation(act, *args).to_numpy()
        assert_close(got, want, dtype, f"{dtype} {act} {M}x{N}x{K}")
        np.testing.assert_array_equal(got, gpu.pullback(gpu.fused_dense_bias_activation, act, *args)[0].to_numpy())


@pytest.mark.parametrize("dtype,M,N,K,split", [
    ("bf16", 1280, 2048, 512, False), ("bf16", 1024, 2048, 512, True), ("bf16", 1536, 2048, 128, True), ("bf16", 1664, 2048, 128, False),
    ("f32", 1664, 2048, 128, False), ("f32", 1536, 2048, 128, True),
])
def test_whole_tiles_that_nearly_fill_the_chip(gpu, dtype, M, N, K, split):
    """Either side of the line between the big-tile kernels and those of gemm_split.h (small whole numbers: exact in fp32)."""
    rng = np.random.default_rng(stable_seed("whole", M, K))
    A, B = rng.integers(-2, 3, size=(M, K)).astype(np.float32), rng.integers(-2, 3, size=(K, N)).astype(np.float32)
    dA, dB = dev(gpu, A, dtype), dev(gpu, B, dtype)
    out = []
    names = kernels_of(gpu, lambda: out.append(gpu.matmul(dA, dB, None, False, False)))
    assert any("split" in n for n in names) == split, names
    want = A @ B
    np.testing.assert_array_equal(out[0].to_numpy(), want if dtype == "f32" else O.round_to_bf16(want))


@pytest.mark.parametrize("dtype,M,K,skinny", [
    ("bf16", 32768, 64, True), ("bf16", 32769, 64, False), ("f32", 32768, 100, True), ("f32", 32769, 100, False),
    ("f32", 32769, 256, True), ("f32", 32769, 260, False), ("f32", 16384, 15, True), ("f32", 16385, 15, False),
])
def test_few_columns_and_many_rows(gpu, dtype, M, K, skinny):
    """Rows for more workgroups than the chip takes at once go to the tiled kernels unless K is long (exact whole numbers)."""
    rng = np.random.default_rng(stable_seed("tall layer", M, K))
    W, x = rng.integers(-2, 3, size=(M, K)).astype(np.float32), rng.integers(-2, 3, size=(K, 3)).astype(np.float32)
    dW, dx, out = dev(gpu, W, dtype), dev(gpu, x, dtype), []
    names = kernels_of(gpu, lambda: out.append(gpu.matmul(dW, dx, None, False, False)))
    assert any("skinny" in n for n in names) == skinny, names
    want = W @ x
    np.testing.assert_array_equal(out[0].to_numpy(), want if dtype == "f32" else O.round_to_bf16(want))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_input_gradient_in_the_inputs_own_memory(gpu, dtype):
    """A caller that is done with x may have dx written over it: dW is finished before dx starts then."""
    M, K, N = 130, 77, 301
    rng = np.random.default_rng(stable_seed("alias", dtype))
    W, x, dz = (dev(gpu, rng.integers(-2, 3, size=s).astype(np.float32), dtype) for s in ((M, K), (K, N), (M, N)))
    want_W, want_x = (O.round_to_bf16(a) if dtype == "bf16" else a for a in (dz.to_numpy() @ x.to_numpy().T, W.to_numpy().T @ dz.to_numpy()))
    dW = gpu.DeviceArray((M, K), dtype)
    call = lambda: gpu._lib.call("luxhip_fused_dense_bwd", gpu.current_stream(), x.code, 0, M, K, N, dz.ptr, None, None, W.ptr, M, x.ptr, K, None,
                                 dW.ptr, x.ptr, None)
    assert not any("pair" in n for n in kernels_of(gpu, call))
    np.testing.assert_array_equal(dW.to_numpy(), want_W)
    np.testing.assert_array_equal(x.to_numpy(), want_x)
