"""Sums of many partial sums of few values: the filter gradient's slices in parts, the bias gradient of a dense layer over a long batch."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, stable_seed

pytestmark = pytest.mark.gpu


# (w, cin, cout, k, n): hundreds of slices of few values (64 parts at most), slices that are no multiple of the parts, a column
# that ends inside a workgroup, few slices (one part)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("w,cin,cout,k,n", [(48, 16, 8, 1, 30), (37, 24, 19, 1, 41), (41, 5, 3, 3, 13), (9, 16, 16, 3, 2)])
def test_filter_gradient(gpu, dtype, w, cin, cout, k, n):
    rng = np.random.default_rng(stable_seed("parts", dtype, w, cin, cout, k, n))
    x, wt, b, d = host_inputs(dtype, rng.normal(size=(w, w, cin, n)), rng.normal(size=(k, k, cin, cout)), rng.normal(size=cout), rng.normal(size=(w, w, cout, n)))
    dims = gpu.DenseConvDims(x.shape, wt.shape, padding=k // 2)
    _, back = gpu.pullback(gpu.fused_conv_bias_activation, "identity", dev(gpu, wt, dtype), dev(gpu, x, dtype), dev(gpu, b, dtype), dims)
    gw, gx, gb = back(dev(gpu, d, dtype))
    p = k // 2
    xp = np.pad(f64(x), ((p, p), (p, p), (0, 0), (0, 0)))
    want = np.empty(wt.shape)
    for i in range(k):
        for j in range(k):
            want[k - 1 - i, k - 1 - j] = np.tensordot(xp[i:i + w, j:j + w], f64(d), ((0, 1, 3), (0, 1, 3)))
    assert_close(gw.to_numpy(), want, dtype, "dw")
    assert_close(gb.to_numpy().reshape(-1), f64(d).sum((0, 1, 3)), dtype, "db")


# 16 channels at a time over more than 128 slices, with and without whole trips of eight; 64 channels at a time
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("M,N", [(248, 1456), (17, 2048), (33, 9000), (70, 300)])
def test_dense_bias_gradient(gpu, dtype, M, N):
    rng = np.random.default_rng(stable_seed("bias", dtype, M, N))
    W, x, b, d = host_inputs(dtype, rng.normal(size=(M, 32)), rng.normal(size=(32, N)), rng.normal(size=M), rng.normal(size=(M, N)))
    _, back = gpu.pullback(gpu.fused_dense_bias_activation, "identity", dev(gpu, W, dtype), dev(gpu, x, dtype), dev(gpu, b, dtype))
    gW, gx, gb = back(dev(gpu, d, dtype))
    assert_close(gb.to_numpy().reshape(-1), f64(d).sum(1), dtype, "db")
    assert_close(gW.to_numpy(), f64(d) @ f64(x).T, dtype, "dW")


@pytest.mark.parametrize("dtype,K", [("bf16", 1440), ("f32", 1203)])
@pytest.mark.parametrize("N", [1, 4, 5, 8, 9, 12, 13, 16])
def test_slices_of_a_few_columns(gpu, dtype, K, N):
    """Serving a few columns, the contraction in several slices: one to four values a thread.  Values are -1, 0 or 1, so every partial sum and
    (below 2^8 in bf16: 1440 terms of variance 4/9 stay within 6.5 x 25) the result are exact."""
    rng = np.random.default_rng(stable_seed("few columns", dtype, N))
    W, x = rng.integers(-1, 2, size=(700, K)).astype(np.float32), rng.integers(-1, 2, size=(K, N)).astype(np.float32)
    dW, dx, out = dev(gpu, W, dtype), dev(gpu, x, dtype), []
    assert set(kernels_of(gpu, lambda: out.append(gpu.matmul(dW, dx, None, False, False)))) == {f"skinny_gemm_kernel<{dtype}>+slices"}
    got = out[0].to_numpy()
    want = W @ x
    assert np.abs(want).max() < 256
    np.testing.assert_array_equal(got, want)
