"""fp32 contractions whose values are cut into three bf16 parts: errors of fp32 size, small operands with large partners, and the
values that leave the range of the parts (infinities, NaN, numbers near its upper end), which take the fp32 instruction."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, in_parts, stable_seed

pytestmark = pytest.mark.gpu

DENSE, SPLIT = "dense_gemm_kernel<f32>", "split_gemm_kernel<f32>"
# M, N, K and the kernel that takes parts: whole 128 x 128 tiles, ragged ones, slices of a long ragged contraction; two sizes that
# stay on the fp32 instruction in 64 x 64 tiles
SIZES = [(2048, 2048, 64, DENSE), (2047, 2050, 40, None), (1280, 1152, 1031, None), (2048, 1664, 16, DENSE), (1921, 2047, 100, SPLIT),
         (1489, 1707, 2311, SPLIT)]


def product(gpu, w, x):
    return gpu.matmul(dev(gpu, w, "f32"), dev(gpu, x, "f32")).to_numpy()


def in_parts_of(gpu, f, *arrays):
    arrays = [dev(gpu, a, "f32") for a in arrays]
    return in_parts(gpu, lambda: f(*arrays))


@pytest.mark.parametrize("size", range(len(SIZES)))
def test_error_is_that_of_fp32(gpu, size):
    """Rounding a partial sum of k terms leaves an error uniform in 2^-24 of it, 2^-24 / sqrt(3) of sqrt(k / K) of the result in
    the mean square; at most K independent ones add up to 2^-24 sqrt(K / 6), twice of which is allowed.  The products are exact
    to 2^-26 of the terms, whose 2-norm is the result's."""
    M, N, K, kernel = SIZES[size]
    rng = np.random.default_rng(stable_seed("split", size))
    w, x = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    assert in_parts_of(gpu, gpu.matmul, w, x) == ({kernel: 1} if kernel else {})
    want = w.astype(np.float64) @ x.astype(np.float64)
    err = product(gpu, w, x).astype(np.float64) - want
    assert np.linalg.norm(err) <= (2.0 ** -23 * np.sqrt(K / 6) + 2.0 ** -26) * np.linalg.norm(want)


@pytest.mark.parametrize("M,N", [(2048, 2048), (1921, 2047)])
def test_an_outer_product_is_rounded_once(gpu, M, N):
    """Whole and ragged 128 x 128 tiles."""
    rng = np.random.default_rng(stable_seed("split-outer", M))
    w, x = rng.normal(size=(M, 1)).astype(np.float32), rng.normal(size=(1, N)).astype(np.float32)
    np.testing.assert_array_equal(product(gpu, w, x), w * x)


@pytest.mark.parametrize("size", range(len(SIZES)))
def test_values_without_parts(gpu, size):
    M, N, K, kernel = SIZES[size]
    rng = np.random.default_rng(stable_seed("split-special", size))
    # multiples of 1/4 up to 2: a value with one bf16 part, so an infinite partner meets parts that are zero
    w, x = (rng.integers(1, 9, size=s).astype(np.float32) / 4 for s in ((M, K), (K, N)))
    big = np.finfo(np.float32).max
    w[3, 1], w[140, 2], w[141, 0], w[M - 1, 3] = np.inf, -np.inf, np.nan, big
    w[M - 1, :3] = w[M - 1, 4:] = 0
    x[3] = 0.5
    got = product(gpu, w, x)
    want = w.astype(np.float64) @ x.astype(np.float64)
    assert (got[3] == np.inf).all() and (got[140] == -np.inf).all() and np.isnan(got[141]).all()
    np.testing.assert_allclose(got[M - 1], 0.5 * big, rtol=1e-6)
    rows = np.setdiff1d(np.arange(M), (3, 140, 141, M - 1))
    np.testing.assert_allclose(got[rows], want[rows], rtol=1e-6)


@pytest.mark.parametrize("scale", [1e-35, 1e-30, 1e30])
def test_numbers_near_the_ends_of_the_range(gpu, scale):
    M, N, K = 2048, 2048, 64
    rng = np.random.default_rng(stable_seed("split-scale", scale))
    w, x = (rng.normal(size=(M, K)) * scale).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    assert_close(product(gpu, w, x) / np.float64(scale), (w.astype(np.float64) @ x.astype(np.float64)) / scale, "f32", "scaled", rel=1e-5)


# channels, width, images and the directions that take parts: whole-tap kernels (96 channels on 32768 rows), any-channel ones (72 on 65536), and
# smaller problems, of which the filter gradient alone has 128 x 128 tiles, or none
FPROP, DGRAD, WGRAD = "conv_fprop_kernel<f32>", "conv_dgrad_kernel<f32>", "conv_wgrad_kernel<f32>"
LAYERS = [((128, 128), 30, 8, [WGRAD]), ((80, 112), 30, 8, [WGRAD]), ((48, 64), 30, 8, []), ((96, 96), 64, 8, [FPROP, DGRAD, WGRAD]),
          ((72, 128), 64, 16, [FPROP, WGRAD]), ((128, 72), 64, 16, [DGRAD, WGRAD])]


@pytest.mark.parametrize("layer", range(len(LAYERS)))
def test_convolution_with_an_infinite_input(gpu, layer):
    """Both gradients and the output of a 3 x 3 convolution: an infinity stays inside the windows that see it."""
    (cin, cout), W, n, kernels = LAYERS[layer]
    H, channels = W, (cin, cout)
    rng = np.random.default_rng(stable_seed("split-conv", channels))
    x = rng.normal(size=(W, H, cin, n)).astype(np.float32)
    w = np.abs(rng.normal(size=(3, 3, cin, cout)) * 0.1).astype(np.float32)
    x[10, 12, 5, 3] = np.inf
    cd = gpu.DenseConvDims(x.shape, w.shape, padding=1)
    dy = rng.normal(size=(W, H, cout, n)).astype(np.float32)
    took = {**in_parts_of(gpu, lambda a, b: gpu.conv(a, b, cd), x, w), **in_parts_of(gpu, lambda a, b: gpu.conv_data_grad(a, b, cd), dy, w),
            **in_parts_of(gpu, lambda a, b: gpu.conv_filter_grad(a, b, cd), x, dy)}
    assert set(took) == set(kernels), took
    y = gpu.conv(dev(gpu, x, "f32"), dev(gpu, w, "f32"), cd).to_numpy()
    inside = np.zeros(y.shape, bool)
    inside[9:12, 11:14, :, 3] = True
    assert (y[inside] == np.inf).all() and np.isfinite(y[~inside]).all()
    x[10, 12, 5, 3] = 0
    clean = gpu.conv(dev(gpu, x, "f32"), dev(gpu, w, "f32"), cd).to_numpy()
    assert_close(y[~inside], clean[~inside].astype(np.float64), "f32", "outside the windows")
    dy[4, 4, 7, 2] = np.inf
    dx = gpu.conv_data_grad(dev(gpu, dy, "f32"), dev(gpu, w, "f32"), cd).to_numpy()
    inside = np.zeros(dx.shape, bool)
    inside[3:6, 3:6, :, 2] = True
    assert (dx[inside] == np.inf).all() and np.isfinite(dx[~inside]).all()
    dw = gpu.conv_filter_grad(dev(gpu, x, "f32"), dev(gpu, dy, "f32"), cd).to_numpy()
    assert np.isfinite(dw[:, :, :, np.arange(cout) != 7]).all() and not np.isfinite(dw[:, :, :, 7]).any()


# Scales of the two operands.  Nothing of an fp32 number may be lost that a large partner brings to light, subnormal numbers included; the last ones
# leave the range that the parts carry (operands from 2^104, sums from 2^80)
PAIRS = [(1e-35, 1e20), (1e20, 1e-36), (1e-37, 1e25), (1e-39, 1e30), (1e30, 1e-41), (1e-41, 1e3), (1e-26, 1.0), (1e30, 1e-30), (1e33, 1e-33), (1e15, 1e15)]


def scaled(rng, scale, shape):
    return (rng.normal(size=shape) * scale).astype(np.float32)


def error(got, want):
    scale = np.linalg.norm(want)
    return np.linalg.norm(got.astype(np.float64) / scale - want / scale)


@pytest.mark.parametrize("a,b", PAIRS)
def test_small_operands_with_large_partners(gpu, a, b):
    """Whole tiles and ragged ones, the bound of test_error_is_that_of_fp32."""
    for M, N, K in ((2048, 2048, 64), (1921, 2047, 100)):
        rng = np.random.default_rng(stable_seed("split-pair", a, b, M))
        w, x = scaled(rng, a, (M, K)), scaled(rng, b, (K, N))
        assert error(product(gpu, w, x), w.astype(np.float64) @ x.astype(np.float64)) <= 2.0 ** -23 * np.sqrt(K / 6) + 2.0 ** -26


@pytest.mark.parametrize("layer", [3, 4, 5])
@pytest.mark.parametrize("a,b", [(1e-37, 1e25), (1e30, 1e-41)])
def test_convolutions_of_small_operands_with_large_partners(gpu, layer, a, b):
    """The three directions of a 3 x 3 convolution that fills the chip; images stand for themselves in the output and the input
    gradient, so only the last one is compared."""
    channels, W, n, kernels = LAYERS[layer]
    cin, cout = channels
    xs, ws = (W, W, cin, n), (3, 3, cin, cout)
    rng = np.random.default_rng(stable_seed("split-pair-conv", a, b, channels))
    x, w, dy = scaled(rng, a, xs), scaled(rng, b, ws), scaled(rng, a, (W, W, cout, n))
    gd, od = gpu.DenseConvDims(xs, ws, padding=1), O.ConvDims(xs[:3] + (1,), ws, padding=1)
    last = lambda t: t[..., -1:].astype(np.float64)
    bound = lambda K: 2.0 ** -23 * np.sqrt(K / 6) + 2.0 ** -26
    got = gpu.conv(dev(gpu, x, "f32"), dev(gpu, w, "f32"), gd).to_numpy()
    assert error(last(got), O.conv(last(x), w.astype(np.float64), od)) <= bound(9 * cin)
    got = gpu.conv_data_grad(dev(gpu, dy, "f32"), dev(gpu, w, "f32"), gd).to_numpy()
    assert error(last(got), O.conv_data_grad(last(dy), w.astype(np.float64), od)) <= bound(9 * cout)
    x, dy = np.ascontiguousarray(x[:32, :32, :, :2]), scaled(rng, b, (32, 32, cout, 2))
    gd, od = (D(x.shape, ws, padding=1) for D in (gpu.DenseConvDims, O.ConvDims))
    got = gpu.conv_filter_grad(dev(gpu, x, "f32"), dev(gpu, dy, "f32"), gd).to_numpy()
    assert error(got, O.conv_filter_grad(x.astype(np.float64), dy.astype(np.float64), od)) <= bound(2 * 32 * 32)
