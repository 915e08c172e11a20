"""The convolution pullback's single pass over the cotangent (dz channel-contiguous with padded channels, as it lies where a kernel reads it so, and the bias
gradient's partial sums) at the ends of its tiles and on either side of its rule."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, rms, stable_seed

pytestmark = pytest.mark.gpu

# (width of the output plane, input channels, output channels, samples, groups, single pass): one position behind a tile of 64 and one before it, channels one behind
# a vector and a tile of 64, whole vectors whose dz is read as it lies (bf16: 64 positions, 8 channels), planes and channel counts below the rule, groups
CASES = [((65, 1), 5, 17, 3, 1, True), ((7, 9), 8, 65, 2, 1, True), ((13, 13), 3, 64, 3, 1, True), ((8, 8), 8, 24, 4, 1, True), ((16, 16), 64, 64, 3, 1, True),
         ((33, 1), 4, 16, 2, 1, True), ((31, 1), 4, 16, 2, 1, False), ((9, 9), 4, 15, 2, 1, False), ((12, 12), 16, 32, 2, 2, True), ((11, 11), 6, 18, 2, 3, False)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["relu", "swish", "identity"])
@pytest.mark.parametrize("plane,cin,cout,n,groups,single", CASES)
def test_pullback(gpu, dtype, act, plane, cin, cout, n, groups, single):
    (W, H), k = plane, 3 if plane[1] > 1 else 1
    xs, ws = (W, H, cin, n), (k, k, cin // groups, cout)
    rng = np.random.default_rng(stable_seed("dz", dtype, act, xs, ws))
    x, w, b, delta = host_inputs(dtype, rng.normal(size=xs), rng.normal(size=ws) / np.sqrt(k * k * cin / groups), rng.normal(size=cout),
                                 rng.normal(size=(W, H, cout, n)))
    gd, od = gpu.DenseConvDims(xs, ws, padding=k // 2, groups=groups), O.ConvDims(xs, ws, padding=k // 2, groups=groups)
    y, back = gpu.pullback(gpu.fused_conv_bias_activation, act, dev(gpu, w, dtype), dev(gpu, x, dtype), dev(gpu, b, dtype), gd)
    dd = dev(gpu, delta, dtype)
    assert ("conv_dz_cwhn_pack_kernel" in kernels_of(gpu, lambda: back(dd))) == single
    gw, gx, gb = back(dd)
    wy, wdw, wdx, wdb = O.fused_conv_pullback(act, f64(w), f64(x), f64(b), od, f64(delta))
    if dtype == "bf16":                                     # y, the pre-activation and dz are stored in bf16 in between
        pre = O.bias_add(O.conv(f64(x), f64(w), od), f64(b))
        yq, preq = (f64(O.round_to_bf16(a.astype(np.float32))) for a in (wy, pre))
        dzx = O.grad_activation(f64(delta), yq, act, preq)
        dz = f64(O.round_to_bf16(dzx.astype(np.float32)))
        wdw, wdx, wdb = O.conv_filter_grad(f64(x), dz, od), O.conv_data_grad(dz, f64(w), od), O.grad_bias_add(b, dzx)
    per = np.sqrt(W * H * n) * rms(delta)                   # terms of a sum over one channel's positions
    assert_close(gw.to_numpy(), wdw, dtype, "dw", scale=per * rms(x) * 0.5)
    assert_close(gx.to_numpy(), wdx, dtype, "dx", scale=np.sqrt(k * k * cout / groups) * rms(delta) * rms(w) * 0.5)
    assert_close(gb.to_numpy(), wdb, dtype, "db", scale=per * 0.5)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("tap", [0, 42])
def test_filter_that_is_large_beside_the_cotangent(gpu, dtype, tap):
    """One tile of the cotangent and 16.9 million filter elements, more than its launch's z slices hold: they are packed in a launch of their own, for
    the general kernels and for the whole-tap ones."""
    xs, ws = (8, 8, 5376, 1), (7, 7, 5376, 64)
    rng = np.random.default_rng(stable_seed("large filter", dtype))
    x, w, b, delta = host_inputs(dtype, rng.standard_normal(xs, np.float32), rng.standard_normal(ws, np.float32), rng.standard_normal(64, np.float32),
                                 rng.standard_normal((8, 8, 64, 1), np.float32))
    gd, od = gpu.DenseConvDims(xs, ws, padding=3), O.ConvDims(xs, ws, padding=3)
    gpu.set_option("conv_tile", tap)
    try:
        _, back = gpu.pullback(gpu.fused_conv_bias_activation, "identity", dev(gpu, w, dtype), dev(gpu, x, dtype), dev(gpu, b, dtype), gd)
        grads, dd = [], dev(gpu, delta, dtype)
        kernels = kernels_of(gpu, lambda: grads.extend(back(dd)))
    finally:
        gpu.set_option("conv_tile", 0)
    assert {"conv_dz_cwhn_pack_kernel", "pack_filter_kernel" if tap else "whcn_to_cwhn_kernel"} <= set(kernels)
    per = rms(delta) * 8                                    # sums of up to 64 positions, and of 7 x 7 x 64 cotangents
    assert_close(grads[0].to_numpy(), O.conv_filter_grad(f64(x), f64(delta), od), dtype, "dw", scale=per * rms(x) * 0.5)
    assert_close(grads[1].to_numpy(), O.conv_data_grad(f64(delta), f64(w), od), dtype, "dx", scale=per * 7 * rms(w) * 0.5)
    assert_close(grads[2].to_numpy(), f64(delta).sum((0, 1, 3)), dtype, "db", scale=per * 0.5)
