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
    if single:
        assert "conv_dz_cwhn_pack_kernel" in kernels_of(gpu, lambda: back(dd))
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
