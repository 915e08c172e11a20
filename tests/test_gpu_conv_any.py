"""Convolutions of any channel count and stride (conv_any.h) against the fp64 oracle: padded channels, the residues of a
strided input gradient apart and merged, taps that some residues do not have and residues without taps, non-finite cotangents,
groups in one launch and a few at a time, contractions shorter than a stage and cut into slices, and the kept copy of x whose
channels the kernels would pad."""
import ctypes as C

import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, rms, stable_seed

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad, dilation, groups, flip
    ((17, 15, 3, 3), (7, 7, 3, 20), 2, 3, 1, 1, False),              # residues merged into columns: 2 x 2 of 3 channels
    ((9, 11, 6, 2), (5, 4, 2, 9), 3, (2, 1, 0, 2), 1, 3, True),      # 9 residues, groups of 2 -> 3 channels
    ((13, 11, 5, 3), (2, 4, 5, 7), (2, 3), (1, 0, 3, 3), (3, 2), 1, False),   # stride and dilation share no factor
    ((14, 10, 6, 2), (3, 3, 6, 5), 2, 2, 2, 1, False),               # ... share a factor: residues without taps
    ((19, 17, 72, 2), (3, 3, 72, 40), 2, 1, 1, 1, False),            # one problem per residue
    ((16, 9, 24, 3), (1, 1, 24, 33), 2, 0, 1, 1, False),             # three of four residues are zero
    ((4, 4, 3, 1), (3, 3, 3, 4), 2, 1, 1, 1, False),                 # 4 output positions: less than a stage
    ((6, 6, 200, 1), (5, 5, 200, 24), 1, 2, 1, 1, False),            # few rows, 5000 k: slices
    ((23, 9, 61, 2), (3, 3, 61, 130), 1, (0, 1, 1, 0), 1, 1, True),  # more than 128 columns, ragged in everything
    ((5, 3, 8, 2), (3, 3, 8, 8), 4, 2, 1, 1, False),                 # stride beyond the filter
    ((16, 15, 32, 2), (4, 5, 32, 24), (4, 5), 0, 1, 1, False),       # as many taps as residues, whole column tiles: one problem
    ((33, 34, 32, 2), (1, 1, 32, 24), 9, 0, 1, 1, False),            # one residue of 81 has taps
    ((20, 19, 33, 1), (3, 2, 33, 8), (7, 6), (2, 0, 1, 3), (2, 3), 1, True),   # 6 of 42, dilated; an odd number of bf16 elements
    ((6, 5, 4, 2), (2, 2, 2, 6), 1000, 0, 1, 2, False),              # stride far beyond the input
    ((9, 8, 40, 2), (3, 3, 1, 40), 1, 1, 1, 40, False),              # depthwise: a group per block of the grid
    ((9, 8, 40, 2), (5, 3, 1, 80), 2, 1, 1, 40, True),               # ... two channels out of one, merged residues
    ((5, 4, 300, 1), (2, 2, 100, 21), 1, 0, 1, 3, False),            # groups with slices
]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_conv_any(gpu, dtype, case):
    xs, ws, stride, pad, dil, groups, flip = CASES[case]
    rng = np.random.default_rng(stable_seed("conv_any", case))
    kw = dict(stride=stride, padding=pad, dilation=dil, groups=groups, flipkernel=flip)
    gd, od = gpu.DenseConvDims(xs, ws, **kw), O.ConvDims(xs, ws, **kw)
    x, w, b, dy = host_inputs(dtype, rng.normal(size=xs), rng.normal(size=ws) / np.sqrt(ws[0] * ws[1] * ws[2]), rng.normal(size=ws[3]),
                              rng.normal(size=od.y_shape()))
    dx_, dw_, db_, ddy = (dev(gpu, a, dtype) for a in (x, w, b, dy))
    wy, wdw, wdx = O.conv(f64(x), f64(w), od), O.conv_filter_grad(f64(x), f64(dy), od), O.conv_data_grad(f64(dy), f64(w), od)
    tag = f"{dtype} conv_any {case}"
    y = gpu.fused_conv_bias_activation("relu", dw_, dx_, db_, gd)
    assert_close(y.to_numpy(), np.maximum(wy + f64(b)[None, None, :, None], 0.0), dtype, tag + " y")
    gx, gw = gpu.conv_data_grad(ddy, dw_, gd), gpu.conv_filter_grad(dx_, ddy, gd)
    assert_close(gx.to_numpy(), wdx, dtype, tag + " dx")
    assert_close(gw.to_numpy(), wdw, dtype, tag + " dw")
    # the fused pullback (identity: dz is the cotangent) makes the same gradients
    _, back = gpu.pullback(gpu.fused_conv_bias_activation, "identity", dw_, dx_, db_, gd)
    fw, fx, fb = back(ddy)
    np.testing.assert_array_equal(fx.to_numpy(), gx.to_numpy())
    np.testing.assert_array_equal(fw.to_numpy(), gw.to_numpy())
    assert_close(fb.to_numpy(), f64(dy).sum(axis=(0, 1, 3)), dtype, tag + " db")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["relu", "gelu"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_fused_pullback_with_an_activation(gpu, dtype, act, case):
    """Derivatives from the output (relu) and from the pre-activation (gelu), through the dz pass of either kind (bf16 channels
    in whole vectors: one pass writes both layouts, else a pass and a padding copy)."""
    xs, ws, stride, pad, dil, groups, flip = CASES[case]
    rng = np.random.default_rng(stable_seed("conv_any act", case, act))
    kw = dict(stride=stride, padding=pad, dilation=dil, groups=groups, flipkernel=flip)
    gd, od = gpu.DenseConvDims(xs, ws, **kw), O.ConvDims(xs, ws, **kw)
    x, w, b, delta = host_inputs(dtype, rng.normal(size=xs), rng.normal(size=ws) / np.sqrt(ws[0] * ws[1] * ws[2]), 0.1 * rng.normal(size=ws[3]),
                                 rng.normal(size=od.y_shape()))
    y, back = gpu.pullback(gpu.fused_conv_bias_activation, act, dev(gpu, w, dtype), dev(gpu, x, dtype), dev(gpu, b, dtype), gd)
    gw, gx, gb = back(dev(gpu, delta, dtype))
    wy, wdw, wdx, wdb = O.fused_conv_pullback(act, f64(w), f64(x), f64(b), od, f64(delta))
    if dtype == "bf16":                                     # y, the pre-activation and dz are stored in bf16 in between
        pre = O.bias_add(O.conv(f64(x), f64(w), od), f64(b))
        yq, preq = (f64(O.round_to_bf16(a.astype(np.float32))) for a in (wy, pre))
        dzx = O.grad_activation(f64(delta), yq, act, preq)
        dz = f64(O.round_to_bf16(dzx.astype(np.float32)))
        wdw, wdx, wdb = O.conv_filter_grad(f64(x), dz, od), O.conv_data_grad(dz, f64(w), od), O.grad_bias_add(b, dzx)
    tag = f"{dtype} {act} conv_any {case}"
    per = np.sqrt(np.prod(od.y_shape()) / ws[3]) * rms(delta)          # terms of a sum over one channel's positions
    assert_close(y.to_numpy(), wy, dtype, tag + " y")
    assert_close(gw.to_numpy(), wdw, dtype, tag + " dw", scale=per * rms(x) * 0.5)
    assert_close(gx.to_numpy(), wdx, dtype, tag + " dx", scale=np.sqrt(ws[0] * ws[1] * ws[3] / groups) * rms(delta) * rms(w) * 0.5)
    assert_close(gb.to_numpy(), wdb, dtype, tag + " db", scale=per * 0.5)


@pytest.mark.parametrize("xs,ws,stride,dil,launches", [
    ((64, 64, 32, 1), (8, 8, 32, 16), 8, 1, 1),              # residues as columns
    ((64, 64, 32, 1), (1, 1, 32, 16), 32, 1, 1),             # one residue has taps, the rest is cleared
    ((64, 64, 8, 1), (3, 3, 8, 8), 4, 2, 1),                 # four residues of sixteen have taps
    ((40, 40, 8, 1), (3, 3, 8, 8), 5, 2, 3),                 # nine of twenty-five
])
def test_input_gradient_of_a_large_stride_takes_few_launches(gpu, xs, ws, stride, dil, launches):
    gd = gpu.DenseConvDims(xs, ws, stride=stride, dilation=dil)
    rng = np.random.default_rng(stable_seed("launches", xs, ws))
    dy, w = (dev(gpu, rng.normal(size=s).astype(np.float32), "f32") for s in (gd.y_shape, ws))
    count = kernels_of(gpu, lambda: gpu.conv_data_grad(dy, w, gd))
    assert count["conv_dgrad_kernel<f32>"] == launches, count


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("xs,ws", [((9, 7, 5, 3), (3, 3, 5, 12)), ((8, 8, 16, 2), (3, 3, 16, 12))])
def test_kept_copy_alone(gpu, dtype, xs, ws):
    """xt_keep is the unpadded channel-contiguous copy whatever the channel count, and the pullback takes it in place of x."""
    rng = np.random.default_rng(stable_seed("kept", xs))
    gd, od = gpu.DenseConvDims(xs, ws, padding=1), O.ConvDims(xs, ws, padding=1)
    x, w, dy = host_inputs(dtype, rng.normal(size=xs), rng.normal(size=ws), rng.normal(size=od.y_shape()))
    dx_, dw_, ddy = (dev(gpu, a, dtype) for a in (x, w, dy))
    y, kept, gw = gpu.DeviceArray(gd.y_shape, dtype), gpu.DeviceArray(xs, dtype), gpu.DeviceArray(ws, dtype)
    s = gpu.current_stream()
    gpu._lib.call("luxhip_conv_fwd", s, y.code, 0, C.byref(gd._c), dx_.ptr, dw_.ptr, None, y.ptr, None, kept.ptr)
    np.testing.assert_array_equal(kept.to_numpy().ravel(order="F").reshape((xs[2], xs[0], xs[1], xs[3]), order="F"),
                                  np.transpose(dx_.to_numpy(), (2, 0, 1, 3)))
    gpu._lib.call("luxhip_fused_conv_bwd", s, y.code, 0, C.byref(gd._c), ddy.ptr, y.ptr, None, None, dw_.ptr, None, gw.ptr, None, None, kept.ptr)
    assert_close(gw.to_numpy(), O.conv_filter_grad(f64(x), f64(dy), od), dtype, f"{dtype} dw from the kept copy")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_whole_tap_kernels_at_small_sizes(gpu, dtype):
    """conv_tile 42 takes the whole-tap kernels where the automatic choice prefers conv_any.h."""
    gpu.set_option("conv_tile", 42)
    try:
        for xs, ws, stride, pad, dil, groups, flip in [((13, 11, 64, 3), (3, 2, 32, 64), (2, 1), (1, 0, 2, 1), (1, 2), 2, True),
                                                       ((8, 8, 32, 5), (3, 3, 32, 320), 1, 1, 1, 1, False)]:
            rng = np.random.default_rng(stable_seed("tap", xs))
            kw = dict(stride=stride, padding=pad, dilation=dil, groups=groups, flipkernel=flip)
            gd, od = gpu.DenseConvDims(xs, ws, **kw), O.ConvDims(xs, ws, **kw)
            x, w, dy = host_inputs(dtype, rng.normal(size=xs), rng.normal(size=ws), rng.normal(size=od.y_shape()))
            assert_close(gpu.conv(dev(gpu, x, dtype), dev(gpu, w, dtype), gd).to_numpy(), O.conv(f64(x), f64(w), od), dtype, "tap y")
            assert_close(gpu.conv_data_grad(dev(gpu, dy, dtype), dev(gpu, w, dtype), gd).to_numpy(), O.conv_data_grad(f64(dy), f64(w), od),
                         dtype, "tap dx")
    finally:
        gpu.set_option("conv_tile", 0)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("xs,ws,stride,pad,groups", [
    ((37, 29, 3, 2), (7, 7, 3, 20), 2, 3, 1),                # one residue column block
    ((9, 11, 6, 2), (5, 4, 2, 9), 3, (2, 1, 0, 2), 3),       # nine residues, groups
    ((9, 8, 3, 1), (5, 5, 3, 640), 2, 2, 1),                 # contraction cut into slices
    ((21, 20, 12, 2), (7, 7, 12, 16), 2, 3, 1),              # residues over more than one column tile
])
def test_nonfinite_cotangent_reaches_its_window_only(gpu, dtype, xs, ws, stride, pad, groups):
    """An infinite and a NaN cotangent: the input gradient is non-finite exactly where the filter's window sees them."""
    rng = np.random.default_rng(stable_seed("nonfinite", xs))
    kw = dict(stride=stride, padding=pad, groups=groups)
    gd, od = gpu.DenseConvDims(xs, ws, **kw), O.ConvDims(xs, ws, **kw)
    w, dy = host_inputs(dtype, rng.normal(size=ws) / np.sqrt(ws[0] * ws[1] * ws[3]), rng.normal(size=od.y_shape()))
    bad = {(1, 2, 0, 0): np.inf, (od.y_shape()[0] - 1, 1, ws[3] - 1, xs[3] - 1): np.nan}
    dy, reach = dy.copy(), np.zeros(od.y_shape())
    for at in bad:
        dy[at], reach[at] = 0, 1
    want, seen = O.conv_data_grad(f64(dy), f64(w), od), O.conv_data_grad(reach, np.ones(ws), od) > 0
    for at, value in bad.items():
        dy[at] = value
    got = f64(gpu.conv_data_grad(dev(gpu, dy, dtype), dev(gpu, w, dtype), gd).to_numpy())
    np.testing.assert_array_equal(np.isfinite(got), ~seen)
    assert_close(np.where(seen, 0.0, got), np.where(seen, 0.0, want), dtype, f"{dtype} finite part of dx")


@pytest.mark.parametrize("dtype,stride", [("f32", 1), ("f32", 2), ("bf16", 1), ("bf16", 2)])
def test_depthwise_copies_take_no_more_than_the_tensor(gpu, dtype, stride):
    """A depthwise layer above 64 MiB: its padded copies are made for a few groups at a time (channels stay apart, so a layer of
    the same images with fewer channels gives each of them the same bits)."""
    xs, ws = (280, 250, 96, 5) if dtype == "bf16" else (280, 250, 50, 5), (3, 3, 1, 96 if dtype == "bf16" else 50)
    kw = dict(stride=stride, padding=1)
    gd = gpu.DenseConvDims(xs, ws, groups=xs[2], **kw)
    rng = np.random.default_rng(stable_seed("depthwise", dtype))
    ints = lambda *s: rng.integers(-2, 3, size=s).astype(np.float32)
    x, w, dy = ints(*xs), ints(*ws), ints(*gd.y_shape)
    y, back = gpu.pullback(gpu.fused_conv_bias_activation, "identity", dev(gpu, w, dtype), dev(gpu, x, dtype), None, gd)
    gw, gx, _ = back(dev(gpu, dy, dtype))
    y, gw, gx = (a.to_numpy() for a in (y, gw, gx))
    for c in (0, 11, 12, 49, xs[2] - 1):                     # first and last channels of the copies among them
        od = O.ConvDims(xs[:2] + (1, xs[3]), (3, 3, 1, 1), **kw)
        xc, wc, dc = f64(x[:, :, c:c + 1]), f64(w[:, :, :, c:c + 1]), f64(dy[:, :, c:c + 1])
        np.testing.assert_array_equal(y[:, :, c:c + 1], O.conv(xc, wc, od))
        np.testing.assert_array_equal(gx[:, :, c:c + 1], O.conv_data_grad(dc, wc, od))
        want = O.conv_filter_grad(xc, dc, od)
        np.testing.assert_array_equal(gw[:, :, :, c:c + 1], want if dtype == "f32" else O.round_to_bf16(want.astype(np.float32)))


def test_groups_share_their_launches(gpu):
    xs, ws = (12, 11, 24, 2), (3, 3, 2, 36)
    gd = gpu.DenseConvDims(xs, ws, padding=1, groups=12)
    rng = np.random.default_rng(3)
    x, w, dy = (dev(gpu, rng.normal(size=s).astype(np.float32), "f32") for s in (xs, ws, gd.y_shape))
    count = kernels_of(gpu, lambda: gpu.conv(x, w, gd))
    assert count == {"whcn_to_cwhn_kernel": 1, "conv_fprop_kernel<f32>": 1}, count
    count = kernels_of(gpu, lambda: gpu.conv_data_grad(dy, w, gd))
    assert count == {"whcn_to_cwhn_kernel": 1, "conv_dgrad_kernel<f32>": 1}, count
