"""Layers next to an image (few channels).  First layers (bf16, at most four channels, windows of 5 to 8 along w): the positions of a window in one row of the copied input
are one stage of the contraction.  Every channel count and window width, odd strides (8-byte alignment of the windows), padding
on either side alone, dilation along h, more rows and columns than a tile."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, stable_seed

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad, dilation, flip
    ((17, 15, 3, 3), (7, 7, 3, 20), 2, 3, 1, False), ((33, 20, 1, 2), (5, 5, 1, 33), 1, 2, 1, False),
    ((21, 19, 4, 2), (6, 3, 4, 65), 3, (4, 0, 0, 1), 1, True), ((40, 9, 2, 3), (8, 2, 2, 130), (2, 1), (0, 5, 1, 0), (1, 3), False),
    ((8, 8, 3, 1), (8, 1, 3, 3), 1, 0, 1, False), ((90, 61, 3, 2), (7, 7, 3, 64), 2, 3, 1, True), ((5, 300, 4, 1), (5, 5, 4, 16), 7, 2, 1, False),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_first_layer(gpu, case):
    xs, ws, stride, pad, dil, flip = CASES[case]
    rng = np.random.default_rng(stable_seed("conv_runs", case))
    kw = dict(stride=stride, padding=pad, dilation=dil, flipkernel=flip)
    gd, od = gpu.DenseConvDims(xs, ws, **kw), O.ConvDims(xs, ws, **kw)
    x, w, b, dy = host_inputs("bf16", rng.normal(size=xs), rng.normal(size=ws) / np.sqrt(ws[0] * ws[1] * ws[2]), rng.normal(size=ws[3]),
                              rng.normal(size=od.y_shape()))
    dx_, dw_, db_, ddy = (dev(gpu, a, "bf16") for a in (x, w, b, dy))
    y, back = gpu.pullback(gpu.fused_conv_bias_activation, "identity", dw_, dx_, db_, gd)
    assert_close(y.to_numpy(), O.conv(f64(x), f64(w), od) + f64(b)[None, None, :, None], "bf16", "y")
    gw, gx, _ = back(ddy)
    assert_close(gw.to_numpy(), O.conv_filter_grad(f64(x), f64(dy), od), "bf16", "dw")
    assert_close(gx.to_numpy(), O.conv_data_grad(f64(dy), f64(w), od), "bf16", "dx")
    np.testing.assert_array_equal(gpu.conv_filter_grad(dx_, ddy, gd).to_numpy(), gw.to_numpy())


@pytest.mark.parametrize("width", [5, 6, 7, 8])
def test_an_infinity_stays_inside_its_windows(gpu, width):
    """What lies behind a window in its run belongs to other windows: it must not meet the filter's padding."""
    xs, ws = (40, 12, 3, 2), (width, 3, 3, 24)
    rng = np.random.default_rng(stable_seed("conv_runs inf", width))
    x, w = host_inputs("bf16", rng.normal(size=xs), np.abs(rng.normal(size=ws)) + 0.1)
    cd = gpu.DenseConvDims(xs, ws, padding=1)
    clean = gpu.conv(dev(gpu, x, "bf16"), dev(gpu, w, "bf16"), cd).to_numpy()
    x[20, 6, 1, 1] = np.inf
    y = gpu.conv(dev(gpu, x, "bf16"), dev(gpu, w, "bf16"), cd).to_numpy()
    sees = np.zeros(y.shape, bool)
    sees[20 + 1 - (width - 1):20 + 2, 5:8, :, 1] = True
    assert (y[sees] == np.inf).all()
    np.testing.assert_array_equal(y[~sees], clean[~sees])
    dy = host_inputs("bf16", rng.normal(size=y.shape))[0]
    gw = gpu.conv_filter_grad(dev(gpu, x, "bf16"), dev(gpu, dy, "bf16"), cd).to_numpy()
    assert np.isfinite(gw[:, :, [0, 2]]).all() and not np.isfinite(gw[:, :, 1]).any()


FEW = [
    # x shape, w shape, stride, pad, flip: rows and residues that end inside a tile, 1 .. 4 taps, 16 .. 64 channels, up to 32 columns
    ((70, 36, 3, 8), (7, 7, 3, 64), 2, 3, False), ((65, 67, 2, 16), (5, 3, 2, 16), 2, 2, True), ((66, 34, 8, 20), (4, 4, 8, 48), 2, 1, False),
    ((97, 99, 1, 8), (9, 9, 1, 32), 3, 4, False), ((64, 40, 1, 33), (8, 6, 1, 64), (4, 2), (2, 2), False), ((34, 33, 3, 40), (2, 2, 3, 64), 2, 0, False),
]


@pytest.mark.parametrize("case", range(len(FEW)))
def test_input_gradient_with_few_channels(gpu, case):
    """All residues as columns, the cotangents of a tile in LDS (conv_few.h), and infinite cotangents: they reach the positions
    that see them and no others."""
    xs, ws, stride, pad, flip = FEW[case]
    rng = np.random.default_rng(stable_seed("conv_few", case))
    gd, od = (D(xs, ws, stride=stride, padding=pad, flipkernel=flip) for D in (gpu.DenseConvDims, O.ConvDims))
    w, dy = host_inputs("bf16", rng.normal(size=ws) / np.sqrt(ws[0] * ws[1] * ws[3]), rng.normal(size=od.y_shape()))
    want = O.conv_data_grad(f64(dy), f64(w), od)
    got = gpu.conv_data_grad(dev(gpu, dy, "bf16"), dev(gpu, w, "bf16"), gd).to_numpy()
    assert_close(got, want, "bf16", "dx")
    one = np.zeros(dy.shape)
    one[3, 5, 1, 2] = 1.0
    sees = O.conv_data_grad(one, np.ones(ws), od) != 0
    dy[3, 5, 1, 2] = np.inf
    bad = gpu.conv_data_grad(dev(gpu, dy, "bf16"), dev(gpu, np.abs(w) + 0.01, "bf16"), gd).to_numpy()
    assert (bad[sees] == np.inf).all() and np.isfinite(bad[~sees]).all()
