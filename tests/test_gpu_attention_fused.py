"""The fused attention kernels (bf16, no mask array, bias or fdrop) at the edges of their tiles: 128 columns per
workgroup, 32 per wave, 64 (32) rows per tile, 32 features per accumulator tile, eight heads per turn over the XCDs."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, stable_seed

pytestmark = pytest.mark.gpu

CASES = [
    # E, Ev, H, G, L, S, B, token_dim, causal
    (8, 8, 1, 1, 1, 1, 1, 3, False), (32, 32, 2, 2, 31, 33, 1, 3, False), (40, 16, 2, 1, 65, 63, 2, 3, True),
    (64, 64, 8, 2, 129, 127, 1, 3, False), (64, 72, 3, 3, 257, 193, 1, 2, True), (96, 96, 4, 4, 128, 256, 2, 3, True),
    (80, 48, 2, 2, 160, 100, 1, 3, True), (128, 128, 8, 8, 256, 256, 1, 2, False), (128, 128, 2, 1, 384, 385, 1, 3, True),
    (128, 104, 16, 8, 97, 300, 1, 3, False), (16, 128, 8, 1, 200, 130, 2, 3, True), (64, 64, 2, 2, 33, 8, 1, 3, False),
    (96, 80, 2, 2, 72, 200, 2, 3, False), (128, 128, 3, 3, 161, 136, 1, 3, True), (72, 64, 1, 1, 40, 16, 3, 2, True),
]


def test_few_long_heads_stay_on_the_step_by_step_products(gpu):
    """2 heads of 1024 tokens are 16 workgroups of the fused kernels; the same tokens in 16 heads are 128."""
    for heads, fused in ((2, False), (16, True)):
        d = dev(gpu, np.zeros((64, heads, 1024, 1), np.float32), "bf16")
        names = kernels_of(gpu, lambda: gpu.scaled_dot_product_attention(d, d, d))
        assert ("attn_fwd_kernel" in names) == fused


ROUTES = [
    # E, Ev, H, G, L, S, B, causal, forward fused, pullback fused: few queries on many keys, the reverse, and either side of both lines
    (64, 64, 32, 32, 1, 4096, 1, False, False, False), (128, 128, 8, 2, 16, 2048, 1, False, False, False), (64, 64, 4, 4, 8, 1024, 1, False, False, True),
    (128, 128, 1, 1, 1024, 16, 2, False, True, False), (128, 64, 4, 2, 1024, 128, 1, True, True, False), (96, 96, 2, 2, 512, 512, 1, True, True, False),
    (64, 64, 2, 2, 1, 512, 1, False, True, True), (64, 64, 2, 1, 33, 1031, 1, False, True, True), (64, 64, 8, 8, 64, 2048, 1, True, True, True),
    # ragged tokens: many queries on few keys, the reverse, and either side of the pullback's line
    (96, 96, 2, 2, 2047, 47, 1, False, True, False), (128, 128, 4, 2, 1605, 52, 1, True, True, False), (64, 64, 1, 1, 635, 3072, 1, False, False, False),
    (64, 64, 2, 2, 1023, 130, 1, False, True, False), (64, 64, 12, 12, 256, 111, 7, False, True, True),
]


@pytest.mark.parametrize("case", range(len(ROUTES)))
def test_forward_and_pullback_choose_their_kernels_apart(gpu, case):
    """Either direction takes the fused kernels where their workgroups fill the chip or their walks are short, and reads what either
    forward pass left.  One query against 2048 keys of 32 heads: the products 38 us, the fused forward kernel 64."""
    E, Ev, H, G, L, S, B, causal, fwd, bwd = ROUTES[case]
    rng = np.random.default_rng(stable_seed("attn-routes", case))
    q, k, v, d_out = host_inputs("bf16", *(rng.normal(size=(e, h, t, B)) for e, h, t in ((E, H, L), (E, G, S), (Ev, G, S), (Ev, H, L))))
    d = lambda a: dev(gpu, a, "bf16")
    q_, k_, v_, d_ = d(q), d(k), d(v), d(d_out)
    keep = []
    names = kernels_of(gpu, lambda: keep.append(gpu.pullback(gpu.scaled_dot_product_attention, q_, k_, v_, 1, 3, None, None, True if causal else None)))
    assert ("attn_fwd_kernel" in names) == fwd, names
    (out, w), back = keep[0]
    names = kernels_of(gpu, lambda: keep.append(back(d_)))
    assert ("attn_dkv_kernel" in names) == ("attn_dq_kernel" in names) == bwd, names
    stored = f64(w.to_numpy())
    assert_close(stored, O.scaled_dot_product_attention(f64(q), f64(k), f64(v), 3, None, None, True if causal else None)[1], "bf16", "weights")
    want = O.scaled_dot_product_attention(f64(q), f64(k), f64(v), 3, None, None, True if causal else None, weights=stored)[0]
    assert_close(out.to_numpy(), want, "bf16", "out")
    want = O.scaled_dot_product_attention_pullback(f64(q), f64(k), f64(v), f64(d_out), 3, None, None, True if causal else None,
                                                   weights=stored, stored=lambda a: f64(O.round_to_bf16(np.asarray(a, np.float32))))
    for g, x, name in zip(keep[1], want, ("dq", "dk", "dv")):
        assert_close(g.to_numpy(), x, "bf16", name, scale=1e-3)


@pytest.mark.parametrize("case", range(len(CASES)))
def test_edges_of_the_tiles(gpu, case):
    E, Ev, H, G, L, S, B, token_dim, causal = CASES[case]
    rng = np.random.default_rng(stable_seed("attn-fused", case))
    shape = (lambda e, h, t: ((e, h, t) if token_dim == 3 else (e, t, h)) + (B,))
    q, k, v = host_inputs("bf16", rng.normal(size=shape(E, H, L)), rng.normal(size=shape(E, G, S)), rng.normal(size=shape(Ev, G, S)))
    dq_, dk_, dv_ = (dev(gpu, a, "bf16") for a in (q, k, v))
    # memory that no kernel wrote would show up as NaN
    poison = [dev(gpu, np.full(n, np.nan, np.float32), "bf16") for n in (S * L * H * B, 2 * Ev * H * L * B, q.size, k.size * (H // G), v.size * (H // G))]
    del poison
    run = lambda: gpu.pullback(gpu.scaled_dot_product_attention, dq_, dk_, dv_, 1, token_dim, None, None, True if causal else None)
    (out, w), back = run()
    wout, ww = O.scaled_dot_product_attention(f64(q), f64(k), f64(v), token_dim, None, None, True if causal else None)
    assert_close(w.to_numpy(), ww, "bf16", "weights")
    stored = f64(w.to_numpy())
    if causal:
        assert not stored[np.arange(S)[:, None] > np.arange(L)[None, :]].any()
    wout, _ = O.scaled_dot_product_attention(f64(q), f64(k), f64(v), token_dim, None, None, True if causal else None, weights=stored)
    assert_close(out.to_numpy(), wout, "bf16", "out")
    (d_out,) = host_inputs("bf16", rng.normal(size=wout.shape))
    got = back(dev(gpu, d_out, "bf16"))
    want = O.scaled_dot_product_attention_pullback(f64(q), f64(k), f64(v), f64(d_out), token_dim, None, None, True if causal else None,
                                                   weights=stored, stored=lambda a: f64(O.round_to_bf16(np.asarray(a, np.float32))))
    # dlogits are differences: where the softmax is saturated they are far below the terms they are made of
    for g, x, name in zip(got, want, ("dq", "dk", "dv")):
        assert_close(g.to_numpy(), x, "bf16", name, scale=1e-3)
    names = kernels_of(gpu, lambda: run()[1](dev(gpu, d_out, "bf16")))
    assert {"attn_fwd_kernel", "attn_dkv_kernel", "attn_dq_kernel"} <= set(names)


def test_an_unaligned_cotangent_takes_the_step_by_step_pullback(gpu):
    """Both pullbacks start from the same stored weights and give the same gradients up to the order of their sums."""
    E, H, L, B = 64, 2, 130, 2
    rng = np.random.default_rng(stable_seed("attn-fused-unaligned"))
    q, k, v, d = host_inputs("bf16", *(rng.normal(size=(E, H, L, B)) for _ in range(4)))
    _, back = gpu.pullback(gpu.scaled_dot_product_attention, dev(gpu, q, "bf16"), dev(gpu, k, "bf16"), dev(gpu, v, "bf16"), 1, 3, None, None, True)
    a = back(dev(gpu, d, "bf16"))
    base = dev(gpu, np.concatenate([np.zeros(1, np.float32), d.ravel(order="F")]), "bf16")
    off = gpu.DeviceArray(d.shape, "bf16", ptr=base.ptr + 2, base=base)
    names = kernels_of(gpu, lambda: back(off))
    assert "attn_dq_kernel" not in names
    for x, y in zip(a, back(off)):
        assert_close(x.to_numpy(), f64(y.to_numpy()), "bf16", "gradients", rel=2.0 ** -7)      # one unit in the last place of either


def test_columns_with_infinite_logits(gpu):
    """A query with an infinite logit: its whole column of weights is NaN, masked positions included, and so is its output;
    the columns beside it are not touched."""
    E, H, L = 64, 2, 200
    rng = np.random.default_rng(stable_seed("attn-fused-inf"))
    q, k, v = host_inputs("bf16", *(rng.normal(size=(E, H, L, 1)) for _ in range(3)))
    q[:, 1, 70, 0] = 3e38
    k[:, 1, 3, 0] = 3e38
    d = lambda a: dev(gpu, a, "bf16")
    y, w = gpu.scaled_dot_product_attention(d(q), d(k), d(v), 1, 3, None, None, True)
    y, w = y.to_numpy(), w.to_numpy()
    assert np.isnan(w[:, 70, 1, 0]).all() and np.isnan(y[:, 1, 70, 0]).all()
    assert np.isfinite(w[:, :, 0]).all() and np.isfinite(w[:, :3, 1]).all() and np.isfinite(y[:, 0]).all() and np.isfinite(y[:, 1, :3]).all()


@pytest.mark.parametrize("scale", [1.0, -1.0, 1e3, 1e-3])
def test_weights_of_large_logits_add_up_to_one(gpu, scale):
    """Equal keys share a column equally, whatever the size of their logits, and so do the largest ones of a column.  The weights are
    fp32 quotients rounded to bf16 (2^-9 of the value); bf16 operands of few bits make the logits themselves exact."""
    E, H, L, S = 64, 16, 130, 100
    rng = np.random.default_rng(stable_seed("attn-fused-large", scale))
    q = rng.integers(1, 9, size=(E, H, L, 1)) * 64.0                 # products of 2^15 and more, sums of up to 2^24: exact in fp32
    k = np.repeat(rng.integers(1, 9, size=(E, H, 1, 1)) * 64.0, S, axis=2)
    k[:, :, 60:] = -k[:, :, 60:] if scale > 0 else k[:, :, 60:]     # a scale below 0: all keys equal still
    v = rng.normal(size=(E, H, S, 1))
    d = lambda a: dev(gpu, a.astype(np.float32), "bf16")
    run = lambda: gpu.scaled_dot_product_attention(d(q), d(k), d(v), 1, 3, 1.0 / scale)
    assert "attn_fwd_kernel" in kernels_of(gpu, run)
    n = 60 if scale > 0 else S
    want = np.zeros((S, L, H, 1))
    want[:n] = 1.0 / n
    np.testing.assert_allclose(run()[1].to_numpy(), want, rtol=2.0 ** -8, atol=0)


@pytest.mark.parametrize("scale", [-3.0, np.inf])
def test_negative_and_zero_scale(gpu, scale):
    """A negative divisor turns the softmax round (the kernels flip q's sign), an infinite one makes all logits equal, masked ones still
    -inf."""
    E, H, L, S = 64, 2, 97, 130
    rng = np.random.default_rng(stable_seed("attn-fused-scale", scale))
    q, k, v, d_out = host_inputs("bf16", *(rng.normal(size=(E, H, t, 1)) for t in (L, S, S, L)))
    (out, w), back = gpu.pullback(gpu.scaled_dot_product_attention, *(dev(gpu, a, "bf16") for a in (q, k, v)), 1, 3, scale, None, True)
    stored = f64(w.to_numpy())
    assert_close(stored, O.scaled_dot_product_attention(f64(q), f64(k), f64(v), 3, scale, None, True)[1], "bf16", "weights")
    assert_close(out.to_numpy(), O.scaled_dot_product_attention(f64(q), f64(k), f64(v), 3, scale, None, True, weights=stored)[0], "bf16", "out")
    grads = []
    assert "attn_dq_kernel" in kernels_of(gpu, lambda: grads.extend(back(dev(gpu, d_out, "bf16"))))
    want = O.scaled_dot_product_attention_pullback(f64(q), f64(k), f64(v), f64(d_out), 3, scale, None, True, weights=stored,
                                                   stored=lambda a: f64(O.round_to_bf16(np.asarray(a, np.float32))))
    for g, x, name in zip(grads, want, ("dq", "dk", "dv")):
        assert_close(g.to_numpy(), x, "bf16", name, scale=1e-3)


@pytest.mark.parametrize("E,size", [(64, 1.0), (96, 1.0), (64, 0.25)])
def test_weights_carry_the_errors_of_fp32_and_no_more(gpu, E, size):
    """How many weights round to another bf16 number than their exact values: an error of r (relative) moves a value of mantissa f in
    [1, 2) past a boundary with probability r f 2^7, 185 r in the mean.  Exponents up to 8 are off by 2^-22 at most, 9.5e-8 of a weight in the root
    mean square; exp2, the reciprocal of the sum, the sum and the product are half a unit in the last place each (3.4e-8).  1.2e-7
    together, 9.5e-8 in the mean of the absolute values: 1.8e-5 of the weights; half as many again are allowed."""
    H, T = 12, 745
    rng = np.random.default_rng(stable_seed("attn-fused-fp32", E, size))
    q, k, v = host_inputs("bf16", *(rng.normal(size=(E, H, T, 1)) * s for s in (size, 1, 1)))
    d = lambda a: dev(gpu, a, "bf16")
    out = []
    assert "attn_fwd_kernel" in kernels_of(gpu, lambda: out.append(gpu.scaled_dot_product_attention(d(q), d(k), d(v))))
    got = f64(out[0][1].to_numpy())[:, :, :, 0]                                     # keys, queries, heads
    off = 0
    for h in range(H):
        z = f64(k[:, h, :, 0]).T @ f64(q[:, h, :, 0]) / np.sqrt(E)
        w = np.exp(z - z.max(axis=0))
        m, e = np.frexp(w / w.sum(axis=0))
        off += np.count_nonzero(got[:, :, h] != np.ldexp(np.rint(m * 256), e - 8))
    assert off <= 1.5 * 1.8e-5 * H * T * T


@pytest.mark.parametrize("causal", [False, True])
def test_columns_of_every_size_beside_each_other(gpu, causal):
    """Logits from 2^-6 to 2^24 in the lanes of one wave, whose maxima grow from tile to tile or lie in the first or the last one: sums change their
    offsets, some columns' because of others'.  Operands of few bits make the logits exact in fp32."""
    E, H, L, S = 64, 16, 130, 200
    rng = np.random.default_rng(stable_seed("attn-fused-offsets", causal))
    q = rng.integers(-2, 3, size=(E, H, L, 1)) * 2.0 ** rng.integers(-6, 21, size=(1, H, L, 1))
    k = rng.integers(-3, 4, size=(E, H, S, 1)).astype(np.float64)
    ramp = 1.0 + np.arange(S) // 20                                  # up to 10: four bits
    for h in range(H):
        k[:, h, :, 0] = k[:, h, [0], 0] * (ramp, ramp[::-1], -ramp, 1.0 + 0 * ramp)[h % 4] if h % 8 < 4 else k[:, h, :, 0]
    d = lambda a: dev(gpu, a.astype(np.float32), "bf16")
    out = []
    assert "attn_fwd_kernel" in kernels_of(gpu, lambda: out.append(gpu.scaled_dot_product_attention(d(q), d(k), d(k), 1, 3, None, None, True if causal else None)))
    got = out[0][1].to_numpy()
    for h in range(H):
        z = k[:, h, :, 0].T @ q[:, h, :, 0] / 8.0
        if causal:
            z = np.where(np.arange(S)[:, None] <= np.arange(L)[None, :], z, -np.inf)
        w = np.exp(z - z.max(axis=0))
        # exponents of 150 at most count, rounded once: 2^-17 of a weight
        np.testing.assert_allclose(got[:, :, h, 0], w / w.sum(axis=0), rtol=2.0 ** -8 + 2.0 ** -16, atol=1e-36)


@pytest.mark.parametrize("E", [24, 96, 128])
def test_gradients_that_cancel_are_zero(gpu, E):
    """Equal values for all keys: the cotangents of the weights are all their mean, so dq and dk are 0.  Small integers make every sum exact, and a
    weight of one or of a power of two, so they are exactly 0 where nothing else rounds (the scale is no power of two)."""
    H, L, S = 4, 300, 64
    rng = np.random.default_rng(stable_seed("attn-fused-cancel", E))
    q, v, d_out = (rng.integers(-4, 5, size=(E, H, t, 1)).astype(np.float64) for t in (L, 1, L))
    k = np.ones((E, H, S, 1))                                        # equal logits: 64 weights of 1 / 64
    d = lambda a: dev(gpu, a.astype(np.float32), "bf16")
    _, back = gpu.pullback(gpu.scaled_dot_product_attention, d(q), d(k), d(np.repeat(v, S, axis=2)), 1, 3)
    grads = []
    assert "attn_dq_kernel" in kernels_of(gpu, lambda: grads.extend(back(d(d_out))))
    assert not grads[0].to_numpy().any() and not grads[1].to_numpy().any()
    np.testing.assert_allclose(grads[2].to_numpy(), np.broadcast_to(d_out.sum(axis=2, keepdims=True) / S, (E, H, S, 1)), rtol=2.0 ** -8)
