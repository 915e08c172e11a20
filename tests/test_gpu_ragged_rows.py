"""Normalisations over rows that are no multiple of a 16-byte vector (RowVec in common.h: the last vector of a row is moved
back and leaves its repeated elements out) against the fp64 oracle, at the edges: rows of exactly one vector, one element more,
one vector less one element, several vectors and a bit; whole waves and partial ones; cached and streaming kernels."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, rms, stable_seed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "swish"])
def test_groupnorm(gpu, dtype, act):
    rng = np.random.default_rng(stable_seed("ragged gn", dtype, act))
    eps = 1e-5 if dtype == "f32" else 1e-3
    for shape, groups in [((3, 3, 8, 3), 4), ((9, 1, 6, 2), 3), ((5, 5, 12, 7), 2), ((35, 35, 8, 2), 4), ((17, 4, 130, 2), 1), ((131, 127, 4, 2), 2)]:
        C = shape[-2]
        x, g, b, delta = host_inputs(dtype, rng.normal(size=shape) + 0.5, rng.uniform(0.8, 1.2, C), 0.05 * rng.normal(size=C), rng.normal(size=shape))
        y, back = gpu.pullback(gpu.groupnorm, dev(gpu, x, dtype), dev(gpu, g, dtype), dev(gpu, b, dtype), groups, act, eps)
        tag = f"{dtype} {act} {shape} G={groups}"
        assert_close(y.to_numpy(), O.groupnorm(f64(x), f64(g), f64(b), groups, act, eps), dtype, tag + " y")
        got = back(dev(gpu, delta, dtype))
        want = O.groupnorm_pullback(f64(x), f64(g), f64(b), groups, act, eps, f64(delta))
        for name, a, w in zip(("dx", "dgamma", "dbeta"), got, want):
            assert_close(a.to_numpy(), w, dtype, f"{tag} {name}", scale=rms(delta) * (1.0 if name == "dx" else np.sqrt(shape[0] * shape[1] * shape[3])))
        again = back(dev(gpu, delta, dtype))
        for a, c in zip(got, again):
            np.testing.assert_array_equal(a.to_numpy(), c.to_numpy())


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "gelu"])
def test_layernorm(gpu, dtype, act):
    rng = np.random.default_rng(stable_seed("ragged ln", dtype, act))
    eps = 1e-5 if dtype == "f32" else 1e-3
    for L, R in [(5, 70), (9, 3), (67, 130), (255, 64), (1023, 101), (1025, 66), (2051, 65), (4099, 9), (8211, 3)]:
        x, g, b, delta = host_inputs(dtype, rng.normal(size=(L, R)) + 0.5, rng.uniform(0.5, 1.5, (L, 1)), 0.1 * rng.normal(size=(L, 1)), rng.normal(size=(L, R)))
        y, back = gpu.pullback(gpu.layernorm, dev(gpu, x, dtype), dev(gpu, g, dtype), dev(gpu, b, dtype), act, (1,), eps)
        tag = f"{dtype} {act} {L}x{R}"
        assert_close(y.to_numpy(), O.layernorm(f64(x), f64(g), f64(b), act, (0,), eps), dtype, tag + " y")
        got = back(dev(gpu, delta, dtype))
        want = O.layernorm_pullback(f64(x), f64(g), f64(b), act, (0,), eps, f64(delta))
        sd = np.sqrt(f64(x).var(axis=0).min() + eps)
        for name, a, w in zip(("dx", "dgamma", "dbeta"), got, want):
            assert_close(a.to_numpy(), w, dtype, f"{tag} {name}", scale=rms(delta) * (1.5 / sd if name == "dx" else np.sqrt(R)))


@pytest.mark.parametrize("dtype,L,R,fused", [
    ("f32", 67, 2048, True), ("f32", 67, 2049, False), ("f32", 237, 2049, True), ("bf16", 406, 2049, False), ("bf16", 409, 2049, True),
    ("bf16", 2293, 767, True), ("bf16", 2293, 768, False),
])
def test_layernorm_on_either_side_of_the_one_pass_pullback(gpu, dtype, L, R, fused):
    rng = np.random.default_rng(stable_seed("ln route", L, R))
    x, g, b, delta = host_inputs(dtype, rng.normal(size=(L, R)) + 0.5, rng.uniform(0.5, 1.5, (L, 1)), 0.1 * rng.normal(size=(L, 1)), rng.normal(size=(L, R)))
    _, back = gpu.pullback(gpu.layernorm, dev(gpu, x, dtype), dev(gpu, g, dtype), dev(gpu, b, dtype), "tanh", (1,), 1e-3)
    got, d = [], dev(gpu, delta, dtype)
    names = kernels_of(gpu, lambda: got.extend(back(d)))
    assert ("ln_bwd_fused_kernel" in names) == fused, names
    want = O.layernorm_pullback(f64(x), f64(g), f64(b), "tanh", (0,), 1e-3, f64(delta))
    sd = np.sqrt(f64(x).var(axis=0).min() + 1e-3)
    for name, a, w in zip(("dx", "dgamma", "dbeta"), got, want):
        assert_close(a.to_numpy(), w, dtype, f"{dtype} {L}x{R} {name}", scale=rms(delta) * (1.5 / sd if name == "dx" else np.sqrt(R)))
