"""bias_activation over rows that are no multiple of a vector or not aligned to one, and its pullback from the operator's input."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, stable_seed

pytestmark = pytest.mark.gpu


def _shifted(gpu, a, dtype, by):
    """`a` on the device, `by` elements behind an aligned address."""
    flat = np.concatenate([np.zeros(by, np.float32), np.asarray(a, np.float32).ravel(order="F")])
    whole = dev(gpu, flat, dtype)
    return gpu.DeviceArray(a.shape, dtype, ptr=whole.ptr + by * whole.itemsize, base=whole)


# rows of one vector (8 or 4 elements) and a bit, the shortest rows of the channel layout, more than four vectors per thread of a channel,
# rows below a vector, whole rows at an odd address
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["identity", "tanh", "swish", "gelu"])
@pytest.mark.parametrize("I,C,N,shift", [(65, 3, 5, 0), (71, 2, 3, 1), (127, 1, 300, 0), (1369, 5, 12, 3), (33, 4, 6, 0), (3, 7, 5, 0), (64, 3, 2, 1), (9001, 1, 2, 0)])
def test_rows(gpu, dtype, act, I, C, N, shift):
    rng = np.random.default_rng(stable_seed("rows", dtype, act, I, C, N))
    x, b, d = host_inputs(dtype, rng.normal(size=(I, C, N)), rng.normal(size=C), rng.normal(size=(I, C, N)))
    dx = _shifted(gpu, x, dtype, shift)
    y, back = gpu.pullback(gpu.bias_activation, act, dx, dev(gpu, b, dtype))
    gx, gb = back(_shifted(gpu, d, dtype, shift))
    wy, wdx, wdb = O.bias_activation_pullback(act, f64(x), f64(b), f64(d))
    if dtype == "bf16":                       # y and x + bias are rounded in front of the derivative
        pre = f64(O.round_to_bf16((f64(x) + f64(b)[None, :, None]).astype(np.float32)))
        wdx = O.grad_activation(f64(d), f64(O.round_to_bf16(wy.astype(np.float32))), act, pre)
        wdb = wdx.sum((0, 2))
    assert_close(y.to_numpy(), wy, dtype, "y")
    assert_close(gx.to_numpy(), wdx, dtype, "dx")
    assert_close(gb.to_numpy().reshape(-1), wdb.reshape(-1), dtype, "db", scale=np.sqrt(I * N))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("act", ["swish", "gelu", "softplus", "relu"])
@pytest.mark.parametrize("I,C,N", [(64, 3, 5), (71, 3, 5), (1, 96, 40), (4, 6, 9), (5, 7, 3)])
def test_from_x_is_the_stored_pre_activation(gpu, dtype, act, I, C, N):
    rng = np.random.default_rng(stable_seed("from x", dtype, act, I, C, N))
    x, b, d = (dev(gpu, a, dtype) for a in host_inputs(dtype, rng.normal(size=(I, C, N)), rng.normal(size=C), rng.normal(size=(I, C, N))))
    code, aid, s = x.code, gpu._lib.ACT_IDS[act], gpu.current_stream()
    y, pre, got, want = (gpu.DeviceArray((I, C, N), dtype) for _ in range(4))
    db, wdb = gpu.DeviceArray((C,), dtype), gpu.DeviceArray((C,), dtype)
    gpu._lib.call("luxhip_bias_activation_fwd", s, code, aid, I, C, N, x.ptr, b.ptr, y.ptr, pre.ptr)
    gpu._lib.call("luxhip_bias_activation_bwd", s, code, aid, I, C, N, d.ptr, y.ptr, pre.ptr, want.ptr, wdb.ptr)
    gpu._lib.call("luxhip_bias_activation_bwd_from_x", s, code, aid, I, C, N, d.ptr, y.ptr, x.ptr, b.ptr, got.ptr, db.ptr)
    np.testing.assert_array_equal(got.to_numpy(), want.to_numpy())
    np.testing.assert_array_equal(db.to_numpy(), wdb.to_numpy())
    with pytest.raises(gpu.LuxHipError, match="dbias"):
        gpu._lib.call("luxhip_bias_activation_bwd_from_x", s, code, aid, I, C, N, d.ptr, y.ptr, x.ptr, b.ptr, got.ptr, None)
