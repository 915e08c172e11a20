"""The native part of the host side (csrc/python_host.cpp) without a device: what the arrays say of themselves, and that calls convert, refuse
and report as the ctypes calls that stand behind them do."""
import ctypes as C
import gc
import weakref

import numpy as np
import pytest


def _borrowed(lux, shape, dtype="f32", ptr=1 << 40, base=None):
    return lux.DeviceArray(shape, dtype, ptr=ptr, base=base)


def test_array_attributes(lux):
    a = _borrowed(lux, [np.int64(3), 4.0, 5], "bf16", ptr=np.int64(1 << 41))
    assert a.shape == (3, 4, 5) and all(type(s) is int for s in a.shape)
    assert (a.size, a.ndim, a.itemsize, a.nbytes, a.code, a.ptr, a.dtype) == (60, 3, 2, 120, lux._lib.BF16, 1 << 41, "bf16")
    assert (_borrowed(lux, ()).size, _borrowed(lux, (7, 0, 3)).nbytes, _borrowed(lux, (6,), "u8").code) == (1, 0, -1)
    assert _borrowed(lux, (0, 1 << 62, 1 << 62)).size == 0
    assert repr(a) == f"DeviceArray(shape=(3, 4, 5), dtype=bf16, ptr=0x{1 << 41:x})"
    with pytest.raises(TypeError, match="unsupported dtype 'f64'"):
        _borrowed(lux, (3,), "f64")
    with pytest.raises(TypeError):
        _borrowed(lux, 3)
    with pytest.raises((TypeError, ValueError)):
        _borrowed(lux, ("x",))


def test_a_view_keeps_its_base(lux):
    class Owner:
        pass

    owner = Owner()
    gone = weakref.ref(owner)
    a = _borrowed(lux, (2, 6), base=owner)
    b = a.reshape(3, 4)
    assert b.shape == (3, 4) and b.ptr == a.ptr
    del owner, a
    gc.collect()
    assert gone() is not None
    del b
    gc.collect()
    assert gone() is None
    loop = Owner()
    loop.a = _borrowed(lux, (1,), base=loop)                     # a cycle through an array is collected
    gone = weakref.ref(loop)
    del loop
    gc.collect()
    assert gone() is None


def _args(lux, **at):
    """luxhip_dropout_mask(stream, dtype, n, p, invp, mask)"""
    v = dict(stream=C.c_void_p(None), dtype=0, n=4, p=0.5, invp=2.0, mask=1 << 40)
    v.update(at)
    return list(v.values())


def test_calls_refuse_what_ctypes_refuses(lux):
    for bad in (dict(n="4"), dict(n=4.0), dict(p="x"), dict(mask=1.5), dict(stream=np.zeros(1))):
        with pytest.raises(C.ArgumentError):
            lux._lib._ctypes_call("luxhip_dropout_mask", *_args(lux, **bad))
        with pytest.raises(C.ArgumentError):
            lux._lib.call("luxhip_dropout_mask", *_args(lux, **bad))
    with pytest.raises(TypeError):
        lux._lib.call("luxhip_dropout_mask", *_args(lux)[:-1])
    with pytest.raises(AttributeError):
        lux._lib.call("luxhip_no_such_entry", 1)
    for wrong in ((C.c_int32 * 4)(1, 2, 3, 4), (C.c_double * 2)(1, 2), 1 << 40):
        with pytest.raises(C.ArgumentError):
            lux._lib.call("luxhip_dropout_mul", None, 0, 2, wrong, wrong, 1 << 40, 1 << 40, 1 << 40)


@pytest.mark.gpu
def test_calls_report_the_librarys_status(gpu):
    with pytest.raises(gpu.LuxHipError) as want:
        gpu._lib._ctypes_call("luxhip_dropout_mask", *_args(gpu, n=-1))
    with pytest.raises(gpu.LuxHipError) as got:
        gpu._lib.call("luxhip_dropout_mask", *_args(gpu, n=-1))
    assert (got.value.status, str(got.value)) == (want.value.status, str(want.value))
    with pytest.raises(gpu.LuxHipError, match="failed"):
        gpu.DeviceArray((1 << 31, 1 << 31, 1 << 31))
    a = gpu.DeviceArray((5,))
    dims = (C.c_int64 * 1)(5)
    x, m = gpu.DeviceArray.from_numpy(np.arange(5)), gpu.DeviceArray.from_numpy(np.full(5, 2.0))
    gpu._lib.call("luxhip_dropout_mul", gpu.current_stream(), 0, 1, dims, dims, x.ptr, m.ptr, a.ptr)
    np.testing.assert_array_equal(a.to_numpy(), 2.0 * np.arange(5))
