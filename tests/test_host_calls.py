"""The native part of the host side (csrc/python_host.cpp) without a device: what the arrays say of themselves, and that calls convert, refuse
and report as the ctypes calls that stand behind them do."""
import ctypes as C
import gc
import importlib.abc
import importlib.util
import os
import sys
import warnings
import weakref

import numpy as np
import pytest


def _package(name, refusal):
    """A copy of the package under `name`, in an interpreter whose import of the native part raises `refusal`."""
    class Refuse(importlib.abc.MetaPathFinder):
        def find_spec(self, fullname, path=None, target=None):
            if fullname == name + "._host":
                raise refusal

    here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lux.jl_amd")
    spec = importlib.util.spec_from_file_location(name, os.path.join(here, "__init__.py"), submodule_search_locations=[here])
    module, refuse = importlib.util.module_from_spec(spec), Refuse()
    sys.modules[name] = module
    sys.meta_path.insert(0, refuse)
    try:
        spec.loader.exec_module(module)
    finally:
        sys.meta_path.remove(refuse)
    return module


@pytest.fixture(scope="module")
def plain():
    """The package where its native part was not built: arrays and calls in Python and ctypes."""
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        return _package("lux_plain", ModuleNotFoundError("No module named 'lux_plain._host'", name="lux_plain._host"))


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


def test_shape_and_dtype_can_be_set(lux, plain):
    for a in (_borrowed(lux, (6, 4)), _borrowed(plain, (6, 4))):
        a.shape = (3, 8)
        assert (a.shape, a.size, a.ndim, a.nbytes) == ((3, 8), 24, 2, 96)
        a.shape, a.dtype = (24,), "bf16"
        assert (a.ndim, a.dtype, a.itemsize, a.nbytes, a.code) == (1, "bf16", 2, 48, lux._lib.BF16)


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


def test_an_argument_whose_class_raises(lux):
    class Odd:
        @property
        def __class__(self):
            raise RuntimeError("no class")

    for call in (lux._lib._ctypes_call, lux._lib.call):
        with pytest.raises(C.ArgumentError):
            call("luxhip_dropout_mul", None, 0, 2, Odd(), Odd(), 1 << 40, 1 << 40, 1 << 40)


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


def test_without_the_native_part(plain):
    assert plain._lib._host is None and plain._lib.call is plain._lib._ctypes_call
    test_array_attributes(plain)
    test_a_view_keeps_its_base(plain)
    test_calls_refuse_what_ctypes_refuses(plain)


def test_a_native_part_that_does_not_load_says_why():
    with pytest.warns(RuntimeWarning, match="undefined symbol: PyThing"):
        broken = _package("lux_broken", ImportError("_host.so: undefined symbol: PyThing"))
    assert broken.DeviceArray((2, 3), ptr=1 << 40).nbytes == 24


@pytest.mark.gpu
def test_operators_without_the_native_part(gpu, plain):
    plain.init(0)
    rng = np.random.default_rng(3)
    W, x, b, d = (rng.normal(size=s).astype(np.float32) for s in ((24, 16), (16, 9), (24,), (24, 9)))
    results = []
    for lux in (gpu, plain):
        y, back = lux.pullback(lux.fused_dense_bias_activation, "gelu", *(lux.DeviceArray.from_numpy(a) for a in (W, x, b)))
        g = lux.DeviceArray.from_numpy(np.ones((24, 1)))
        z, back2 = lux.pullback(lux.layernorm, y, g, g, "identity", (1,), 1e-5)              # its statistics are StatArrays
        results.append([a.to_numpy() for a in (y, z, *back(lux.DeviceArray.from_numpy(d)), *back2(lux.DeviceArray.from_numpy(d)))])
    for native, ctypes_only in zip(*results):
        np.testing.assert_array_equal(native, ctypes_only)
    with pytest.raises(plain.LuxHipError, match="failed"):
        plain.DeviceArray((1 << 30, 1 << 30))
