// Native part of the Python host side: the arrays' allocation and release, and calls of the C ABI without ctypes' argument objects.
//
// A training step of a small layer is a handful of launches of a few microseconds each; ctypes took 0.6 us for an allocation, as much for its
// release and 2 to 4 us for a call of 17 to 22 arguments on the way to them.  Host time of a pass in training, with the library's entry points empty, on one
// core of the build machine: dense 43 -> 5.3 us, groupnorm 45 -> 5.4, batchnorm and activation 93 -> 10.3, convolution 66 -> 10.9; on the device's host a
// dense layer of 128 x 256 x 64 32.0 -> 23.5 us, groupnorm 11 x 11 x 12 x 2 27.1 -> 17.7.  The entry points are wrapped with the types that include/luxhip.h
// declares; what a wrapper does not convert itself (byref() and the like) it leaves to ctypes, which then also raises what ctypes raises.
// The addresses come from the library that _lib.load() has opened: importing this module opens nothing.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cstddef>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/luxhip.h"

namespace {

PyObject *g_load, *g_slow_call, *g_check;                        // _lib.load, its ctypes call and its status check
PyObject *g_void_p, *g_ctypes_array, *g_conv_dims;               // ctypes.c_void_p, ctypes.Array, _lib.ConvDimsStruct
PyObject *g_f32, *g_bf16, *g_u8;                                 // storage type names

enum class Conv { DONE, SLOW };

// The memory of a ctypes instance; int64: an array of 64-bit integers ("<l" or "<q")
bool ctypes_memory(PyObject* o, Py_ssize_t least, bool int64, void** out) {
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, int64 ? PyBUF_FORMAT : PyBUF_SIMPLE) != 0) {
        PyErr_Clear();
        return false;
    }
    const char* f = int64 ? b.format : nullptr;
    if (f != nullptr && *f == '<') ++f;
    const bool fits = b.len >= least && (!int64 || (b.itemsize == 8 && f != nullptr && (*f == 'l' || *f == 'q') && f[1] == 0));
    *out = b.buf;
    PyBuffer_Release(&b);                                        // the arguments outlive the call
    return fits;
}

template <class T>
Conv convert(PyObject* o, T* out) {
    if constexpr (std::is_integral_v<T>) {
        if (!PyLong_Check(o)) return Conv::SLOW;
        *out = (T)PyLong_AsUnsignedLongLongMask(o);              // as ctypes: no overflow check
        return Conv::DONE;
    } else if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_CheckExact(o)) return Conv::SLOW;
        *out = PyFloat_AS_DOUBLE(o);
        return Conv::DONE;
    } else if constexpr (std::is_same_v<T, void*> || std::is_same_v<T, const void*> || std::is_same_v<T, float*> || std::is_same_v<T, const float*>) {
        if (o == Py_None) {
            *out = nullptr;
        } else if (PyLong_Check(o)) {
            *out = (T)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
        } else if ((PyObject*)Py_TYPE(o) == g_void_p) {
            void* where;
            if (!ctypes_memory(o, sizeof(void*), false, &where)) return Conv::SLOW;
            *out = (T)*(void**)where;
        } else {
            return Conv::SLOW;
        }
        return Conv::DONE;
    } else if constexpr (std::is_same_v<T, const int64_t*> || std::is_same_v<T, const luxhip_conv_dims_t*>) {
        constexpr bool dims = std::is_same_v<T, const luxhip_conv_dims_t*>;
        void* where;
        const int is = dims ? (PyObject*)Py_TYPE(o) == g_conv_dims : PyObject_IsInstance(o, g_ctypes_array);
        if (is < 0) PyErr_Clear();                               // an error of the argument's own: ctypes says what it makes of it
        if (is != 1) return Conv::SLOW;
        if (!ctypes_memory(o, dims ? (Py_ssize_t)sizeof(luxhip_conv_dims_t) : 8, !dims, &where)) return Conv::SLOW;
        *out = (T)where;
        return Conv::DONE;
    } else {
        return Conv::SLOW;                                       // results through pointers, strings: not on an operator's path
    }
}

struct Entry {
    const char* name;
    Conv (*call)(void* address, PyObject* const* args, Py_ssize_t n, int* status);
    void* address;
};

template <class F>
struct Caller;
template <class... A>
struct Caller<int (*)(A...)> {
    template <size_t... I>
    static Conv run(void* address, PyObject* const* args, Py_ssize_t n, int* status, std::index_sequence<I...>) {
        if (n != (Py_ssize_t)sizeof...(A)) return Conv::SLOW;
        std::tuple<A...> v;
        if (!((convert(args[I], &std::get<I>(v)) == Conv::DONE) && ...)) return Conv::SLOW;
        Py_BEGIN_ALLOW_THREADS
        *status = ((int (*)(A...))address)(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        return Conv::DONE;
    }
    static Conv call(void* address, PyObject* const* args, Py_ssize_t n, int* status) {
        return run(address, args, n, status, std::index_sequence_for<A...>());
    }
};

#define ENTRY(f) {#f, &Caller<decltype(&f)>::call, nullptr}
Entry g_entries[] = {
    ENTRY(luxhip_malloc), ENTRY(luxhip_free),
    ENTRY(luxhip_bias_activation_fwd), ENTRY(luxhip_bias_activation_bwd), ENTRY(luxhip_bias_activation_bwd_from_x),
    ENTRY(luxhip_batchnorm_fwd), ENTRY(luxhip_batchnorm_bwd), ENTRY(luxhip_groupnorm_fwd), ENTRY(luxhip_groupnorm_bwd),
    ENTRY(luxhip_instancenorm_fwd), ENTRY(luxhip_instancenorm_running_stats), ENTRY(luxhip_layernorm_fwd), ENTRY(luxhip_layernorm_bwd),
    ENTRY(luxhip_attention_softmax_fwd), ENTRY(luxhip_attention_softmax_bwd), ENTRY(luxhip_attention_fwd), ENTRY(luxhip_attention_bwd),
    ENTRY(luxhip_attention_weights_pullback), ENTRY(luxhip_rand_uniform), ENTRY(luxhip_dropout_fwd), ENTRY(luxhip_dropout_mask),
    ENTRY(luxhip_dropout_mul), ENTRY(luxhip_alpha_dropout_fwd), ENTRY(luxhip_alpha_dropout_bwd), ENTRY(luxhip_matmul),
    ENTRY(luxhip_batched_matmul), ENTRY(luxhip_batched_matmul_strided), ENTRY(luxhip_batch_sum), ENTRY(luxhip_fused_dense_fwd),
    ENTRY(luxhip_fused_dense_bwd), ENTRY(luxhip_conv_fwd), ENTRY(luxhip_conv_bwd_data), ENTRY(luxhip_conv_bwd_filter),
    ENTRY(luxhip_fused_conv_bwd), ENTRY(luxhip_conv_depth_unfold), ENTRY(luxhip_conv_depth_fold), ENTRY(luxhip_swap_middle_dims),
    ENTRY(luxhip_convert), ENTRY(luxhip_permute_leading3),
};
PyObject* g_index;                                               // name -> position in g_entries
enum { MALLOC = 0, FREE = 1 };

bool loaded() {
    if (g_entries[MALLOC].address != nullptr) return true;
    PyObject* r = PyObject_CallNoArgs(g_load);                   // binds the addresses
    if (r == nullptr) return false;
    Py_DECREF(r);
    if (g_entries[MALLOC].address != nullptr) return true;
    PyErr_SetString(PyExc_ImportError, "the library's entry points are not bound");
    return false;
}

// bind(name, address): the entry point's address; names that have no wrapper are left to ctypes
PyObject* host_bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    PyObject* at = PyDict_GetItemString(g_index, name);
    if (at != nullptr) g_entries[PyLong_AsLong(at)].address = (void*)(uintptr_t)address;
    Py_RETURN_NONE;
}

// configure(load, slow_call, check, c_void_p, Array, ConvDimsStruct)
PyObject* host_configure(PyObject*, PyObject* args) {
    PyObject* v[6];
    if (!PyArg_ParseTuple(args, "OOOOOO", &v[0], &v[1], &v[2], &v[3], &v[4], &v[5])) return nullptr;
    PyObject** const to[6] = {&g_load, &g_slow_call, &g_check, &g_void_p, &g_ctypes_array, &g_conv_dims};
    for (int i = 0; i < 6; ++i) {
        Py_INCREF(v[i]);
        Py_XSETREF(*to[i], v[i]);
    }
    Py_RETURN_NONE;
}

PyObject* raise_status(int status) { return PyObject_CallFunction(g_check, "i", status); }

// call(name, *args): an entry point of the library; raises on a status other than 0
PyObject* host_call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n < 1 || !PyUnicode_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "call(name, *args)");
        return nullptr;
    }
    PyObject* at = PyDict_GetItemWithError(g_index, args[0]);
    if (at == nullptr && PyErr_Occurred()) return nullptr;
    if (at != nullptr) {
        if (!loaded()) return nullptr;
        const Entry& e = g_entries[PyLong_AsLong(at)];
        int status = 0;
        if (e.address != nullptr && e.call(e.address, args + 1, n - 1, &status) == Conv::DONE) {
            if (status == 0) Py_RETURN_NONE;
            return raise_status(status);
        }
    }
    return PyObject_Vectorcall(g_slow_call, args, (size_t)n, nullptr);
}

int device_alloc(size_t bytes, uintptr_t* out) {
    if (!loaded()) return -1;
    void* p = nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = ((int (*)(void**, size_t))g_entries[MALLOC].address)(&p, bytes);
    Py_END_ALLOW_THREADS
    *out = (uintptr_t)p;
    if (status == 0) return 0;
    PyObject* r = raise_status(status);
    Py_XDECREF(r);
    return -1;
}
void device_free(uintptr_t p) {
    if (p != 0 && g_entries[FREE].address != nullptr) (void)((int (*)(void*))g_entries[FREE].address)((void*)p);
}

// ------------------------------------------------------------------------------------------------ arrays
struct Array {
    PyObject_HEAD
    PyObject *shape, *dtype, *base;
    unsigned long long ptr;
    char owner;
};

// The product of a shape, or the largest number that an allocation can only refuse
bool shape_size(PyObject* shape, int64_t* out) {
    int64_t n = 1;
    bool over = false, zero = false;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); ++i) {
        int past = 0;
        const long long s = PyLong_AsLongLongAndOverflow(PyTuple_GET_ITEM(shape, i), &past);
        if (s == -1 && past == 0 && PyErr_Occurred()) return false;
        zero = zero || (s == 0 && past == 0);
        over = over || past != 0 || __builtin_mul_overflow(n, (int64_t)s, &n);
    }
    *out = zero ? 0 : over ? INT64_MAX / 8 : n;
    return true;
}

// A new reference to the shape as a tuple of ints
PyObject* shape_tuple(PyObject* shape) {
    bool plain = PyTuple_CheckExact(shape);
    for (Py_ssize_t i = 0; plain && i < PyTuple_GET_SIZE(shape); ++i) plain = PyLong_CheckExact(PyTuple_GET_ITEM(shape, i));
    if (plain) {
        Py_INCREF(shape);
        return shape;
    }
    PyObject* all = PySequence_Tuple(shape);
    if (all == nullptr) return nullptr;
    PyObject* out = PyTuple_New(PyTuple_GET_SIZE(all));
    for (Py_ssize_t i = 0; out != nullptr && i < PyTuple_GET_SIZE(all); ++i) {
        PyObject* v = PyObject_CallOneArg((PyObject*)&PyLong_Type, PyTuple_GET_ITEM(all, i));
        if (v == nullptr) Py_CLEAR(out);
        else PyTuple_SET_ITEM(out, i, v);
    }
    Py_DECREF(all);
    return out;
}

// The storage type of a name: its own (borrowed) string, or NULL with an error
PyObject* storage_type(PyObject* dtype, int* item, int* code) {
    auto is = [&](PyObject* name) { return dtype == name || (PyUnicode_Check(dtype) && PyUnicode_Compare(dtype, name) == 0); };
    if (is(g_f32)) { *item = 4; *code = LUXHIP_F32; return g_f32; }
    if (is(g_bf16)) { *item = 2; *code = LUXHIP_BF16; return g_bf16; }
    if (is(g_u8)) { *item = 1; *code = -1; return g_u8; }
    return PyErr_Format(PyExc_TypeError, "unsupported dtype %R (use 'f32' or 'bf16'; 'u8' for masks)", dtype);
}

int array_init(Array* self, PyObject* args, PyObject* kw) {
    static const char* names[] = {"shape", "dtype", "ptr", "base", nullptr};
    PyObject *shape = nullptr, *dtype = g_f32, *ptr = Py_None, *base = Py_None;
    if (kw == nullptr && PyTuple_GET_SIZE(args) >= 1 && PyTuple_GET_SIZE(args) <= 2) {
        shape = PyTuple_GET_ITEM(args, 0);
        if (PyTuple_GET_SIZE(args) == 2) dtype = PyTuple_GET_ITEM(args, 1);
    } else if (!PyArg_ParseTupleAndKeywords(args, kw, "O|OOO", const_cast<char**>(names), &shape, &dtype, &ptr, &base)) {
        return -1;
    }
    int item = 0, code = 0;
    dtype = storage_type(dtype, &item, &code);
    if (dtype == nullptr) return -1;
    shape = shape_tuple(shape);
    if (shape == nullptr) return -1;
    int64_t size;
    if (!shape_size(shape, &size)) {
        Py_DECREF(shape);
        return -1;
    }
    if (self->owner) device_free((uintptr_t)self->ptr);          // a second __init__
    self->owner = 0;
    self->ptr = 0;
    Py_XSETREF(self->shape, shape);
    Py_INCREF(dtype);
    Py_XSETREF(self->dtype, dtype);
    Py_INCREF(base);
    Py_XSETREF(self->base, base);
    if (ptr == Py_None) {
        uintptr_t p;
        const int64_t bytes = size > INT64_MAX / 8 ? INT64_MAX : size * item;
        if (device_alloc(bytes < 1 ? 1 : (size_t)bytes, &p) != 0) return -1;
        self->ptr = p;
        self->owner = 1;
    } else {
        PyObject* v = PyObject_CallOneArg((PyObject*)&PyLong_Type, ptr);
        if (v == nullptr) return -1;
        self->ptr = PyLong_AsUnsignedLongLong(v);
        Py_DECREF(v);
        if (PyErr_Occurred()) return -1;
    }
    return 0;
}
int array_traverse(Array* self, visitproc visit, void* arg) {
    Py_VISIT(self->shape);
    Py_VISIT(self->dtype);
    Py_VISIT(self->base);
    return 0;
}
int array_clear(Array* self) {
    Py_CLEAR(self->base);
    return 0;
}
void array_dealloc(Array* self) {
    PyObject_GC_UnTrack(self);
    if (self->owner) device_free((uintptr_t)self->ptr);
    Py_XDECREF(self->shape);
    Py_XDECREF(self->dtype);
    Py_XDECREF(self->base);
    Py_TYPE(self)->tp_free((PyObject*)self);
}
// shape and dtype may be set, as attributes of any Python object: what follows from them is worked out when it is asked for
bool size_now(Array* self, int64_t* size) {
    PyObject* shape = self->shape != nullptr ? shape_tuple(self->shape) : nullptr;
    if (shape == nullptr) {
        if (self->shape == nullptr) PyErr_SetString(PyExc_AttributeError, "shape");      // __init__ has not run
        return false;
    }
    const bool ok = shape_size(shape, size);
    Py_DECREF(shape);
    return ok;
}
bool type_now(Array* self, int* item, int* code) {
    if (self->dtype != nullptr) return storage_type(self->dtype, item, code) != nullptr;
    PyErr_SetString(PyExc_AttributeError, "dtype");
    return false;
}
PyObject* array_size(Array* self, void*) {
    int64_t size;
    return size_now(self, &size) ? PyLong_FromLongLong(size) : nullptr;
}
PyObject* array_ndim(Array* self, void*) {
    if (self->shape == nullptr) return PyErr_Format(PyExc_AttributeError, "shape");
    const Py_ssize_t n = PyObject_Length(self->shape);
    return n < 0 ? nullptr : PyLong_FromSsize_t(n);
}
PyObject* array_nbytes(Array* self, void*) {
    int64_t size;
    int item, code;
    return size_now(self, &size) && type_now(self, &item, &code) ? PyLong_FromLongLong(size * item) : nullptr;
}
PyObject* array_itemsize(Array* self, void*) {
    int item, code;
    return type_now(self, &item, &code) ? PyLong_FromLong(item) : nullptr;
}
PyObject* array_code(Array* self, void*) {
    int item, code;
    return type_now(self, &item, &code) ? PyLong_FromLong(code) : nullptr;
}

PyMemberDef array_members[] = {
    {"shape", T_OBJECT_EX, offsetof(Array, shape), 0, nullptr},
    {"dtype", T_OBJECT_EX, offsetof(Array, dtype), 0, nullptr},
    {"ptr", T_ULONGLONG, offsetof(Array, ptr), 0, nullptr},
    {"_base", T_OBJECT, offsetof(Array, base), 0, nullptr},
    {"_owner", T_BOOL, offsetof(Array, owner), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};
PyGetSetDef array_getset[] = {
    {"itemsize", (getter)array_itemsize, nullptr, nullptr, nullptr},
    {"code", (getter)array_code, nullptr, nullptr, nullptr},
    {"size", (getter)array_size, nullptr, nullptr, nullptr},
    {"ndim", (getter)array_ndim, nullptr, nullptr, nullptr},
    {"nbytes", (getter)array_nbytes, nullptr, nullptr, nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr},
};
PyTypeObject ArrayType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// fp32 statistics (saved mean / inverse standard deviation) of n entries
struct Stat {
    PyObject_HEAD
    long long n;
    unsigned long long ptr;
};
int stat_init(Stat* self, PyObject* args, PyObject* kw) {
    static const char* names[] = {"n", nullptr};
    PyObject* n;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "O", const_cast<char**>(names), &n)) return -1;
    PyObject* v = PyObject_CallOneArg((PyObject*)&PyLong_Type, n);
    if (v == nullptr) return -1;
    const long long count = PyLong_AsLongLong(v);
    Py_DECREF(v);
    if (count == -1 && PyErr_Occurred()) return -1;
    uintptr_t p;
    if (device_alloc(count < 1 ? 4 : (size_t)count * 4, &p) != 0) return -1;
    device_free((uintptr_t)self->ptr);
    self->n = count;
    self->ptr = p;
    return 0;
}
void stat_dealloc(Stat* self) {
    device_free((uintptr_t)self->ptr);
    Py_TYPE(self)->tp_free((PyObject*)self);
}
PyMemberDef stat_members[] = {
    {"n", T_LONGLONG, offsetof(Stat, n), 0, nullptr},
    {"ptr", T_ULONGLONG, offsetof(Stat, ptr), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};
PyTypeObject StatType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyMethodDef methods[] = {
    {"call", (PyCFunction)(void (*)(void))host_call, METH_FASTCALL, "call(name, *args): an entry point of the library; raises on a status other than 0"},
    {"bind", host_bind, METH_VARARGS, "bind(name, address)"},
    {"configure", host_configure, METH_VARARGS, "configure(load, slow_call, check, c_void_p, Array, ConvDimsStruct)"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native part of the Python host side", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    ArrayType.tp_name = "lux_jl_amd._host.Array";
    ArrayType.tp_basicsize = sizeof(Array);
    ArrayType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
    ArrayType.tp_new = PyType_GenericNew;
    ArrayType.tp_init = (initproc)array_init;
    ArrayType.tp_dealloc = (destructor)array_dealloc;
    ArrayType.tp_traverse = (traverseproc)array_traverse;
    ArrayType.tp_clear = (inquiry)array_clear;
    ArrayType.tp_members = array_members;
    ArrayType.tp_getset = array_getset;
    StatType.tp_name = "lux_jl_amd._host.Stat";
    StatType.tp_basicsize = sizeof(Stat);
    StatType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    StatType.tp_new = PyType_GenericNew;
    StatType.tp_init = (initproc)stat_init;
    StatType.tp_dealloc = (destructor)stat_dealloc;
    StatType.tp_members = stat_members;
    if (PyType_Ready(&ArrayType) < 0 || PyType_Ready(&StatType) < 0) return nullptr;
    g_f32 = PyUnicode_InternFromString("f32");
    g_bf16 = PyUnicode_InternFromString("bf16");
    g_u8 = PyUnicode_InternFromString("u8");
    g_index = PyDict_New();
    if (g_f32 == nullptr || g_bf16 == nullptr || g_u8 == nullptr || g_index == nullptr) return nullptr;
    for (size_t i = 0; i < sizeof(g_entries) / sizeof(g_entries[0]); ++i) {
        PyObject* at = PyLong_FromSize_t(i);
        if (at == nullptr || PyDict_SetItemString(g_index, g_entries[i].name, at) < 0) return nullptr;
        Py_DECREF(at);
    }
    PyObject* m = PyModule_Create(&module);
    if (m == nullptr) return nullptr;
    Py_INCREF(&ArrayType);
    Py_INCREF(&StatType);
    if (PyModule_AddObject(m, "Array", (PyObject*)&ArrayType) < 0 || PyModule_AddObject(m, "Stat", (PyObject*)&StatType) < 0) return nullptr;
    return m;
}
