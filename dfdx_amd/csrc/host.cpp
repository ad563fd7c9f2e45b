// The native half of the Python front-end (dfdx_amd/rocm.py, encoder.py): calls into libdfdx_rocm.so, device memory from torch's
// allocator, and the Views that a call returns.
//
// What bounds a small call is the host: a launch takes 2.9 us of it, and the front-end took as much again in argument conversions
// (0.45 us a call through ctypes, 0.1 here), allocations through Python (1.2 us, 0.8 here) and pieces of one allocation (torch.Tensor.split:
// 0.9 us a piece, 0.2 here).  Host time of a pass, before and after: one small product 7.2 -> 5.8 us, a Linear layer's forward and backward on
// 64 rows 23.4 -> 15.1, attention's ops 72 -> 53, a training step of a small encoder block 102 -> 87 (16 launches and the caller's own 10).
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/dfdx_rocm.h"

namespace {

PyObject *s_storage, *s_dtype, *s_shape, *s_strides, *s_offset, *s_owner, *s_value, *s_data_ptr, *s_at, *s_check, *s_forget, *s_ordinal;

int64_t item_size(PyObject *dtype) {
    const char *name = PyUnicode_Check(dtype) ? PyUnicode_AsUTF8(dtype) : nullptr;
    if (name) {
        if (!std::strcmp(name, "f16") || !std::strcmp(name, "bf16")) return 2;
        if (!std::strcmp(name, "f32")) return 4;
        if (!std::strcmp(name, "f64")) return 8;
    }
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, dtype);
    return -1;
}

// The address of a tensor's data.
bool tensor_address(PyObject *t, char **out) {
    if (THPVariable_Check(t)) {
        *out = (char *)THPVariable_Unpack(t).data_ptr();
        return true;
    }
    PyObject *at = PyObject_CallMethodNoArgs(t, s_data_ptr);
    if (!at) return false;
    *out = (char *)PyLong_AsVoidPtr(at);
    Py_DECREF(at);
    return !PyErr_Occurred();
}

// A pointer argument: None, an address, the contents of a bytes object, a View, or anything with a `value` (ctypes.c_void_p).
bool address(PyObject *o, char **out) {
    if (o == Py_None) {
        *out = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        *out = (char *)PyLong_AsVoidPtr(o);
        return *out || !PyErr_Occurred();
    }
    if (PyBytes_Check(o)) {
        *out = PyBytes_AS_STRING(o);
        return true;
    }
    if (PyObject *storage = PyObject_GetAttr(o, s_storage)) {
        bool ok = tensor_address(storage, out);
        Py_DECREF(storage);
        PyObject *offset = ok ? PyObject_GetAttr(o, s_offset) : nullptr;
        if (!offset) return false;
        const int64_t n = PyLong_AsLongLong(offset);
        Py_DECREF(offset);
        if (n == -1 && PyErr_Occurred()) return false;
        if (n) {
            PyObject *dtype = PyObject_GetAttr(o, s_dtype);
            const int64_t es = dtype ? item_size(dtype) : -1;
            Py_XDECREF(dtype);
            if (es < 0) return false;
            *out += n * es;
        }
        return true;
    }
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return false;
    PyErr_Clear();
    PyObject *value = PyObject_GetAttr(o, s_value);
    if (!value) return false;
    const bool ok = (value == Py_None || PyLong_Check(value)) && address(value, out);
    if (!ok && !PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "not an address");
    Py_DECREF(value);
    return ok;
}

// One argument of an entry point, by its C type.
template <typename T, typename = void> struct Arg;
template <typename T> struct Arg<T, std::enable_if_t<std::is_integral_v<T>>> {
    T v;
    bool load(PyObject *o) {
        const long long n = PyLong_AsLongLong(o);
        v = (T)n;
        return n != -1 || !PyErr_Occurred();
    }
    T value() const { return v; }
};
template <typename T> struct Arg<T, std::enable_if_t<std::is_floating_point_v<T>>> {
    T v;
    bool load(PyObject *o) {
        const double d = PyFloat_AsDouble(o);
        v = (T)d;
        return d != -1.0 || !PyErr_Occurred();
    }
    T value() const { return v; }
};
template <typename T> struct Arg<T *> {
    char *v;
    bool load(PyObject *o) { return address(o, &v); }
    T *value() const { return (T *)v; }
};
// a small array: a tuple or list of whole numbers (addresses, too), or as any other pointer
template <typename E, int MOST> struct ArrayArg {
    E own[MOST];
    char *v = (char *)own;
    bool load(PyObject *o) {
        if (!PyTuple_Check(o) && !PyList_Check(o)) return address(o, &v);
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
        if (n > MOST) {
            PyErr_SetString(PyExc_ValueError, "too many elements");
            return false;
        }
        for (Py_ssize_t i = 0; i < n; i++) {
            const long long e = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(o, i));
            if (e == -1 && PyErr_Occurred()) return false;
            own[i] = (E)e;
        }
        return true;
    }
    const E *value() const { return (const E *)v; }
};
template <> struct Arg<const int64_t *> : ArrayArg<int64_t, 8> {};
template <> struct Arg<void *const *> : ArrayArg<void *, DFDX_ROCM_ENCODER_PARAMS> {};

// An entry point as a Python function; other threads run while it does.
template <typename... A, size_t... I> bool load_all(std::tuple<Arg<A>...> &t, PyObject *const *args, std::index_sequence<I...>) {
    return (std::get<I>(t).load(args[I]) && ...);
}
template <auto F> struct Entry;
template <typename... A, int (*F)(A...)> struct Entry<F> {
    static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
        if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%zd arguments given, %zd taken", n, (Py_ssize_t)sizeof...(A));
        std::tuple<Arg<A>...> t;
        if (!load_all<A...>(t, args, std::index_sequence_for<A...>{})) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = std::apply([](const auto &...a) { return F(a.value()...); }, t);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
};

template <typename F> PyObject *guarded(F f) {  // C++ exceptions of torch as Python ones
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

struct WithoutGil {  // other threads run meanwhile, as under torch's own allocation calls
    PyThreadState *const state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};
at::Tensor allocate(int64_t ordinal, int64_t bytes) {
    WithoutGil free;
    return at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(at::Device(at::kCUDA, (c10::DeviceIndex)ordinal)));
}

// `bytes` bytes of a tensor of bytes as a tensor of their own on the same storage.
at::Tensor piece(const at::Tensor &from, int64_t offset, int64_t bytes) {
    at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(from.storage()), from.key_set(), from.dtype());
    c10::TensorImpl *impl = t.unsafeGetTensorImpl();
    impl->set_storage_offset(from.storage_offset() + offset);
    impl->set_sizes_contiguous({bytes});
    impl->set_version_counter(from.unsafeGetTensorImpl()->version_counter());  // changes in place count for all pieces
    return t;
}

// View(storage, dtype, shape, strides, 0, owner); steals `storage`.
PyObject *make_view(PyTypeObject *cls, PyObject *storage, PyObject *dtype, PyObject *shape, PyObject *strides, PyObject *owner) {
    static PyObject *const zero = PyLong_FromLong(0);
    if (!storage) return nullptr;
    PyObject *view = cls->tp_alloc(cls, 0);
    const bool ok = view && !PyObject_SetAttr(view, s_storage, storage) && !PyObject_SetAttr(view, s_dtype, dtype) && !PyObject_SetAttr(view, s_shape, shape) &&
                    !PyObject_SetAttr(view, s_strides, strides) && !PyObject_SetAttr(view, s_offset, zero) && !PyObject_SetAttr(view, s_owner, owner);
    Py_DECREF(storage);
    if (ok) return view;
    Py_XDECREF(view);
    return nullptr;
}

// Strides of a tuple of extents, and the bytes of as many elements of `size` bytes (at least 16).  Numbers beyond 64 bits are an
// OverflowError, also on the way to a product of zero.
PyObject *row_major(PyObject *shape, int64_t size, int64_t *bytes) {
    const Py_ssize_t n = PyTuple_GET_SIZE(shape);
    PyObject *strides = PyTuple_New(n);
    int64_t step = 1;
    for (Py_ssize_t i = n - 1; strides && i >= 0; i--) {
        PyTuple_SET_ITEM(strides, i, PyLong_FromLongLong(step));
        const int64_t e = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i));
        if (!(e == -1 && PyErr_Occurred()) && __builtin_mul_overflow(step, e, &step)) PyErr_SetString(PyExc_OverflowError, "more elements than 64 bits count");
        if (PyErr_Occurred()) Py_CLEAR(strides);
    }
    if (!strides) return nullptr;
    if (__builtin_mul_overflow(step, size, bytes)) {
        PyErr_SetString(PyExc_OverflowError, "more bytes than 64 bits count");
        Py_CLEAR(strides);
    }
    *bytes = std::max<int64_t>(*bytes, 16);
    return strides;
}

// bytes(ordinal, n): uninitialised device memory
PyObject *py_bytes(PyObject *ordinal, PyObject *const *args, Py_ssize_t n) {
    if (n != 1) return PyErr_Format(PyExc_TypeError, "one argument taken");
    const int64_t dev = PyLong_AsLongLong(ordinal), bytes = PyLong_AsLongLong(args[0]);
    if (PyErr_Occurred()) return nullptr;
    return guarded([&] { return THPVariable_Wrap(allocate(dev, bytes)); });
}
PyMethodDef bytes_def = {"bytes", (PyCFunction)(void *)py_bytes, METH_FASTCALL, nullptr};
// allocator(ordinal): the function above for one device
PyObject *py_allocator(PyObject *, PyObject *ordinal) { return PyCFunction_New(&bytes_def, ordinal); }

// empty(View, ordinal, dtype, shape): a contiguous View of uninitialised memory
PyObject *py_empty(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 4 || !PyType_Check(args[0]) || !PyTuple_Check(args[3])) return PyErr_Format(PyExc_TypeError, "empty(View, ordinal, dtype, shape)");
    const int64_t es = item_size(args[2]), dev = PyLong_AsLongLong(args[1]);
    int64_t bytes = 0;
    PyObject *strides = es < 0 || PyErr_Occurred() ? nullptr : row_major(args[3], es, &bytes);
    if (!strides) return nullptr;
    PyObject *view = make_view((PyTypeObject *)args[0], guarded([&] { return THPVariable_Wrap(allocate(dev, bytes)); }), args[2], args[3], strides, Py_None);
    Py_DECREF(strides);
    return view;
}

// carve(dev, View, Arena, likes, deferred): zeroed Views of the shapes of `likes`, each on its own 256 B-aligned piece of one
// allocation; see Rocm.zeros_many.
PyObject *py_carve(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 5 || !PyType_Check(args[1])) return PyErr_Format(PyExc_TypeError, "carve(dev, View, Arena, likes, deferred)");
    PyObject *const dev = args[0], *const cls = args[1];
    const int deferred = PyObject_IsTrue(args[4]);
    if (deferred < 0) return nullptr;
    PyObject *likes = PySequence_List(args[3]), *ordinal = nullptr, *at = nullptr, *arena = nullptr, *owner = nullptr, *views = nullptr;
    if (!likes) return nullptr;
    const Py_ssize_t count = PyList_GET_SIZE(likes);
    struct Part {
        PyObject *dtype, *shape, *strides;
        int64_t offset, bytes;
    };
    std::vector<Part> parts;
    parts.reserve((size_t)count);
    auto done = [&](PyObject *result) -> PyObject * {
        for (Part &p : parts) {
            Py_XDECREF(p.dtype);
            Py_XDECREF(p.shape);
            Py_XDECREF(p.strides);
        }
        Py_XDECREF(ordinal);
        Py_XDECREF(at);
        Py_XDECREF(arena);
        Py_XDECREF(owner);
        Py_DECREF(likes);
        if (!result) Py_XDECREF(views);
        return result;
    };
    int64_t total = 0;
    for (Py_ssize_t i = 0; i < count; i++) {
        PyObject *like = PyList_GET_ITEM(likes, i), *shape = PyObject_GetAttr(like, s_shape);
        parts.push_back({PyObject_GetAttr(like, s_dtype), shape ? PySequence_Tuple(shape) : nullptr, nullptr, total, 0});
        Py_XDECREF(shape);
        Part &p = parts.back();
        if (!p.dtype || !p.shape) return done(nullptr);
        const int64_t es = item_size(p.dtype);
        if (es < 0 || !(p.strides = row_major(p.shape, es, &p.bytes))) return done(nullptr);
        if (__builtin_add_overflow(total, p.bytes, &total) || __builtin_add_overflow(total, -p.bytes & 255, &total)) {
            PyErr_SetString(PyExc_OverflowError, "more bytes than 64 bits count");
            return done(nullptr);
        }
    }
    ordinal = PyObject_GetAttr(dev, s_ordinal);
    at = PyObject_GetAttr(dev, s_at);
    if (!ordinal || !at) return done(nullptr);
    dfdx_rocm_ctx *const ctx = (dfdx_rocm_ctx *)PyLong_AsVoidPtr(at);
    const int64_t index = PyLong_AsLongLong(ordinal);
    if (PyErr_Occurred()) return done(nullptr);
    total = std::max<int64_t>(total, 16);
    arena = guarded([&] { return THPVariable_Wrap(allocate(index, total)); });
    if (!arena) return done(nullptr);
    char *const base = (char *)THPVariable_Unpack(arena).data_ptr();
    owner = deferred ? PyObject_CallFunctionObjArgs(args[2], dev, arena, nullptr) : Py_NewRef(Py_None);
    if (!owner) return done(nullptr);
    int rc = 0;
    Py_BEGIN_ALLOW_THREADS
    if (!deferred) rc = dfdx_rocm_memset_zero(ctx, base, (size_t)total);
    else
        for (size_t i = 0; i < parts.size() && !rc; i++) rc = dfdx_rocm_zero_deferred(ctx, base + parts[i].offset, (size_t)parts[i].bytes);
    Py_END_ALLOW_THREADS
    if (rc) {
        if (deferred) Py_XDECREF(PyObject_CallMethodNoArgs(owner, s_forget));
        if (!PyErr_Occurred()) {
            PyObject *code = PyLong_FromLong(rc);
            Py_XDECREF(code ? PyObject_CallMethodOneArg(dev, s_check, code) : nullptr);
            Py_XDECREF(code);
        }
        return done(nullptr);
    }
    views = PyList_New(count);
    for (Py_ssize_t i = 0; views && i < count; i++) {
        const Part &p = parts[(size_t)i];
        PyObject *view = make_view((PyTypeObject *)cls, guarded([&] { return THPVariable_Wrap(piece(THPVariable_Unpack(arena), p.offset, p.bytes)); }), p.dtype,
                                   p.shape, p.strides, owner);
        if (!view) return done(nullptr);
        PyList_SET_ITEM(views, i, view);
    }
    return done(views);
}

// pieces(View, arena, dtype, ((name, offset, bytes, shape, strides), ..)): {name: View} into one allocation
PyObject *py_pieces(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 4 || !PyType_Check(args[0]) || !THPVariable_Check(args[1]) || !PyTuple_Check(args[3]))
        return PyErr_Format(PyExc_TypeError, "pieces(View, arena, dtype, places)");
    PyObject *views = PyDict_New();
    for (Py_ssize_t i = 0; views && i < PyTuple_GET_SIZE(args[3]); i++) {
        PyObject *name, *shape, *strides, *view = nullptr;
        long long offset, bytes;
        if (PyArg_ParseTuple(PyTuple_GET_ITEM(args[3], i), "OLLOO", &name, &offset, &bytes, &shape, &strides))
            view = make_view((PyTypeObject *)args[0], guarded([&] { return THPVariable_Wrap(piece(THPVariable_Unpack(args[1]), offset, bytes)); }), args[2],
                             shape, strides, Py_None);
        if (!view || PyDict_SetItem(views, name, view)) Py_CLEAR(views);
        Py_XDECREF(view);
    }
    return views;
}

// parameters(desc, views, dtype, ((name, shape, strides), ..)): the bytes of a dfdx_rocm_encoder with its parameters' addresses,
// or None where one is not of that type and shape.
PyObject *py_parameters(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 4 || !PyBytes_Check(args[0]) || PyBytes_GET_SIZE(args[0]) != (Py_ssize_t)sizeof(dfdx_rocm_encoder) || !PyTuple_Check(args[3]) ||
        PyTuple_GET_SIZE(args[3]) != DFDX_ROCM_ENCODER_PARAMS)
        return PyErr_Format(PyExc_TypeError, "parameters(desc, views, dtype, shapes)");
    dfdx_rocm_encoder desc;
    std::memcpy(&desc, PyBytes_AS_STRING(args[0]), sizeof(desc));
    for (Py_ssize_t i = 0; i < DFDX_ROCM_ENCODER_PARAMS; i++) {
        PyObject *name, *shape, *strides;
        if (!PyArg_ParseTuple(PyTuple_GET_ITEM(args[3], i), "OOO", &name, &shape, &strides)) return nullptr;
        PyObject *view = PyObject_GetItem(args[1], name);
        if (!view) return nullptr;
        int same = 1;
        PyObject *const want[3] = {shape, strides, args[2]}, *const attr[3] = {s_shape, s_strides, s_dtype};
        for (int a = 0; a < 3 && same == 1; a++) {
            PyObject *have = PyObject_GetAttr(view, attr[a]);
            same = have ? PyObject_RichCompareBool(have, want[a], Py_EQ) : -1;
            Py_XDECREF(have);
        }
        char *at = nullptr;
        if (same == 1 && !address(view, &at)) same = -1;
        Py_DECREF(view);
        if (same < 0) return nullptr;
        if (!same) Py_RETURN_NONE;
        desc.params[i] = at;
    }
    return PyBytes_FromStringAndSize((const char *)&desc, sizeof(desc));
}

#define ENTRY(name) {#name, (PyCFunction)(void *)Entry<&dfdx_rocm_##name>::call, METH_FASTCALL, nullptr}
#define OWN(name, f, flags) {#name, (PyCFunction)(void *)f, flags, nullptr}
PyMethodDef methods[] = {
    ENTRY(memset_zero), ENTRY(zero_deferred), ENTRY(settle_zeros), ENTRY(forget_zeros),
    ENTRY(matmat_forward), ENTRY(matmat_backward), ENTRY(matmat_br_forward), ENTRY(matmat_br_backward),
    ENTRY(matmat_batch3_forward), ENTRY(matmat_batch3_backward), ENTRY(matmat_batch4_forward), ENTRY(matmat_batch4_backward),
    ENTRY(linear_forward), ENTRY(linear_backward), ENTRY(bias_forward), ENTRY(bias_backward),
    ENTRY(scalar_mul_forward), ENTRY(scalar_mul_backward), ENTRY(softmax_forward), ENTRY(softmax_backward),
    ENTRY(reshape_forward), ENTRY(reshape_backward), ENTRY(attention_forward), ENTRY(attention_backward),
    ENTRY(layer_norm_forward), ENTRY(layer_norm_backward), ENTRY(relu_forward), ENTRY(relu_backward), ENTRY(add_forward), ENTRY(add_backward),
    ENTRY(conv2d_forward), ENTRY(conv2d_backward), ENTRY(encoder_forward), ENTRY(encoder_backward),
    OWN(allocator, py_allocator, METH_O), OWN(empty, py_empty, METH_FASTCALL), OWN(carve, py_carve, METH_FASTCALL),
    OWN(pieces, py_pieces, METH_FASTCALL), OWN(parameters, py_parameters, METH_FASTCALL), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "The native half of the Python front-end.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    const struct {
        PyObject **at;
        const char *text;
    } names[] = {{&s_storage, "storage"}, {&s_dtype, "dtype"}, {&s_shape, "shape"}, {&s_strides, "strides"}, {&s_offset, "offset"}, {&s_owner, "owner"},
                 {&s_value, "value"}, {&s_data_ptr, "data_ptr"}, {&s_at, "_at"}, {&s_check, "_check"}, {&s_forget, "forget"}, {&s_ordinal, "ordinal"}};
    for (const auto &n : names)
        if (!(*n.at = PyUnicode_InternFromString(n.text))) return nullptr;
    return PyModule_Create(&module);
}
