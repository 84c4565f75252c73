// The calls a serving program makes per layer and per round, from Python to the C ABI without ctypes: arguments are
// read where Python holds them and the library is entered with the interpreter released, as ctypes does.
//
// Bound: host instructions. A step of one launch takes 2.8 us of host time from C and of two 5.1; through ctypes, which
// converts every argument by its declared type, and the packing of the items in Python they took 4.3 and 7.5, and with
// two launches of 7.2 us of device time a decode forward was the host's to finish. Host time a layer, ctypes -> this: 8
// layers of one row at 4,096 7.65 -> 6.3 us, of preparing steps 8.65 -> 6.9, f32 8.2 -> 6.6.
//
// Only plain arguments are taken here: exact ints, floats and bools, items in lists or tuples, C-contiguous float32
// arrays. Whatever else a caller passes (numpy scalars, pointer objects, other sequences) is answered with kNotPlain before
// anything is called, and hip_compute.py then makes the same call through ctypes with that module's conversions.
//
// The library's functions are bound by address (bind), so that this module serves whichever build is loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#define NPY_NO_DEPRECATED_API NPY_2_0_API_VERSION
#include <numpy/arrayobject.h>

#include <cmath>
#include <cstdint>

#include "../../include/itak_hip_kv.h"

namespace {

constexpr long kNotPlain = -1;
constexpr Py_ssize_t kMostItems = 64;

decltype(&itak_attention_step_device) step_fn;
decltype(&itak_attention_prep_step_device) prep_step_fn;
decltype(&itak_kv_truncate) truncate_fn;
decltype(&itak_compute_attention) compute_fn;
decltype(&itak_gqa_attention) gqa_fn;
PyTypeObject *cache_type;  // hip_compute.KvCache
PyObject *slot_name;

// An exact int as ctypes takes it for an unsigned 64-bit argument or a pointer: modulo 2^64.
bool plain_u64(PyObject *o, uint64_t &v) {
    if (!PyLong_CheckExact(o)) return false;
    v = PyLong_AsUnsignedLongLongMask(o);
    return true;
}
template <typename T>
bool plain_ptr(PyObject *o, T *&p) {
    uint64_t v;
    if (!plain_u64(o, v)) return false;
    p = reinterpret_cast<T *>(uintptr_t(v));
    return true;
}
// An exact int that is an unsigned value of `bits` bits.
bool plain_within(PyObject *o, int bits, uint64_t &v) {
    if (!PyLong_CheckExact(o)) return false;
    v = PyLong_AsUnsignedLongLong(o);
    if (v == ~0ull && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return bits == 64 || v >> bits == 0;
}
bool plain_float(PyObject *o, float &f) {
    if (PyFloat_CheckExact(o)) {
        f = float(PyFloat_AS_DOUBLE(o));
        return true;
    }
    if (!PyLong_CheckExact(o)) return false;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    f = float(d);
    return true;
}
// None is the default scale.
bool plain_scale(PyObject *o, float &f) {
    if (o != Py_None) return plain_float(o, f);
    f = NAN;
    return true;
}
bool plain_slot(PyObject *o, uint32_t &slot) {
    uint64_t v;
    if (Py_TYPE(o) == cache_type) {
        PyObject *s = PyObject_GetAttr(o, slot_name);
        if (!s) {
            PyErr_Clear();
            return false;
        }
        const bool ok = plain_within(s, 32, v);
        Py_DECREF(s);
        if (!ok) return false;
    } else if (!plain_within(o, 32, v)) {
        return false;
    }
    slot = uint32_t(v);
    return true;
}
bool plain_sequence(PyObject *o, PyObject **&at, Py_ssize_t &n) {
    if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
    at = PySequence_Fast_ITEMS(o);
    n = PySequence_Fast_GET_SIZE(o);
    return true;
}
bool plain_items(PyObject *o, itak_batch_item *items, uint32_t &count) {
    PyObject **at;
    Py_ssize_t n;
    if (!plain_sequence(o, at, n) || n > kMostItems) return false;
    for (Py_ssize_t i = 0; i < n; ++i) {
        uint64_t rows;
        if (!PyTuple_CheckExact(at[i]) || PyTuple_GET_SIZE(at[i]) != 2 ||
            !plain_slot(PyTuple_GET_ITEM(at[i], 0), items[i].slot) || !plain_within(PyTuple_GET_ITEM(at[i], 1), 32, rows))
            return false;
        items[i].rows = uint32_t(rows);
    }
    count = uint32_t(n);
    return true;
}
// A C-contiguous array of native floats; its address is null where it is empty.
bool plain_array(PyObject *o, const float *&data, uint64_t &size) {
    if (!PyArray_CheckExact(o)) return false;
    PyArrayObject *a = reinterpret_cast<PyArrayObject *>(o);
    if (PyArray_TYPE(a) != NPY_FLOAT32 || !PyArray_ISCARRAY_RO(a)) return false;
    size = uint64_t(PyArray_SIZE(a));
    data = size ? static_cast<const float *>(PyArray_DATA(a)) : nullptr;
    return true;
}
PyObject *not_plain() { return PyLong_FromLong(kNotPlain); }
bool arity(Py_ssize_t got, Py_ssize_t want) {
    if (got != want) PyErr_Format(PyExc_TypeError, "%zd arguments, not %zd", want, got);
    return got == want;
}

// step(pool, layer, items, q, k, v, out, q_heads, scale, softcap) -> status
PyObject *step(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 10)) return nullptr;
    itak_pool *pool;
    const float *q, *k, *v;
    float *out, scale, softcap;
    uint64_t layer, heads;
    uint32_t count;
    itak_batch_item items[kMostItems];
    if (!plain_ptr(a[0], pool) || !plain_u64(a[1], layer) || !plain_items(a[2], items, count) || !plain_ptr(a[3], q) ||
        !plain_ptr(a[4], k) || !plain_ptr(a[5], v) || !plain_ptr(a[6], out) || !plain_u64(a[7], heads) ||
        !plain_scale(a[8], scale) || !plain_float(a[9], softcap))
        return not_plain();
    itak_status st;
    Py_BEGIN_ALLOW_THREADS
    st = step_fn(pool, layer, items, count, q, k, v, out, heads, scale, softcap);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(st);
}

// prep_step(pool, layer, items, q, k, v, gate, out, q_heads, scale, softcap, q_norm, k_norm, eps, rope_base, interleaved,
// rotary_dim) -> status
PyObject *prep_step(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 17)) return nullptr;
    itak_pool *pool;
    const float *q, *k, *v, *gate;
    float *out, scale, softcap;
    uint64_t layer, heads, rotary;
    uint32_t count;
    itak_batch_item items[kMostItems];
    itak_prep_params prep{};
    if (!plain_ptr(a[0], pool) || !plain_u64(a[1], layer) || !plain_items(a[2], items, count) || !plain_ptr(a[3], q) ||
        !plain_ptr(a[4], k) || !plain_ptr(a[5], v) || !plain_ptr(a[6], gate) || !plain_ptr(a[7], out) ||
        !plain_u64(a[8], heads) || !plain_float(a[9], scale) || !plain_float(a[10], softcap) ||
        !plain_ptr(a[11], prep.q_norm_weight) || !plain_ptr(a[12], prep.k_norm_weight) || !plain_float(a[13], prep.eps) ||
        !plain_float(a[14], prep.rope_base) || !PyBool_Check(a[15]) || !plain_u64(a[16], rotary))
        return not_plain();
    prep.rope_interleaved = a[15] == Py_True ? 1 : 0;
    prep.rotary_dim = uint32_t(rotary);
    itak_status st;
    Py_BEGIN_ALLOW_THREADS
    st = prep_step_fn(pool, layer, items, count, q, k, v, gate, out, heads, scale, softcap, &prep);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(st);
}

// truncate(pool, slots, lengths) -> status
PyObject *truncate(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 3)) return nullptr;
    itak_pool *pool;
    PyObject **slot_at, **length_at;
    Py_ssize_t slots, lengths;
    uint32_t slot[kMostItems];
    uint64_t length[kMostItems];
    if (!plain_ptr(a[0], pool) || !plain_sequence(a[1], slot_at, slots) || !plain_sequence(a[2], length_at, lengths) ||
        slots > kMostItems || lengths != slots)
        return not_plain();
    for (Py_ssize_t i = 0; i < slots; ++i)
        if (!plain_slot(slot_at[i], slot[i]) || !plain_within(length_at[i], 64, length[i])) return not_plain();
    itak_status st;
    Py_BEGIN_ALLOW_THREADS
    st = truncate_fn(pool, slot, length, uint32_t(slots));
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(st);
}

// compute(pool, slot, layer, q, k, v, q_heads, position, softcap, rope_base) -> outputs, or a status
PyObject *compute(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 10)) return nullptr;
    itak_pool *pool;
    const float *q, *k, *v;
    uint64_t slot, layer, q_size, k_size, v_size, heads, position;
    float softcap, base;
    if (!plain_ptr(a[0], pool) || !plain_u64(a[1], slot) || !plain_u64(a[2], layer) || !plain_array(a[3], q, q_size) ||
        !plain_array(a[4], k, k_size) || !plain_array(a[5], v, v_size) || !plain_u64(a[6], heads) ||
        !plain_u64(a[7], position) || !plain_float(a[8], softcap) || !plain_float(a[9], base))
        return not_plain();
    npy_intp dims[] = {npy_intp(q_size)};
    PyObject *out = PyArray_SimpleNew(1, dims, NPY_FLOAT32);  // every element is written, or a status comes back
    if (!out) return nullptr;
    float *to = q_size ? static_cast<float *>(PyArray_DATA(reinterpret_cast<PyArrayObject *>(out))) : nullptr;
    itak_status st;
    Py_BEGIN_ALLOW_THREADS
    st = compute_fn(pool, uint32_t(slot), layer, q, q_size, k, k_size, v, v_size, heads, position, softcap, base, to);
    Py_END_ALLOW_THREADS
    if (st == ITAK_OK) return out;
    Py_DECREF(out);
    return PyLong_FromLong(st);
}

// gqa(pool, slot, layer, q, queries, q_heads, positions, scale, softcap) -> outputs, or a status
PyObject *gqa(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 9)) return nullptr;
    itak_pool *pool;
    const float *q;
    uint64_t slot, layer, q_size, queries, heads, position[kMostItems];
    float scale, softcap;
    PyObject **position_at;
    Py_ssize_t positions;
    if (!plain_ptr(a[0], pool) || !plain_u64(a[1], slot) || !plain_u64(a[2], layer) || !plain_array(a[3], q, q_size) ||
        !plain_u64(a[4], queries) || !plain_u64(a[5], heads) || !plain_sequence(a[6], position_at, positions) ||
        positions > kMostItems || !plain_scale(a[7], scale) || !plain_float(a[8], softcap))
        return not_plain();
    for (Py_ssize_t i = 0; i < positions; ++i)
        if (!plain_within(position_at[i], 64, position[i])) return not_plain();
    npy_intp dims[] = {npy_intp(q_size)};
    PyObject *out = PyArray_SimpleNew(1, dims, NPY_FLOAT32);
    if (!out) return nullptr;
    float *to = q_size ? static_cast<float *>(PyArray_DATA(reinterpret_cast<PyArrayObject *>(out))) : nullptr;
    itak_status st;
    Py_BEGIN_ALLOW_THREADS
    st = gqa_fn(pool, uint32_t(slot), layer, q, q_size, queries, heads, positions ? position : nullptr, uint64_t(positions),
                scale, softcap, to);
    Py_END_ALLOW_THREADS
    if (st == ITAK_OK) return out;
    Py_DECREF(out);
    return PyLong_FromLong(st);
}

// bind(KvCache, address of each of the five functions above, in their order)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 6)) return nullptr;
    uint64_t at[5];
    if (!PyType_Check(a[0])) {
        PyErr_SetString(PyExc_TypeError, "the cache's type comes first");
        return nullptr;
    }
    for (int i = 0; i < 5; ++i)
        if (!plain_within(a[i + 1], 64, at[i]) || at[i] == 0) {
            PyErr_SetString(PyExc_TypeError, "an address is an int that is not zero");
            return nullptr;
        }
    Py_INCREF(a[0]);
    Py_XDECREF(reinterpret_cast<PyObject *>(cache_type));
    cache_type = reinterpret_cast<PyTypeObject *>(a[0]);
    step_fn = reinterpret_cast<decltype(step_fn)>(uintptr_t(at[0]));
    prep_step_fn = reinterpret_cast<decltype(prep_step_fn)>(uintptr_t(at[1]));
    truncate_fn = reinterpret_cast<decltype(truncate_fn)>(uintptr_t(at[2]));
    compute_fn = reinterpret_cast<decltype(compute_fn)>(uintptr_t(at[3]));
    gqa_fn = reinterpret_cast<decltype(gqa_fn)>(uintptr_t(at[4]));
    Py_RETURN_NONE;
}

template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyMethodDef method(const char *name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}
PyMethodDef methods[] = {method<bind>("bind"), method<step>("step"),       method<prep_step>("prep_step"),
                         method<truncate>("truncate"), method<compute>("compute"), method<gqa>("gqa"),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_itak_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__itak_front(void) {
    import_array();
    slot_name = PyUnicode_InternFromString("slot");
    return slot_name ? PyModule_Create(&module) : nullptr;
}
