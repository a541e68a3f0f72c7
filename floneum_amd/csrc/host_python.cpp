// The Python mirror's calls of a decode step in native code: descriptors are read from the Tensor objects, the library is called and
// the views it returns become Tensors, without a ctypes structure or a Python call per tensor.
//
// Only plain calls are taken: exact Tensor objects of rank 4 whose numbers fit the C fields, and arguments of the documented
// types.  For everything else each function returns None, having done nothing, and the caller goes the general way, which
// accepts or refuses the call.
//
// Host time of a call besides the library's own (2.7 us a launch and more): attention 2.9 -> 0.7 us, rotation and append 5.0 -> 0.8.
// A step of 301 keys in f16 16.1 -> 8.8 us, of 1361 keys 19.1 -> 11.3, a 50-row prompt's layer 20.9 -> 13.9.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cmath>
#include <cstring>

#include "../../include/fusor_hip.h"

namespace {

// The classes of the mirror and where their instances keep what is read here (set by `bind`).
struct Slots {
    PyTypeObject *type = nullptr;
    Py_ssize_t at[5] = {};
};
Slots tensor, view;  // Tensor: buffer, dtype, shape, strides, offset; _View: device, ptr, keepalive
PyTypeObject *cache_type, *rope_type, *norm_type, *lens_type;

PyObject *n_ptr, *n_device, *n_buffer, *n_offset, *n_shape, *n_dtype, *n_stream, *n_value, *n_compute_units, *n_workspace, *n_handle, *n_cos,
    *n_sin, *n_rows, *n_weight, *n_bias, *n_eps, *s_i32;

// a new reference that is let go with the block
struct Ref {
    PyObject *o;
    explicit Ref(PyObject *p) : o(p) {}
    ~Ref() { Py_XDECREF(o); }
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
};

inline PyObject *slot(const Slots &s, PyObject *o, int i) { return *(PyObject **)((char *)o + s.at[i]); }

// A call that is not plain: nothing has been done, no exception is left.
bool not_plain() {
    PyErr_Clear();
    return false;
}

bool as_u64(PyObject *o, uint64_t *out) {
    if (!o || !PyLong_Check(o)) return false;
    *out = PyLong_AsUnsignedLongLong(o);
    return !(*out == (uint64_t)-1 && PyErr_Occurred()) || not_plain();
}
bool as_i64(PyObject *o, int64_t *out) {
    if (!o || !PyLong_Check(o)) return false;
    *out = PyLong_AsLongLong(o);
    return !(*out == -1 && PyErr_Occurred()) || not_plain();
}
template <typename T>
bool as_narrow(PyObject *o, T *out) {
    int64_t v;
    if (!as_i64(o, &v) || (int64_t)(T)v != v) return false;
    *out = (T)v;
    return true;
}
bool attr_u64(PyObject *o, PyObject *name, uint64_t *out) {
    Ref v(PyObject_GetAttr(o, name));
    return v.o ? as_u64(v.o, out) : not_plain();
}
// a pointer held by a ctypes.c_void_p attribute
bool attr_handle(PyObject *o, PyObject *name, void **out) {
    Ref h(PyObject_GetAttr(o, name));
    if (!h.o) return not_plain();
    uint64_t p;
    if (!attr_u64(h.o, n_value, &p)) return false;
    *out = (void *)(uintptr_t)p;
    return true;
}
bool attr_memory(PyObject *o, PyObject *name, void **out) {  // o.name.buffer.ptr
    Ref t(PyObject_GetAttr(o, name));
    if (!t.o) return not_plain();
    Ref b(PyObject_GetAttr(t.o, n_buffer));
    if (!b.o) return not_plain();
    uint64_t p;
    if (!attr_u64(b.o, n_ptr, &p)) return false;
    *out = (void *)(uintptr_t)p;
    return true;
}

template <int RANK, typename C>
bool describe(PyObject *t, C *c, int32_t *dtype, PyObject *device) {
    if (Py_TYPE(t) != tensor.type) return false;
    // (held: an attribute of the memory may be Python code, and so may another thread's turn)
    const Ref memory(Py_XNewRef(slot(tensor, t, 0))), extents(Py_XNewRef(slot(tensor, t, 2))), steps(Py_XNewRef(slot(tensor, t, 3)));
    PyObject *const buffer = memory.o, *const shape = extents.o, *const strides = steps.o;
    if (!buffer || !shape || !strides || !PyTuple_CheckExact(shape) || !PyTuple_CheckExact(strides) || PyTuple_GET_SIZE(shape) != RANK ||
        PyTuple_GET_SIZE(strides) != RANK)
        return false;
    uint64_t ptr;
    if (!attr_u64(buffer, n_ptr, &ptr) || !as_narrow(slot(tensor, t, 1), dtype) || !as_u64(slot(tensor, t, 4), &c->offset)) return false;
    c->ptr = (void *)(uintptr_t)ptr;
    for (int i = 0; i < RANK; i++)
        if (!as_narrow(PyTuple_GET_ITEM(shape, i), &c->shape[i]) || !as_i64(PyTuple_GET_ITEM(strides, i), &c->stride[i])) return false;
    if (!device) return true;
    Ref d(PyObject_GetAttr(buffer, n_device));
    return d.o ? d.o == device : not_plain();
}

PyObject *instance(const Slots &s, int n, PyObject *const *values) {
    PyObject *o = s.type->tp_alloc(s.type, 0);
    if (!o) return nullptr;
    for (int i = 0; i < n; i++) {
        Py_INCREF(values[i]);
        *(PyObject **)((char *)o + s.at[i]) = values[i];
    }
    return o;
}

PyObject *tuple4(const uint32_t *u, const int64_t *i) {
    PyObject *t = PyTuple_New(4);
    for (int n = 0; t && n < 4; n++) {
        PyObject *v = u ? PyLong_FromUnsignedLong(u[n]) : PyLong_FromLongLong(i[n]);
        if (!v) {
            Py_DECREF(t);
            return nullptr;
        }
        PyTuple_SET_ITEM(t, n, v);
    }
    return t;
}

// the tensor that a descriptor the library filled in describes: a view of `cache`'s memory
PyObject *cache_tensor(PyObject *cache, PyObject *device, PyObject *dtype, const fhip_tensor4 &c) {
    Ref ptr(PyLong_FromUnsignedLongLong((uintptr_t)c.ptr));
    if (!ptr.o) return nullptr;
    PyObject *vv[3] = {device, ptr.o, cache};
    Ref v(instance(view, 3, vv)), shape(tuple4(c.shape, nullptr)), strides(tuple4(nullptr, c.stride)),
        offset(PyLong_FromUnsignedLongLong(c.offset));
    if (!v.o || !shape.o || !strides.o || !offset.o) return nullptr;
    PyObject *tv[5] = {v.o, dtype, shape.o, strides.o, offset.o};
    return instance(tensor, 5, tv);
}

// The descriptor of attention(q, k, v, scale, mask, analytic, kv_lens, out_dtype, force_kernel, out), without a workspace (and without a
// result where `out` is None), and the device (a new reference) of a plain call.
PyObject *attention_args(PyObject *const *a, fhip_attn_args *args) {
    memset(args, 0, sizeof(*args));
    if (Py_TYPE(a[0]) != tensor.type || !slot(tensor, a[0], 0)) return nullptr;
    const Ref memory(Py_NewRef(slot(tensor, a[0], 0)));
    Ref device(PyObject_GetAttr(memory.o, n_device));
    if (!device.o) {
        not_plain();
        return nullptr;
    }
    int32_t dtypes[4], mask_dtype, kind;
    if (!describe<4>(a[0], &args->q, &dtypes[0], nullptr) || !describe<4>(a[1], &args->k, &dtypes[1], device.o) ||
        !describe<4>(a[2], &args->v, &dtypes[2], device.o) || (a[9] != Py_None && !describe<4>(a[9], &args->out, &dtypes[3], nullptr)) ||
        dtypes[1] != dtypes[0] || dtypes[2] != dtypes[0])
        return nullptr;
    args->dtype = (fhip_dtype)dtypes[0];
    int32_t out_dtype = dtypes[0];
    if ((a[7] != Py_None && !as_narrow(a[7], &out_dtype)) || !PyFloat_Check(a[3]) || !as_narrow(a[8], &args->force_kernel)) return nullptr;
    args->out_dtype = (fhip_dtype)out_dtype;
    const double scale = PyFloat_AS_DOUBLE(a[3]);
    if (!(std::fabs(scale) < 1e38)) return nullptr;
    args->scale = (float)scale;
    if (a[4] != Py_None) {
        if (!PyTuple_CheckExact(a[4]) || PyTuple_GET_SIZE(a[4]) < 2 || PyTuple_GET_SIZE(a[4]) > 3) return nullptr;
        if (!describe<2>(PyTuple_GET_ITEM(a[4], 0), &args->mask, &mask_dtype, device.o) || mask_dtype != dtypes[0] ||
            !as_narrow(PyTuple_GET_ITEM(a[4], 1), &kind))
            return nullptr;
        args->mask_kind = (fhip_mask_kind)kind;
        if (PyTuple_GET_SIZE(a[4]) == 3) {
            Ref memory(PyObject_GetAttr(PyTuple_GET_ITEM(a[4], 2), n_buffer));
            uint64_t ptr;
            if (!memory.o || !attr_u64(memory.o, n_ptr, &ptr)) {
                not_plain();
                return nullptr;
            }
            args->mask_intervals = (const void *)(uintptr_t)ptr;
        }
    }
    if (a[5] != Py_None) {
        if (!PyTuple_CheckExact(a[5]) || PyTuple_GET_SIZE(a[5]) != 3 || !PyBool_Check(PyTuple_GET_ITEM(a[5], 0)) ||
            !as_i64(PyTuple_GET_ITEM(a[5], 1), &args->analytic.q_pos_offset) || !as_i64(PyTuple_GET_ITEM(a[5], 2), &args->analytic.window))
            return nullptr;
        args->analytic.enabled = 1;
        args->analytic.causal = PyTuple_GET_ITEM(a[5], 0) == Py_True;
    }
    if (a[6] != Py_None) {
        if (Py_TYPE(a[6]) != lens_type) return nullptr;
        Ref dtype(PyObject_GetAttr(a[6], n_dtype)), shape(PyObject_GetAttr(a[6], n_shape)), memory(PyObject_GetAttr(a[6], n_buffer));
        uint64_t ptr, offset;
        uint32_t sequences;
        if (!dtype.o || !shape.o || !memory.o || !PyUnicode_Check(dtype.o) || PyUnicode_Compare(dtype.o, s_i32) != 0 ||
            !PyTuple_CheckExact(shape.o) || PyTuple_GET_SIZE(shape.o) != 1 || !as_narrow(PyTuple_GET_ITEM(shape.o, 0), &sequences) ||
            sequences != args->q.shape[0] || !attr_u64(memory.o, n_ptr, &ptr) || !attr_u64(a[6], n_offset, &offset)) {
            not_plain();
            return nullptr;
        }
        args->kv_lens = (const int32_t *)(uintptr_t)ptr + offset;
    }
    Py_INCREF(device.o);
    return device.o;
}

// attention_descriptor(...): the bytes of what `attention` hands to the library, or None (for tests; nothing is called)
PyObject *attention_descriptor(PyObject *, PyObject *const *a, Py_ssize_t n) {
    fhip_attn_args args;
    if (n != 10 || a[9] == Py_None) Py_RETURN_NONE;
    Ref device(attention_args(a, &args));
    if (!device.o) Py_RETURN_NONE;
    return PyBytes_FromStringAndSize((const char *)&args, sizeof(args));
}

bool norm_of(PyObject *o, fhip_rms_norm *out) {
    if (Py_TYPE(o) != norm_type) return false;
    void *weight, *bias = nullptr;
    if (!attr_memory(o, n_weight, &weight)) return false;
    Ref b(PyObject_GetAttr(o, n_bias)), dtype(PyObject_GetAttr(o, n_dtype)), eps(PyObject_GetAttr(o, n_eps));
    int32_t type;
    if (!b.o || !dtype.o || !eps.o || !as_narrow(dtype.o, &type) || !PyFloat_Check(eps.o) || !(std::fabs(PyFloat_AS_DOUBLE(eps.o)) < 1e38) ||
        (b.o != Py_None && !attr_memory(o, n_bias, &bias)))
        return not_plain();
    out->weight = weight, out->bias = bias, out->dtype = (fhip_dtype)type, out->eps = (float)PyFloat_AS_DOUBLE(eps.o);
    return true;
}

struct AppendArgs {
    fhip_tensor4 q, q_out, k, v;
    int32_t q_dtype, out_dtype, k_dtype, v_dtype;
    fhip_rope_tables tables;
    fhip_rms_norm q_norm, k_norm;
};

// The descriptors of append(cache, rope, q, q_out, k, v, start_pos, interleaved, q_norm, k_norm)
bool append_args(PyObject *const *a, Py_ssize_t n, AppendArgs *c) {
    memset(c, 0, sizeof(*c));
    void *cos, *sin;
    if (n != 10 || Py_TYPE(a[0]) != cache_type || Py_TYPE(a[1]) != rope_type || !PyBool_Check(a[7]) ||
        !describe<4>(a[2], &c->q, &c->q_dtype, nullptr) || !describe<4>(a[3], &c->q_out, &c->out_dtype, nullptr) ||
        !describe<4>(a[4], &c->k, &c->k_dtype, nullptr) || !describe<4>(a[5], &c->v, &c->v_dtype, nullptr) || c->k_dtype != c->v_dtype ||
        !attr_memory(a[1], n_cos, &cos) || !attr_memory(a[1], n_sin, &sin) || !attr_u64(a[1], n_rows, &c->tables.table_rows) ||
        !as_u64(a[6], &c->tables.start_pos) || (a[8] != Py_None && !norm_of(a[8], &c->q_norm)) ||
        (a[9] != Py_None && !norm_of(a[9], &c->k_norm)))
        return false;
    c->tables.cos = (const float *)cos, c->tables.sin = (const float *)sin, c->tables.interleaved = a[7] == Py_True;
    return true;
}

// append(...): (status, keys, values), or None
PyObject *append(PyObject *, PyObject *const *a, Py_ssize_t n) {
    AppendArgs c;
    fhip_tensor4 keys, values;
    void *handle, *stream;
    if (!append_args(a, n, &c)) Py_RETURN_NONE;
    Ref device(PyObject_GetAttr(a[0], n_device)), dtype(PyObject_GetAttr(a[0], n_dtype));
    if (!device.o || !dtype.o || !attr_handle(a[0], n_handle, &handle) || !attr_handle(device.o, n_stream, &stream)) {
        not_plain();
        Py_RETURN_NONE;
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fhip_kv_cache_qkv_rope_append((fhip_kv_cache *)handle, (fhip_stream *)stream, a[8] != Py_None ? &c.q_norm : nullptr,
                                       a[9] != Py_None ? &c.k_norm : nullptr, &c.tables, &c.q, (fhip_dtype)c.q_dtype, &c.q_out,
                                       (fhip_dtype)c.out_dtype, &c.k, &c.v, (fhip_dtype)c.k_dtype, &keys, &values);
    Py_END_ALLOW_THREADS
    if (rc != FHIP_OK) return Py_BuildValue("iOO", rc, Py_None, Py_None);
    Ref tkeys(cache_tensor(a[0], device.o, dtype.o, keys)), tvalues(cache_tensor(a[0], device.o, dtype.o, values));
    if (!tkeys.o || !tvalues.o) return nullptr;
    return Py_BuildValue("iOO", rc, tkeys.o, tvalues.o);
}

// append_descriptors(...): the bytes of what `append` hands to the library (q, q_out, k, v, dtypes, tables, norms), or None (for tests)
PyObject *append_descriptors(PyObject *, PyObject *const *a, Py_ssize_t n) {
    AppendArgs c;
    if (!append_args(a, n, &c)) Py_RETURN_NONE;
    return PyBytes_FromStringAndSize((const char *)&c, sizeof(c));
}

// contiguous(Buffer, device, bytes of an element, dtype, shape): a Tensor of that shape on memory of its own, or None
PyObject *contiguous(PyObject *, PyObject *const *a, Py_ssize_t n) {
    uint32_t element;
    if (n != 5 || !as_narrow(a[2], &element) || !PyTuple_CheckExact(a[4])) Py_RETURN_NONE;
    const Py_ssize_t rank = PyTuple_GET_SIZE(a[4]);
    Ref strides(PyTuple_New(rank));
    if (!strides.o) return nullptr;
    int64_t count = 1;
    for (Py_ssize_t i = rank - 1; i >= 0; i--) {
        uint32_t extent;
        PyObject *const e = PyTuple_GET_ITEM(a[4], i);
        if (!PyLong_CheckExact(e) || !as_narrow(e, &extent)) Py_RETURN_NONE;
        PyObject *const stride = PyLong_FromLongLong(count);
        if (!stride) return nullptr;
        PyTuple_SET_ITEM(strides.o, i, stride);
        if (__builtin_mul_overflow(count, (int64_t)extent, &count) || count > ((int64_t)1 << 56)) Py_RETURN_NONE;
    }
    Ref bytes(PyLong_FromLongLong(count * element)), zero(PyLong_FromLong(0));
    if (!bytes.o || !zero.o) return nullptr;
    PyObject *const of[2] = {a[1], bytes.o};
    Ref buffer(PyObject_Vectorcall(a[0], of, 2, nullptr));
    if (!buffer.o) return nullptr;
    PyObject *const values[5] = {buffer.o, a[3], a[4], strides.o, zero.o};
    return instance(tensor, 5, values);
}

// a Tensor of q's shape for a result of that type (a new reference, None where it is left to the general way, null with an exception)
PyObject *result(PyObject *buffer_type, PyObject *device, PyObject *q, fhip_dtype dtype) {
    if (dtype != FHIP_F32 && dtype != FHIP_F16 && dtype != FHIP_BF16) Py_RETURN_NONE;
    Ref element(PyLong_FromLong(dtype == FHIP_F32 ? 4 : 2)), type(PyLong_FromLong(dtype)), shape(Py_NewRef(slot(tensor, q, 2)));
    if (!element.o || !type.o) return nullptr;
    PyObject *const of[5] = {buffer_type, device, element.o, type.o, shape.o};
    return contiguous(nullptr, of, 5);
}

// attention(q, k, v, scale, mask, analytic, kv_lens, out_dtype, force_kernel, out, Buffer): the library's status, or None.  Where `out` is
// None, the result (on memory of its own, once the arguments have been looked at) instead of the status 0.
PyObject *attention(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 11) Py_RETURN_NONE;
    fhip_attn_args args;
    void *stream;
    uint64_t cus;
    Ref device(attention_args(a, &args));
    if (!device.o || !attr_handle(device.o, n_stream, &stream) || !attr_u64(device.o, n_compute_units, &cus)) Py_RETURN_NONE;
    Ref made(a[9] == Py_None ? result(a[10], device.o, a[0], args.out_dtype) : nullptr);
    if (a[9] == Py_None) {
        int32_t dtype;
        if (!made.o) return nullptr;
        if (made.o == Py_None || !describe<4>(made.o, &args.out, &dtype, nullptr)) Py_RETURN_NONE;
    }
    size_t need = 0;
    int rc = fhip_flash_attention_workspace_bytes(&args, (int32_t)cus, &need);
    if (rc == FHIP_OK && need) {
        Ref bytes(PyLong_FromSize_t(need));
        if (!bytes.o) return nullptr;
        Ref ws(PyObject_CallMethodOneArg(device.o, n_workspace, bytes.o));
        if (!ws.o) return nullptr;  // what the caller's own call of it would raise
        uint64_t ptr, size;
        if (!PyTuple_CheckExact(ws.o) || PyTuple_GET_SIZE(ws.o) != 2 || !as_u64(PyTuple_GET_ITEM(ws.o, 0), &ptr) ||
            !as_u64(PyTuple_GET_ITEM(ws.o, 1), &size))
            Py_RETURN_NONE;
        args.workspace = (void *)(uintptr_t)ptr;
        args.workspace_bytes = size;
    }
    if (rc == FHIP_OK) {
        Py_BEGIN_ALLOW_THREADS
        rc = fhip_flash_attention((fhip_stream *)stream, &args);
        Py_END_ALLOW_THREADS
    }
    if (rc == FHIP_OK && made.o) return Py_NewRef(made.o);
    return PyLong_FromLong(rc);
}

bool find(Slots *s, PyObject *type, int n, const char *const *names) {
    s->type = (PyTypeObject *)type;
    for (int i = 0; i < n; i++) {
        Ref d(PyObject_GetAttrString(type, names[i]));
        if (!d.o) return false;
        if (Py_TYPE(d.o) != &PyMemberDescr_Type || ((PyMemberDescrObject *)d.o)->d_member->type != T_OBJECT_EX) {
            PyErr_Format(PyExc_TypeError, "%s.%s is not a slot", s->type->tp_name, names[i]);
            return false;
        }
        s->at[i] = ((PyMemberDescrObject *)d.o)->d_member->offset;
    }
    return true;
}

// bind(Tensor, _View, KvCache, RopeCache, RmsNorm, IntTensor): once, with the module's classes
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    static const char *const of_tensor[] = {"buffer", "dtype", "shape", "strides", "offset"}, *const of_view[] = {"device", "ptr", "keepalive"};
    if (n != 6) return PyErr_Format(PyExc_TypeError, "bind takes six classes");
    for (int i = 0; i < n; i++) {
        if (!PyType_Check(a[i])) return PyErr_Format(PyExc_TypeError, "bind takes six classes");
        Py_INCREF(a[i]);  // (they live as long as the process)
    }
    if (!find(&tensor, a[0], 5, of_tensor) || !find(&view, a[1], 3, of_view)) return nullptr;
    cache_type = (PyTypeObject *)a[2], rope_type = (PyTypeObject *)a[3], norm_type = (PyTypeObject *)a[4], lens_type = (PyTypeObject *)a[5];
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void *)bind, METH_FASTCALL, nullptr},
    {"attention", (PyCFunction)(void *)attention, METH_FASTCALL, nullptr},
    {"contiguous", (PyCFunction)(void *)contiguous, METH_FASTCALL, nullptr},
    {"attention_descriptor", (PyCFunction)(void *)attention_descriptor, METH_FASTCALL, nullptr},
    {"append_descriptors", (PyCFunction)(void *)append_descriptors, METH_FASTCALL, nullptr},
    {"append", (PyCFunction)(void *)append, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    const struct {
        PyObject **name;
        const char *text;
    } names[] = {{&n_ptr, "ptr"},       {&n_device, "device"},   {&n_buffer, "buffer"}, {&n_offset, "offset"},
                 {&n_shape, "shape"},   {&n_dtype, "dtype"},     {&n_stream, "stream"}, {&n_value, "value"},
                 {&n_handle, "handle"}, {&n_cos, "cos"},         {&n_sin, "sin"},       {&n_rows, "rows"},
                 {&n_weight, "weight"}, {&n_bias, "bias"},       {&n_eps, "eps"},       {&n_compute_units, "compute_units"},
                 {&s_i32, "i32"},       {&n_workspace, "workspace"}};
    for (const auto &e : names)
        if (!(*e.name = PyUnicode_InternFromString(e.text))) return nullptr;
    return PyModule_Create(&module);
}
