// The calls a program makes in its inner loop, for HipExecutor (executor.py): Python objects straight to
// the C ABI.  A call through ctypes with numpy metadata spends 5 to 8 us on conversions (an array's
// data_as alone is more than 1 us), as much as a small kernel takes; here it is 0.3 to 0.5 us.
// Metadata may be anything numpy turns into an array of its type; what already is a contiguous array of
// that type is used where it lies.  The interpreter is released around every call: those that only encode
// may wait as well (a weight's first use, tables that wait for a slot), and what they are given is held
// by the caller's arguments.
#define PY_SSIZE_T_CLEAN
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <Python.h>
#include <numpy/arrayobject.h>

#include <stddef.h>
#include <stdint.h>

#include "../../include/mlc_hip.h"

namespace {

// One argument list being read: the first failure is remembered (as the Python error it set) and
// everything behind it reads as nothing.
class Args {
public:
    Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : args_(args) {
        if (n != want) {
            PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
            ok_ = false;
        }
    }
    ~Args() {
        for (int i = 0; i < n_held_; ++i) Py_DECREF(held_[i]);
    }
    bool ok() const { return ok_; }
    // a device pointer: an integer, or None for null
    void* ptr() {
        PyObject* o = next();
        if (!o || o == Py_None) return nullptr;
        const unsigned long long v = PyLong_CheckExact(o) ? PyLong_AsUnsignedLongLong(o) : as_index(o);
        if (v == (unsigned long long)-1 && PyErr_Occurred()) ok_ = false;
        return reinterpret_cast<void*>(static_cast<uintptr_t>(v));
    }
    size_t size() {
        PyObject* o = next();
        if (!o) return 0;
        const size_t v = PyLong_CheckExact(o) ? PyLong_AsSize_t(o) : (size_t)as_index(o);
        if (v == (size_t)-1 && PyErr_Occurred()) ok_ = false;
        return v;
    }
    int truth() {
        PyObject* o = next();
        if (!o) return 0;
        const int v = PyObject_IsTrue(o);
        if (v < 0) ok_ = false;
        return v > 0;
    }
    float real() {
        PyObject* o = next();
        if (!o) return 0.f;
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) ok_ = false;
        return (float)v;
    }
    const char* text() {
        PyObject* o = next();
        const char* v = o ? PyUnicode_AsUTF8(o) : nullptr;
        if (!v) ok_ = false;
        return v;
    }
    // host array of a numpy type: its first element and its size
    template <class T, int TYPE>
    const T* array(size_t* size) {
        PyObject* o = next();
        if (!o) return nullptr;
        if (!(PyArray_Check(o) && PyArray_TYPE((PyArrayObject*)o) == TYPE && PyArray_IS_C_CONTIGUOUS((PyArrayObject*)o) &&
              PyArray_ISALIGNED((PyArrayObject*)o) && PyArray_ISNOTSWAPPED((PyArrayObject*)o))) {
            o = PyArray_FROM_OTF(o, TYPE, NPY_ARRAY_C_CONTIGUOUS | NPY_ARRAY_ALIGNED | NPY_ARRAY_NOTSWAPPED | NPY_ARRAY_FORCECAST);
            if (!o) {
                ok_ = false;
                return nullptr;
            }
            held_[n_held_++] = o;
        }
        *size = (size_t)PyArray_SIZE((PyArrayObject*)o);
        return static_cast<const T*>(PyArray_DATA((PyArrayObject*)o));
    }
    const uint32_t* u32(size_t* size) { return array<uint32_t, NPY_UINT32>(size); }
    const uint32_t* u32_or_none(size_t* size) {
        if (ok_ && args_[i_] == Py_None) {
            ++i_;
            return nullptr;
        }
        return u32(size);
    }

private:
    PyObject* next() { return ok_ ? args_[i_++] : nullptr; }
    unsigned long long as_index(PyObject* o) {   // (numpy integers and the like)
        PyObject* whole = PyNumber_Index(o);
        if (!whole) {
            ok_ = false;
            return (unsigned long long)-1;
        }
        const unsigned long long v = PyLong_AsUnsignedLongLong(whole);
        Py_DECREF(whole);
        return v;
    }
    PyObject* const* args_;
    Py_ssize_t i_ = 0;
    bool ok_ = true;
    PyObject* held_[8];
    int n_held_ = 0;
};

// The result of an ABI call, made without the interpreter's lock, as a bool.
template <class F>
PyObject* answer(const Args& a, F&& call) {
    if (!a.ok()) return nullptr;
    int done = 0;
    Py_BEGIN_ALLOW_THREADS
    done = call();
    Py_END_ALLOW_THREADS
    return PyBool_FromLong(done);
}

#define MLC_CALL(name) PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t n)

MLC_CALL(begin) {
    const Args a(args, n, 0);
    return answer(a, [] { return mlc_hip_begin(); });
}
MLC_CALL(flush) {
    const Args a(args, n, 0);
    return answer(a, [] { return mlc_hip_flush(); });
}
// q, k_pages, v_pages, o, flat table, offsets, seq_lens, q_positions, batch, heads, kv_heads, head_dim, page size, causal, sync
MLC_CALL(attention) {
    Args a(args, n, 15);
    void *q = a.ptr(), *k = a.ptr(), *v = a.ptr(), *o = a.ptr();
    size_t n_flat = 0, n_off = 0, n_seq = 0, n_pos = 0;
    const uint32_t *flat = a.u32(&n_flat), *off = a.u32(&n_off), *seq = a.u32(&n_seq), *pos = a.u32(&n_pos);
    const size_t batch = a.size(), heads = a.size(), kv = a.size(), dim = a.size(), page = a.size();
    const int causal = a.truth(), sync = a.truth();
    // the reference rejects vectors of the wrong length (metal_runtime.mm:7747-7748)
    if (a.ok() && (n_off != batch + 1 || n_seq != batch || n_pos != batch)) Py_RETURN_FALSE;
    return answer(a, [=] { return mlc_hip_paged_attn_decode(q, k, v, o, flat, n_flat, off, seq, pos, batch, heads, kv, dim, page, causal, sync); });
}
// q, k_pages, v_pages, o, flat table, offsets, seq_lens, q_start, batch, chunk, heads, kv_heads, head_dim, page size, sync
MLC_CALL(prefill) {
    Args a(args, n, 15);
    void *q = a.ptr(), *k = a.ptr(), *v = a.ptr(), *o = a.ptr();
    size_t n_flat = 0, n_off = 0, n_seq = 0, n_start = 0;
    const uint32_t *flat = a.u32(&n_flat), *off = a.u32(&n_off), *seq = a.u32(&n_seq), *start = a.u32(&n_start);
    const size_t batch = a.size(), chunk = a.size(), heads = a.size(), kv = a.size(), dim = a.size(), page = a.size();
    const int sync = a.truth();
    if (a.ok() && (n_off != batch + 1 || n_seq != batch || n_start != batch)) Py_RETURN_FALSE;
    return answer(a, [=] { return mlc_hip_paged_attn_prefill(q, k, v, o, flat, n_flat, off, seq, start, batch, chunk, heads, kv, dim, page, sync); });
}
// page storage, page ids, slots, page size, kv_heads, head_dim, batch, src, sync
MLC_CALL(scatter_batched) {
    Args a(args, n, 9);
    void* pages = a.ptr();
    size_t n_ids = 0, n_slots = 0;
    const uint32_t *ids = a.u32(&n_ids), *slots = a.u32(&n_slots);
    const size_t page = a.size(), kv = a.size(), dim = a.size(), batch = a.size();
    void* src = a.ptr();
    const int sync = a.truth();
    if (a.ok() && (n_ids < batch || n_slots < batch || (sync && (n_ids != batch || n_slots != batch)))) Py_RETURN_FALSE;  // metal_runtime.mm:7243
    return answer(a, [=] { return mlc_hip_scatter_kv_paged_batched_f16(pages, ids, slots, page, kv, dim, batch, src, sync); });
}
// page storage, page table, page size, kv_heads, head_dim, tokens, start slot, src, dtype bytes
MLC_CALL(scatter) {
    Args a(args, n, 9);
    void* pages = a.ptr();
    size_t n_table = 0;
    const uint32_t* table = a.u32(&n_table);
    const size_t page = a.size(), kv = a.size(), dim = a.size(), tokens = a.size(), start = a.size();
    void* src = a.ptr();
    const size_t bytes = a.size();
    return answer(a, [=] { return mlc_hip_scatter_kv_paged(pages, table, n_table, page, kv, dim, tokens, start, src, bytes); });
}
// page storage, page table, page size, kv_heads, head_dim, tokens, dst, dtype bytes
MLC_CALL(gather) {
    Args a(args, n, 8);
    void* pages = a.ptr();
    size_t n_table = 0;
    const uint32_t* table = a.u32(&n_table);
    const size_t page = a.size(), kv = a.size(), dim = a.size(), tokens = a.size();
    void* dst = a.ptr();
    const size_t bytes = a.size();
    return answer(a, [=] { return mlc_hip_gather_kv_pages(pages, table, n_table, page, kv, dim, tokens, dst, bytes); });
}
// qkv, q, k, v, k_f16, v_f16, cos, sin, batch, heads, kv_heads, head_dim, qkv_rows, q_rows, k_rows, v_rows, rotary_dim, sync
MLC_CALL(rope_cast) {
    Args a(args, n, 18);
    void* p[8];
    size_t d[9];
    for (void*& x : p) x = a.ptr();
    for (size_t& x : d) x = a.size();
    const int sync = a.truth();
    return answer(a, [&] {
        return mlc_hip_qkv_split_rope_cast(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7], d[8], sync);
    });
}
// in, weight, epsilon, batch, length, out, sync
MLC_CALL(rms_norm) {
    Args a(args, n, 7);
    void* in = a.ptr();
    size_t n_weight = 0;
    const float* weight = a.array<float, NPY_FLOAT32>(&n_weight);
    const float eps = a.real();
    const size_t batch = a.size(), length = a.size();
    void* out = a.ptr();
    const int sync = a.truth();
    return answer(a, [=] { return mlc_hip_rms_norm_batched(in, n_weight ? weight : nullptr, n_weight, eps, batch, length, out, sync); });
}
// a, b, out, elements, sync
MLC_CALL(add) {
    Args a(args, n, 5);
    void *x = a.ptr(), *y = a.ptr(), *out = a.ptr();
    const size_t count = a.size();
    const int sync = a.truth();
    return answer(a, [=] { return mlc_hip_add_batched(x, y, out, count, sync); });
}
// gate_up, gate, up, out, batch, ffn_inner, gate_up rows, sync
MLC_CALL(gate_up) {
    Args a(args, n, 8);
    void *gu = a.ptr(), *gate = a.ptr(), *up = a.ptr(), *out = a.ptr();
    const size_t batch = a.size(), inner = a.size(), rows = a.size();
    const int sync = a.truth();
    return answer(a, [=] { return mlc_hip_gate_up_split_silu_mul(gu, gate, up, out, batch, inner, rows, sync); });
}
// name, weights, in, batch, rows, cols, row stride, quant version, out, sync
MLC_CALL(matmul_q4_0) {
    Args a(args, n, 10);
    const char* name = a.text();
    size_t n_bytes = 0;
    const uint8_t* w = a.array<uint8_t, NPY_UINT8>(&n_bytes);
    void* in = a.ptr();
    const size_t batch = a.size(), rows = a.size(), cols = a.size(), stride = a.size(), version = a.size();
    void* out = a.ptr();
    const int sync = a.truth();
    return answer(a, [=] { return mlc_hip_matmul_q4_0_batched(name, w, n_bytes, in, batch, rows, cols, stride, (uint32_t)version, out, sync); });
}
// name, weights, in, batch, rows, cols, row stride, out, sync
MLC_CALL(matmul_q6_k) {
    Args a(args, n, 9);
    const char* name = a.text();
    size_t n_bytes = 0;
    const uint8_t* w = a.array<uint8_t, NPY_UINT8>(&n_bytes);
    void* in = a.ptr();
    const size_t batch = a.size(), rows = a.size(), cols = a.size(), stride = a.size();
    void* out = a.ptr();
    const int sync = a.truth();
    return answer(a, [=] { return mlc_hip_matmul_q6_k_batched(name, w, n_bytes, in, batch, rows, cols, stride, out, sync); });
}
// handle, flat table, offsets, seq_lens, q_positions, page ids or None, slots or None
MLC_CALL(replay_update) {
    Args a(args, n, 7);
    const size_t handle = a.size();
    size_t n_flat = 0, batch = 0, unused = 0;
    const uint32_t *flat = a.u32(&n_flat), *off = a.u32(&unused), *seq = a.u32(&batch), *pos = a.u32(&unused);
    const uint32_t *ids = a.u32_or_none(&unused), *slots = a.u32_or_none(&unused);
    return answer(a, [=] { return mlc_hip_replay_update((int)handle, flat, n_flat, off, seq, pos, ids, slots, batch); });
}
MLC_CALL(replay) {
    Args a(args, n, 1);
    const size_t handle = a.size();
    return answer(a, [=] { return mlc_hip_replay((int)handle); });
}
#undef MLC_CALL

#define MLC_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    MLC_METHOD(begin),    MLC_METHOD(flush), MLC_METHOD(attention), MLC_METHOD(prefill), MLC_METHOD(scatter_batched),
    MLC_METHOD(scatter),  MLC_METHOD(gather), MLC_METHOD(rope_cast), MLC_METHOD(rms_norm), MLC_METHOD(add),
    MLC_METHOD(gate_up),  MLC_METHOD(matmul_q4_0), MLC_METHOD(matmul_q6_k), MLC_METHOD(replay_update), MLC_METHOD(replay),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", "HipExecutor's inner-loop calls into libmlc_hip.so", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    import_array();
    return PyModule_Create(&module);
}
