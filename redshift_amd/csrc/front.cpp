// The torch front end's ordinary calls (attention.py: attention,
// attention_fused) without their Python: one function call checks the
// tensors, allocates the output and calls the C ABI.  An eager decode or
// verification layer is two kernels of 7 to 19 us; checked and launched from
// Python through ctypes it took the host 16-18 us (raw) and 31 us (a session's
// layer), so the GPU waited for the host.  Of that the C call itself is about
// 4 us for one launch and 8 for two.
//
// Every function returns None, before anything is enqueued, for a call that
// it does not take (a tensor subclass, which nn.Parameter is not here, a tensor
// that needs a copy, a wrong type, shape or device, a call off the GPU);
// attention.py then does the same in Python, copies included, or raises its
// error.  No exception is thrown for a refusal, which would cost the call 2 us
// (a strided query 20.4 against 18.2 us of host time, 19.4 in Python alone).  An
// error of the library is raised here, as redshift_amd.runtime.check raises it.
//
// Tensors are read through their public metadata; nothing is kept between
// calls but the library's function pointers.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <limits>
#include <utility>

#include "runtime.h"

namespace {

constexpr int kQHeads = 24, kKvHeads = 4, kHeadDim = 256;          // the fused model
constexpr uint64_t kMinWorkspace = 256;

decltype(&qv_attention) attention = nullptr;
decltype(&qv_attention_workspace) attention_workspace = nullptr;
decltype(&qv_attention_fused) fused = nullptr;
decltype(&qv_attention_fused_workspace) fused_workspace = nullptr;
decltype(&qv_error) last_error = nullptr;
PyObject *get_device = nullptr, *get_stream = nullptr;
PyObject *name_k, *name_v, *name_dtype, *name_kv_heads, *name_head_dim, *name_capacity;

// A call this module does not take.
PyObject *not_taken() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

// The readers below return false for what the module does not take.
// A plain torch tensor (subclasses go to Python).
bool tensor(PyObject *o, const at::Tensor *&t) {
    if (!THPVariable_CheckExact(o)) return false;
    t = &THPVariable_Unpack(o);
    return t->defined() && t->layout() == at::kStrided && t->has_storage();
}

bool integer(PyObject *o, int &value) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow || v < std::numeric_limits<int>::min() || v > std::numeric_limits<int>::max()) return false;
    value = (int)v;
    return true;
}

bool real(PyObject *o, float &value) {
    if (!PyFloat_Check(o)) return false;
    value = (float)PyFloat_AS_DOUBLE(o);
    return true;
}

struct Ref {
    PyObject *o = nullptr;
    ~Ref() { Py_XDECREF(o); }
};

// A PagedKV's fields (its tensors held while the call runs).
struct Cache {
    Ref k_ref, v_ref;
    const at::Tensor *k = nullptr, *v = nullptr;
    at::ScalarType dtype = at::ScalarType::Undefined;
    int kv_heads = 0, head_dim = 0, capacity = 0;

    bool read(PyObject *o) {
        k_ref.o = PyObject_GetAttr(o, name_k);
        v_ref.o = k_ref.o ? PyObject_GetAttr(o, name_v) : nullptr;
        if (!v_ref.o || !tensor(k_ref.o, k) || !tensor(v_ref.o, v)) return false;
        if (!k->is_cuda() || v->device() != k->device()) return false;
        Ref d{PyObject_GetAttr(o, name_dtype)};
        if (!d.o || !THPDtype_Check(d.o)) return false;
        dtype = reinterpret_cast<THPDtype *>(d.o)->scalar_type;
        return field(o, name_kv_heads, kv_heads) && field(o, name_head_dim, head_dim) &&
               field(o, name_capacity, capacity);
    }
    static bool field(PyObject *o, PyObject *name, int &value) {
        Ref f{PyObject_GetAttr(o, name)};
        return f.o && integer(f.o, value);
    }
};

// torch's current stream, as torch.cuda.current_stream() gives it.
bool current_stream(void *&stream) {
    Ref device{PyObject_CallNoArgs(get_device)};
    Ref s{device.o ? PyObject_CallOneArg(get_stream, device.o) : nullptr};
    if (!s.o) return false;
    stream = PyLong_AsVoidPtr(s.o);
    return !PyErr_Occurred();
}

// The call's allocations and launches run without the interpreter's lock, as
// torch.empty and ctypes run them: an allocation may wait for the device.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

PyObject *raise_library_error() {
    const char *message = last_error();
    Ref text{PyUnicode_DecodeUTF8(message, (Py_ssize_t)std::strlen(message), "replace")};
    if (text.o) PyErr_SetObject(PyExc_RuntimeError, text.o);
    return nullptr;
}

// A workspace of `bytes` on `like`'s device.
at::Tensor make_workspace(uint64_t bytes, const at::Tensor &like) {
    return at::empty({(int64_t)std::max(bytes, kMinWorkspace)}, like.options().dtype(at::kByte));
}

// attention(q, cache, position, scale, out, ws, out_dtype)
PyObject *py_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    constexpr int64_t kMost = std::numeric_limits<int>::max();
    const at::Tensor *q = nullptr, *out = nullptr, *ws = nullptr;
    Cache cache;
    int position = 0;
    float scale = 0.f;
    if (n != 7 || !attention || !tensor(args[0], q) || !cache.read(args[1]) || !integer(args[2], position) ||
        !real(args[3], scale))
        return not_taken();
    if (cache.dtype != at::kHalf && cache.dtype != at::kBFloat16) return not_taken();
    if (q->dim() != 3 || q->scalar_type() != cache.dtype || q->size(2) != cache.head_dim ||
        q->device() != cache.k->device() || !q->is_contiguous() || q->size(0) > kMost || q->size(1) > kMost)
        return not_taken();
    const int tokens = (int)q->size(0), q_heads = (int)q->size(1);
    at::ScalarType out_type = cache.dtype;
    if (args[4] != Py_None) {
        if (!tensor(args[4], out) || out->sizes() != q->sizes() || !out->is_contiguous() ||
            out->device() != q->device())
            return not_taken();
        out_type = out->scalar_type();
    } else if (args[6] != Py_None) {
        if (!THPDtype_Check(args[6])) return not_taken();
        out_type = reinterpret_cast<THPDtype *>(args[6])->scalar_type;
    }
    if (out_type != cache.dtype && out_type != at::kFloat) return not_taken();
    if (args[5] != Py_None && (!tensor(args[5], ws) || ws->device() != q->device())) return not_taken();
    void *stream = nullptr;
    if (!current_stream(stream)) return not_taken();
    const int dtype = cache.dtype == at::kHalf ? QV_F16 : QV_BF16, out_code = out_type == at::kFloat ? QV_F32 : dtype;
    int code = 0;
    at::Tensor made;
    try {
        const void *qp = q->data_ptr(), *k = cache.k->data_ptr(), *v = cache.v->data_ptr();
        void *o = out ? out->data_ptr() : nullptr, *w = ws ? ws->data_ptr() : nullptr;
        uint64_t bytes = ws ? (uint64_t)ws->nbytes() : 0;
        at::Tensor scratch;
        Unlocked unlocked;
        if (!out) {
            made = at::empty(q->sizes(), q->options().dtype(out_type));
            o = made.data_ptr();
        }
        if (!ws) {
            code = attention_workspace(&bytes, q_heads, cache.kv_heads, cache.head_dim, tokens, position);
            if (!code) {
                scratch = make_workspace(bytes, *q);
                w = scratch.data_ptr();
                bytes = (uint64_t)scratch.nbytes();
            }
        }
        if (!code)
            code = attention(o, qp, k, v, dtype, out_code, q_heads, cache.kv_heads, cache.head_dim, tokens, position,
                             cache.capacity, scale, w, bytes, stream);
    } catch (...) {
        return not_taken();   // nothing was launched (an allocation failed): Python raises it
    }
    if (code) return raise_library_error();
    return out ? Py_NewRef(args[4]) : THPVariable_Wrap(std::move(made));
}

// attention_fused(q_gate, key, value, q_norm, k_norm, cache, position, epsilon, out, ws)
PyObject *py_attention_fused(PyObject *, PyObject *const *args, Py_ssize_t n) {
    Cache cache;
    int position = 0;
    float epsilon = 0.f;
    if (n != 10 || !fused || !cache.read(args[5]) || !integer(args[6], position) || !real(args[7], epsilon))
        return not_taken();
    if (cache.dtype != at::kHalf || cache.kv_heads != kKvHeads || cache.head_dim != kHeadDim) return not_taken();
    const at::Tensor *t[5] = {}, *out = nullptr, *ws = nullptr;
    for (int i = 0; i < 5; ++i)
        if (!tensor(args[i], t[i])) return not_taken();
    if (t[0]->dim() < 1 || t[0]->size(0) > std::numeric_limits<int>::max()) return not_taken();
    const int64_t batch = t[0]->size(0);
    const int64_t numel[5] = {batch * kQHeads * 2 * kHeadDim, batch * kKvHeads * kHeadDim,
                              batch * kKvHeads * kHeadDim, kHeadDim, kHeadDim};
    for (int i = 0; i < 5; ++i)
        if (t[i]->scalar_type() != at::kFloat || t[i]->numel() != numel[i] || t[i]->device() != cache.k->device() ||
            !t[i]->is_contiguous())
            return not_taken();
    if (args[8] != Py_None &&
        (!tensor(args[8], out) || out->scalar_type() != at::kFloat || out->numel() != batch * kQHeads * kHeadDim ||
         !out->is_contiguous() || out->device() != cache.k->device()))
        return not_taken();
    if (args[9] != Py_None && (!tensor(args[9], ws) || ws->device() != cache.k->device())) return not_taken();
    void *stream = nullptr;
    if (!current_stream(stream)) return not_taken();
    int code = 0;
    at::Tensor made;
    try {
        const float *in[5];
        for (int i = 0; i < 5; ++i) {
            in[i] = static_cast<const float *>(t[i]->data_ptr());
            if (reinterpret_cast<uintptr_t>(in[i]) % 16) return not_taken();
        }
        void *k = cache.k->data_ptr(), *v = cache.v->data_ptr();
        float *o = out ? static_cast<float *>(out->data_ptr()) : nullptr;
        void *w = ws ? ws->data_ptr() : nullptr;
        uint64_t bytes = ws ? (uint64_t)ws->nbytes() : 0;
        at::Tensor scratch;
        Unlocked unlocked;
        if (!out) {
            made = at::empty({batch, kQHeads, kHeadDim}, t[0]->options());
            o = static_cast<float *>(made.data_ptr());
        }
        if (!ws) {
            code = fused_workspace(&bytes, (int)batch, position);
            if (!code) {
                scratch = make_workspace(bytes, *t[0]);
                w = scratch.data_ptr();
                bytes = (uint64_t)scratch.nbytes();
            }
        }
        if (!code)
            code = fused(o, k, v, in[0], in[1], in[2], in[3], in[4], (int)batch, position, cache.capacity, epsilon, w,
                         bytes, stream);
    } catch (...) {
        return not_taken();   // nothing was launched (an allocation failed): Python raises it
    }
    if (code) return raise_library_error();
    return out ? Py_NewRef(args[8]) : THPVariable_Wrap(std::move(made));
}

// bind(qv_attention, qv_attention_workspace, qv_attention_fused,
//      qv_attention_fused_workspace, qv_error, get_device, get_stream):
// function addresses, and torch's current device and raw stream functions.
PyObject *py_bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 7) {
        PyErr_SetString(PyExc_TypeError, "bind takes seven arguments");
        return nullptr;
    }
    void *f[5];
    for (int i = 0; i < 5; ++i) {
        f[i] = PyLong_AsVoidPtr(args[i]);
        if (!f[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null function address");
            return nullptr;
        }
    }
    attention = reinterpret_cast<decltype(attention)>(f[0]);
    attention_workspace = reinterpret_cast<decltype(attention_workspace)>(f[1]);
    fused = reinterpret_cast<decltype(fused)>(f[2]);
    fused_workspace = reinterpret_cast<decltype(fused_workspace)>(f[3]);
    last_error = reinterpret_cast<decltype(last_error)>(f[4]);
    Py_XSETREF(get_device, Py_NewRef(args[5]));
    Py_XSETREF(get_stream, Py_NewRef(args[6]));
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))py_bind, METH_FASTCALL, nullptr},
    {"attention", (PyCFunction)(void (*)(void))py_attention, METH_FASTCALL, nullptr},
    {"attention_fused", (PyCFunction)(void (*)(void))py_attention_fused, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "redshift_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_redshift_front(void) {
    name_k = PyUnicode_InternFromString("k");
    name_v = PyUnicode_InternFromString("v");
    name_dtype = PyUnicode_InternFromString("dtype");
    name_kv_heads = PyUnicode_InternFromString("kv_heads");
    name_head_dim = PyUnicode_InternFromString("head_dim");
    name_capacity = PyUnicode_InternFromString("capacity");
    return PyModule_Create(&module);
}
