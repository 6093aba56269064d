// The torch front end's ordinary calls (attention.py: attention,
// attention_fused) without their Python: one function call checks the
// tensors, allocates the output and calls the C ABI.  An eager decode or
// verification layer is two kernels of 7 to 19 us; checked and launched from
// Python through ctypes it took the host 16-18 us (raw) and 31 us (a session's
// layer), so the GPU waited for the host.  Of that the two launches
// themselves are about 7 us.
//
// Every function returns None, before anything is enqueued, for a call that
// it does not take (a tensor subclass, a tensor that needs a copy, a wrong
// type, shape or device, a call off the GPU); attention.py then does the same
// in Python, copies included, or raises its error.  An error of the library
// is raised here, as redshift_amd.runtime.check raises it.
//
// Tensors are read through their public metadata; nothing is kept between
// calls but the library's function pointers.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <limits>
#include <optional>

namespace {

using Attention = int (*)(void *, const void *, const void *, const void *, int, int, int, int, int, int, int, int,
                          float, void *, uint64_t, void *);
using AttentionWorkspace = int (*)(uint64_t *, int, int, int, int, int);
using Fused = int (*)(float *, void *, void *, const float *, const float *, const float *, const float *,
                      const float *, int, int, int, float, void *, uint64_t, void *);
using FusedWorkspace = int (*)(uint64_t *, int, int);
using Error = const char *(*)();

constexpr int kF16 = 1, kBF16 = 2, kF32 = 3;                       // include/runtime.h
constexpr int kQHeads = 24, kKvHeads = 4, kHeadDim = 256;          // the fused model
constexpr uint64_t kMinWorkspace = 256;

Attention attention = nullptr;
AttentionWorkspace attention_workspace = nullptr;
Fused fused = nullptr;
FusedWorkspace fused_workspace = nullptr;
Error last_error = nullptr;
PyObject *get_device = nullptr, *get_stream = nullptr;
PyObject *name_k, *name_v, *name_dtype, *name_kv_heads, *name_head_dim, *name_capacity;

// A call this module does not take.
struct NotTaken {};
void require(bool condition) {
    if (!condition) throw NotTaken{};
}

// A plain torch tensor (subclasses go to Python).
const at::Tensor &tensor(PyObject *o) {
    require(THPVariable_CheckExact(o));
    const at::Tensor &t = THPVariable_Unpack(o);
    require(t.defined() && t.layout() == at::kStrided && t.has_storage());
    return t;
}

int integer(PyObject *o) {
    require(PyLong_CheckExact(o));
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    require(!overflow && v >= std::numeric_limits<int>::min() && v <= std::numeric_limits<int>::max());
    return (int)v;
}

float real(PyObject *o) {
    require(PyFloat_Check(o));
    return (float)PyFloat_AS_DOUBLE(o);
}

struct Ref {
    PyObject *o;
    ~Ref() { Py_XDECREF(o); }
};

// A PagedKV's fields.
struct Cache {
    Ref k_ref, v_ref;
    at::Tensor k, v;
    at::ScalarType dtype;
    int kv_heads, head_dim, capacity;
    explicit Cache(PyObject *o)
        : k_ref{PyObject_GetAttr(o, name_k)}, v_ref{PyObject_GetAttr(o, name_v)} {
        require(k_ref.o && v_ref.o);
        k = tensor(k_ref.o);
        v = tensor(v_ref.o);
        require(k.is_cuda() && v.device() == k.device());
        Ref d{PyObject_GetAttr(o, name_dtype)};
        require(d.o && THPDtype_Check(d.o));
        dtype = reinterpret_cast<THPDtype *>(d.o)->scalar_type;
        kv_heads = field(o, name_kv_heads);
        head_dim = field(o, name_head_dim);
        capacity = field(o, name_capacity);
    }
    static int field(PyObject *o, PyObject *name) {
        Ref f{PyObject_GetAttr(o, name)};
        require(f.o);
        return integer(f.o);
    }
};

// torch's current stream, as torch.cuda.current_stream() gives it.
void *current_stream() {
    Ref device{PyObject_CallNoArgs(get_device)};
    require(device.o);
    Ref stream{PyObject_CallOneArg(get_stream, device.o)};
    require(stream.o);
    void *s = PyLong_AsVoidPtr(stream.o);
    require(!PyErr_Occurred());
    return s;
}

PyObject *raise_library_error() {
    const char *message = last_error();
    Ref text{PyUnicode_DecodeUTF8(message, (Py_ssize_t)strlen(message), "replace")};
    if (text.o) PyErr_SetObject(PyExc_RuntimeError, text.o);
    return nullptr;
}

// Runs `call`; None when it takes no such call.
template <class Call>
PyObject *taken(Call call) {
    try {
        return call();
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// The caller's workspace, or one of `bytes` on `like`'s device.
at::Tensor workspace_of(PyObject *given, uint64_t bytes, const at::Tensor &like) {
    if (given != Py_None) return tensor(given);
    return at::empty({(int64_t)std::max(bytes, kMinWorkspace)}, like.options().dtype(at::kByte));
}

int code_of(at::ScalarType t) {
    require(t == at::kHalf || t == at::kBFloat16);
    return t == at::kHalf ? kF16 : kBF16;
}

// attention(q, cache, position, scale, out, ws, out_dtype)
PyObject *py_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return taken([&]() -> PyObject * {
        require(n == 7 && attention);
        const at::Tensor &q = tensor(args[0]);
        const Cache cache(args[1]);
        const int position = integer(args[2]);
        const float scale = real(args[3]);
        require(q.dim() == 3 && q.scalar_type() == cache.dtype && q.size(2) == cache.head_dim &&
                q.device() == cache.k.device() && q.is_contiguous());
        require(q.size(0) <= std::numeric_limits<int>::max() && q.size(1) <= std::numeric_limits<int>::max());
        const int tokens = (int)q.size(0), q_heads = (int)q.size(1), dtype = code_of(cache.dtype);
        at::Tensor out;
        if (args[4] != Py_None) {
            out = tensor(args[4]);
            require(out.sizes() == q.sizes() && out.is_contiguous() && out.device() == q.device());
        } else {
            at::ScalarType t = cache.dtype;
            if (args[6] != Py_None) {
                require(THPDtype_Check(args[6]));
                t = reinterpret_cast<THPDtype *>(args[6])->scalar_type;
            }
            require(t == cache.dtype || t == at::kFloat);
            out = at::empty(q.sizes(), q.options().dtype(t));
        }
        require(out.scalar_type() == cache.dtype || out.scalar_type() == at::kFloat);
        uint64_t bytes = 0;
        if (args[5] == Py_None && attention_workspace(&bytes, q_heads, cache.kv_heads, cache.head_dim, tokens, position))
            return raise_library_error();
        const at::Tensor ws = workspace_of(args[5], bytes, q);
        require(ws.device() == q.device());
        void *stream = current_stream();
        const int out_code = out.scalar_type() == at::kFloat ? kF32 : dtype;
        void *o = out.data_ptr(), *w = ws.data_ptr();
        const void *qp = q.data_ptr(), *k = cache.k.data_ptr(), *v = cache.v.data_ptr();
        const uint64_t ws_bytes = (uint64_t)ws.nbytes();
        int code;
        Py_BEGIN_ALLOW_THREADS
        code = attention(o, qp, k, v, dtype, out_code, q_heads, cache.kv_heads, cache.head_dim, tokens, position,
                         cache.capacity, scale, w, ws_bytes, stream);
        Py_END_ALLOW_THREADS
        if (code) return raise_library_error();
        if (args[4] != Py_None) return Py_NewRef(args[4]);
        return THPVariable_Wrap(std::move(out));
    });
}

// attention_fused(q_gate, key, value, q_norm, k_norm, cache, position, epsilon, out, ws)
PyObject *py_attention_fused(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return taken([&]() -> PyObject * {
        require(n == 10 && fused);
        const Cache cache(args[5]);
        const int position = integer(args[6]);
        const float epsilon = real(args[7]);
        require(cache.dtype == at::kHalf && cache.kv_heads == kKvHeads && cache.head_dim == kHeadDim);
        const at::Tensor &q_gate = tensor(args[0]);
        require(q_gate.dim() >= 1 && q_gate.size(0) <= std::numeric_limits<int>::max());
        const int64_t batch = q_gate.size(0);
        const int64_t numel[5] = {batch * kQHeads * 2 * kHeadDim, batch * kKvHeads * kHeadDim,
                                  batch * kKvHeads * kHeadDim, kHeadDim, kHeadDim};
        const float *in[5];
        for (int i = 0; i < 5; ++i) {
            const at::Tensor &t = tensor(args[i]);
            require(t.scalar_type() == at::kFloat && t.numel() == numel[i] && t.device() == cache.k.device() &&
                    t.is_contiguous());
            in[i] = static_cast<const float *>(t.data_ptr());
            require(reinterpret_cast<uintptr_t>(in[i]) % 16 == 0);
        }
        at::Tensor out;
        if (args[8] != Py_None) {
            out = tensor(args[8]);
            require(out.scalar_type() == at::kFloat && out.numel() == batch * kQHeads * kHeadDim &&
                    out.is_contiguous() && out.device() == cache.k.device());
        } else {
            out = at::empty({batch, kQHeads, kHeadDim}, q_gate.options());
        }
        uint64_t bytes = 0;
        if (args[9] == Py_None && fused_workspace(&bytes, (int)batch, position)) return raise_library_error();
        const at::Tensor ws = workspace_of(args[9], bytes, q_gate);
        require(ws.device() == cache.k.device());
        void *stream = current_stream();
        float *o = static_cast<float *>(out.data_ptr());
        void *k = cache.k.data_ptr(), *v = cache.v.data_ptr(), *w = ws.data_ptr();
        const uint64_t ws_bytes = (uint64_t)ws.nbytes();
        int code;
        Py_BEGIN_ALLOW_THREADS
        code = fused(o, k, v, in[0], in[1], in[2], in[3], in[4], (int)batch, position, cache.capacity, epsilon, w,
                     ws_bytes, stream);
        Py_END_ALLOW_THREADS
        if (code) return raise_library_error();
        if (args[8] != Py_None) return Py_NewRef(args[8]);
        return THPVariable_Wrap(std::move(out));
    });
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
    attention = reinterpret_cast<Attention>(f[0]);
    attention_workspace = reinterpret_cast<AttentionWorkspace>(f[1]);
    fused = reinterpret_cast<Fused>(f[2]);
    fused_workspace = reinterpret_cast<FusedWorkspace>(f[3]);
    last_error = reinterpret_cast<Error>(f[4]);
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
