// Per-call host path of the Python entry points, as a CPython extension over
// torch's C++ tensors.
//
// A small launch takes less time on the GPU than Python spends on checking
// its tensors and converting its arguments: 12 us of host work for a call of
// two kernels and 14 us more than here for an append of two, of which each
// launch itself takes 2.3 us (the C caller's figure).  Each object here is
// one entry point's call for a fixed configuration: it takes the common form
// of the arguments (plain GPU tensors of the expected shapes and types on the
// current device, Python floats and ints), checks exactly what the Python
// entry checks, allocates the outputs and calls the C ABI on the current
// stream.  For anything else it returns None, with nothing launched, and the
// Python entry goes on with its general path, conversions and error messages.
// A status of the C call other than PCPA_OK comes back as an int for the
// Python entry to raise: kernels may be queued by then, so the call is not made
// again.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <initializer_list>
#include <new>
#include <vector>

#include "pcp_attention_hip.h"

namespace {

// What the calls take and return, checked when the module is loaded (as is
// PCPA_TORCH_VERSION, the torch that the build line names).
constexpr int kVersion = 2;

PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream
PyObject* g_device = nullptr;      // torch._C._cuda_getDevice

// A plain torch.Tensor (no subclass), or nullptr.
const at::Tensor* plain(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool shaped(const at::Tensor& t, std::initializer_list<int64_t> shape) {
    return t.sizes() == at::IntArrayRef(shape.begin(), shape.size());
}

// A contiguous strided tensor of `type` on GPU `dev`.
bool on_gpu(const at::Tensor& t, at::ScalarType type, int dev) {
    return t.is_cuda() && t.get_device() == dev && t.scalar_type() == type && t.layout() == at::kStrided &&
           t.is_contiguous();
}

bool table_on(const at::Tensor& t, int dev) {
    return on_gpu(t, at::kInt, dev) || on_gpu(t, at::kLong, dev);
}

// The current device if it is `dev`, and its current stream; false otherwise
// (with any Python error cleared).
bool current_stream(int dev, void*& stream) {
    PyObject* d = PyObject_CallNoArgs(g_device);
    const long cur = d ? PyLong_AsLong(d) : -1;
    Py_XDECREF(d);
    if (cur != dev) {
        PyErr_Clear();
        return false;
    }
    PyObject* index = PyLong_FromLong(dev);
    PyObject* s = index ? PyObject_CallOneArg(g_raw_stream, index) : nullptr;
    Py_XDECREF(index);
    if (!s) {
        PyErr_Clear();
        return false;
    }
    stream = PyLong_AsVoidPtr(s);
    Py_DECREF(s);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

bool real(PyObject* o, float& x) {
    if (!PyFloat_CheckExact(o)) return false;
    x = (float)PyFloat_AS_DOUBLE(o);
    return true;
}

bool whole(PyObject* o, int64_t& x) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    x = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow;
}

// One entry point's call.
struct Call {
    PyObject_HEAD
    vectorcallfunc call;
    pcpa_params p;
    at::ScalarType kv_type;
    int32_t interleave;
    int dev;
    void* fn;
    // history
    int n_split;
    bool workspace;        // the split entry, with a workspace of ws_bytes
    int64_t ws_bytes;
    PyObject* ws_maker;    // f(bytes, stream) -> uint8 tensor
    struct Space {
        void* stream;
        at::Tensor tensor;
    };
    std::vector<Space>* spaces;
};

#define GIVE_UP Py_RETURN_NONE

using HistoryLse = decltype(&pcpa_history_attention_lse);
using HistorySplit = decltype(&pcpa_history_attention_split);
using Current = decltype(&pcpa_current_attention);
using Write = decltype(&pcpa_kv_cache_write);
using Alloc = decltype(&pcpa_page_alloc);

template <class F>
int32_t launch(F&& f) {
    int32_t status;
    Py_BEGIN_ALLOW_THREADS
    status = f();
    Py_END_ALLOW_THREADS
    return status;
}

PyObject* tensors(const at::Tensor& out, const at::Tensor& lse) {
    if (!lse.defined()) return THPVariable_Wrap(out);
    PyObject* a = THPVariable_Wrap(out);
    PyObject* b = THPVariable_Wrap(lse);
    PyObject* t = a && b ? PyTuple_Pack(2, a, b) : nullptr;
    Py_XDECREF(a);
    Py_XDECREF(b);
    return t;
}

// Forget the remembered workspaces.  Freeing a tensor can release the GIL, and
// another thread's call then looks through the same vector: it must find it
// whole, so the tensors are freed after they have left it.
void forget(Call* c) {
    std::vector<Call::Space> old;
    old.swap(*c->spaces);
}

// The workspace kept for `stream`: the Python object's (ws_maker), remembered
// here until it is told to forget.
void* workspace_for(Call* c, void* stream, at::Tensor& hold) {
    for (const Call::Space& s : *c->spaces)
        if (s.stream == stream) {
            hold = s.tensor;
            return hold.data_ptr();
        }
    PyObject* t = PyObject_CallFunction(c->ws_maker, "Ln", (long long)c->ws_bytes, (Py_ssize_t)(intptr_t)stream);
    if (!t) {
        // an interrupt is the caller's; errors are the general path's to meet
        if (PyErr_ExceptionMatches(PyExc_Exception)) PyErr_Clear();
        return nullptr;
    }
    hold = THPVariable_Unpack(t);
    Py_DECREF(t);
    if (c->spaces->size() >= 16) forget(c);
    c->spaces->push_back({stream, hold});
    return hold.data_ptr();
}

// (q, kv_pages, block_table, page_valid_len, k_scale, v_scale, out, return_lse) -> outputs or a status
PyObject* history(Call* c, PyObject* const* a) {
    const at::Tensor *q = plain(a[0]), *kv = plain(a[1]), *table = plain(a[2]), *valid = plain(a[3]);
    const at::Tensor* given = a[6] == Py_None ? nullptr : plain(a[6]);
    if (!q || !kv || !table || !valid || (a[6] != Py_None && !given)) GIVE_UP;
    pcpa_params p = c->p;
    if (!real(a[4], p.k_scale) || !real(a[5], p.v_scale) || !PyBool_Check(a[7])) GIVE_UP;
    const int dev = c->dev;
    const int64_t page = 2 * (int64_t)p.num_kv_heads * p.block_size * p.head_dim;
    if (!on_gpu(*q, at::kBFloat16, dev) || !shaped(*q, {p.pcp_size, p.num_q_heads, p.local_q_len, p.head_dim}) ||
        !on_gpu(*kv, c->kv_type, dev) || kv->dim() != 2 || kv->size(1) != page || kv->size(0) > INT32_MAX ||
        !table_on(*table, dev) || !shaped(*table, {p.pcp_size, p.max_local_blocks}) ||
        !on_gpu(*valid, at::kInt, dev) || !shaped(*valid, {p.pcp_size, p.max_local_blocks}))
        GIVE_UP;
    if (given && (!on_gpu(*given, at::kBFloat16, dev) || given->sizes() != q->sizes())) GIVE_UP;
    void* stream = nullptr;
    if (!current_stream(dev, stream)) GIVE_UP;
    p.num_pages = (int32_t)kv->size(0);
    if (table->scalar_type() == at::kLong) p.flags |= PCPA_FLAG_TABLE_INT64;
    const at::Tensor out = given ? *given : at::empty(q->sizes(), q->options().requires_grad(false));
    at::Tensor lse, ws;
    if (a[7] == Py_True)
        lse = at::empty({p.pcp_size, p.num_q_heads, p.local_q_len}, q->options().dtype(at::kFloat).requires_grad(false));
    float* const lse_ptr = lse.defined() ? (float*)lse.data_ptr() : nullptr;
    const void *qp = q->data_ptr(), *kp = kv->data_ptr(), *tp = table->data_ptr();
    const int32_t* const vp = (const int32_t*)valid->data_ptr();
    void* const op = out.data_ptr();
    int32_t status;
    if (c->workspace) {
        void* const w = workspace_for(c, stream, ws);
        if (!w) {
            if (PyErr_Occurred()) return nullptr;
            GIVE_UP;
        }
        status = launch([&] {
            return ((HistorySplit)c->fn)(&p, c->n_split, qp, kp, tp, vp, op, lse_ptr, w, c->ws_bytes, stream);
        });
    } else {
        status = launch([&] { return ((HistoryLse)c->fn)(&p, qp, kp, tp, vp, op, lse_ptr, stream); });
    }
    if (status) return PyLong_FromLong(status);
    return tensors(out, lse);
}

// (q, kv_current, hist_out, hist_lse, out, return_lse) -> outputs or a status
PyObject* current(Call* c, PyObject* const* a) {
    const at::Tensor *q = plain(a[0]), *kv = plain(a[1]);
    const at::Tensor* hist = a[2] == Py_None ? nullptr : plain(a[2]);
    const at::Tensor* hlse = a[3] == Py_None ? nullptr : plain(a[3]);
    const at::Tensor* given = a[4] == Py_None ? nullptr : plain(a[4]);
    if (!q || !kv || (a[2] != Py_None && !hist) || (a[3] != Py_None && !hlse) || (a[4] != Py_None && !given) ||
        !hist != !hlse || !PyBool_Check(a[5]) || !q->is_cuda())
        GIVE_UP;
    const pcpa_params& p = c->p;
    const int dev = q->get_device();
    const int64_t len = (int64_t)p.pcp_size * p.local_q_len;
    if (!on_gpu(*q, at::kBFloat16, dev) || !shaped(*q, {p.pcp_size, p.num_q_heads, p.local_q_len, p.head_dim}) ||
        !on_gpu(*kv, at::kBFloat16, dev) || !shaped(*kv, {2, p.num_kv_heads, len, p.head_dim}))
        GIVE_UP;
    if (hist && (!on_gpu(*hist, at::kBFloat16, dev) || hist->sizes() != q->sizes() ||
                 !on_gpu(*hlse, at::kFloat, dev) || !shaped(*hlse, {p.pcp_size, p.num_q_heads, p.local_q_len})))
        GIVE_UP;
    if (given && (!on_gpu(*given, at::kBFloat16, dev) || given->sizes() != q->sizes())) GIVE_UP;
    void* stream = nullptr;
    if (!current_stream(dev, stream)) GIVE_UP;
    const at::Tensor out = given ? *given : at::empty(q->sizes(), q->options().requires_grad(false));
    at::Tensor lse;
    if (a[5] == Py_True)
        lse = at::empty({p.pcp_size, p.num_q_heads, p.local_q_len}, q->options().dtype(at::kFloat).requires_grad(false));
    const void *qp = q->data_ptr(), *kp = kv->data_ptr(), *hp = hist ? hist->data_ptr() : nullptr;
    const float* const hl = hlse ? (const float*)hlse->data_ptr() : nullptr;
    void* const op = out.data_ptr();
    float* const lp = lse.defined() ? (float*)lse.data_ptr() : nullptr;
    const int32_t status =
        launch([&] { return ((Current)c->fn)(&p, c->interleave, qp, kp, hp, hl, op, lp, stream); });
    if (status) return PyLong_FromLong(status);
    return tensors(out, lse);
}

// (k, v, kv_pages, block_table, first_pos, k_scale, v_scale, page_valid_len) -> status
PyObject* write(Call* c, PyObject* const* a) {
    const at::Tensor *k = plain(a[0]), *v = plain(a[1]), *kv = plain(a[2]), *table = plain(a[3]);
    const at::Tensor* valid = a[7] == Py_None ? nullptr : plain(a[7]);
    pcpa_params p = c->p;
    int64_t first;
    if (!k || !v || !kv || !table || (a[7] != Py_None && !valid) || !whole(a[4], first) || first < 0 ||
        !real(a[5], p.k_scale) || !real(a[6], p.v_scale) || !k->is_cuda() || k->dim() != 3)
        GIVE_UP;
    const int dev = k->get_device();
    const int64_t page = 2 * (int64_t)p.num_kv_heads * p.block_size * p.head_dim, n = k->size(1);
    if (n > INT32_MAX || !on_gpu(*k, at::kBFloat16, dev) || !shaped(*k, {p.num_kv_heads, n, p.head_dim}) ||
        !on_gpu(*v, at::kBFloat16, dev) || v->sizes() != k->sizes() || !on_gpu(*kv, c->kv_type, dev) ||
        kv->dim() != 2 || kv->size(1) != page || kv->size(0) > INT32_MAX || !table_on(*table, dev) ||
        !shaped(*table, {p.pcp_size, p.max_local_blocks}) ||
        (valid && (!on_gpu(*valid, at::kInt, dev) || valid->sizes() != table->sizes())))
        GIVE_UP;
    void* stream = nullptr;
    if (!current_stream(dev, stream)) GIVE_UP;
    p.num_pages = (int32_t)kv->size(0);
    if (table->scalar_type() == at::kLong) p.flags |= PCPA_FLAG_TABLE_INT64;
    const void *kp = k->data_ptr(), *vp = v->data_ptr(), *tp = table->data_ptr();
    void* const pages = kv->data_ptr();
    int32_t* const lens = valid ? (int32_t*)valid->data_ptr() : nullptr;
    const int32_t status = launch([&] {
        return ((Write)c->fn)(&p, c->interleave, first, (int32_t)n, kp, vp, tp, pages, lens, stream);
    });
    return PyLong_FromLong(status);
}

// (first_pos, num_tokens, block_table, free_pages, free_count) -> status
PyObject* alloc(Call* c, PyObject* const* a) {
    const at::Tensor *table = plain(a[2]), *pages = plain(a[3]), *count = plain(a[4]);
    int64_t first, n;
    if (!table || !pages || !count || !whole(a[0], first) || !whole(a[1], n) || n < 0 || n > INT32_MAX ||
        !pages->is_cuda())
        GIVE_UP;
    pcpa_params p = c->p;
    const int dev = pages->get_device();
    if (!table_on(*table, dev) || !shaped(*table, {p.pcp_size, p.max_local_blocks})) GIVE_UP;
    void* stream = nullptr;
    if (!current_stream(dev, stream)) GIVE_UP;
    if (table->scalar_type() == at::kLong) p.flags |= PCPA_FLAG_TABLE_INT64;
    void* const tp = table->data_ptr();
    const int32_t* const pp = (const int32_t*)pages->data_ptr();
    int32_t* const cp = (int32_t*)count->data_ptr();
    const int32_t status =
        launch([&] { return ((Alloc)c->fn)(&p, c->interleave, first, (int32_t)n, tp, pp, cp, stream); });
    return PyLong_FromLong(status);
}

template <PyObject* (*F)(Call*, PyObject* const*), Py_ssize_t N>
PyObject* vector(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    if (PyVectorcall_NARGS(nargsf) != N || kwnames) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    try {
        return F((Call*)self, args);
    } catch (...) {
        // e.g. a tensor without storage: the general path says so
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

void call_dealloc(PyObject* self) {
    Call* c = (Call*)self;
    PyObject_GC_UnTrack(self);
    Py_CLEAR(c->ws_maker);
    delete c->spaces;
    Py_TYPE(self)->tp_free(self);
}
int call_traverse(PyObject* self, visitproc visit, void* arg) {
    Py_VISIT(((Call*)self)->ws_maker);
    return 0;
}
int call_clear(PyObject* self) {
    Py_CLEAR(((Call*)self)->ws_maker);
    return 0;
}
PyObject* call_forget(PyObject* self, PyObject*) {
    forget((Call*)self);
    Py_RETURN_NONE;
}
PyMethodDef call_methods[] = {
    {"forget", call_forget, METH_NOARGS, "Drop the workspaces remembered for streams."},
    {nullptr, nullptr, 0, nullptr},
};
PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

Call* new_call(vectorcallfunc f, const char* params, Py_ssize_t size, int fp8, int interleave, unsigned long long fn) {
    if (size != (Py_ssize_t)sizeof(pcpa_params)) {
        PyErr_SetString(PyExc_ValueError, "launch parameters of another size");
        return nullptr;
    }
    Call* c = PyObject_GC_New(Call, &CallType);
    if (!c) return nullptr;
    c->call = f;
    memcpy(&c->p, params, sizeof(pcpa_params));
    c->kv_type = fp8 ? at::kFloat8_e4m3fn : at::kBFloat16;
    c->interleave = interleave;
    c->dev = -1;
    c->fn = (void*)(uintptr_t)fn;
    c->n_split = 1;
    c->workspace = false;
    c->ws_bytes = 0;
    c->ws_maker = nullptr;
    c->spaces = new (std::nothrow) std::vector<Call::Space>();
    PyObject_GC_Track((PyObject*)c);
    if (!c->spaces) {
        Py_DECREF(c);
        PyErr_NoMemory();
        return nullptr;
    }
    return c;
}

// make(kind, params bytes, fp8 cache, interleave, C function address)
PyObject* make(PyObject*, PyObject* args) {
    const char *kind, *params;
    Py_ssize_t size;
    int fp8, interleave;
    unsigned long long fn;
    if (!PyArg_ParseTuple(args, "sy#piK", &kind, &params, &size, &fp8, &interleave, &fn)) return nullptr;
    vectorcallfunc f = !strcmp(kind, "current") ? vector<current, 6>
                       : !strcmp(kind, "write") ? vector<write, 8>
                       : !strcmp(kind, "alloc") ? vector<alloc, 5>
                                                : nullptr;
    if (!f) {
        PyErr_SetString(PyExc_ValueError, "unknown call");
        return nullptr;
    }
    return (PyObject*)new_call(f, params, size, fp8, interleave, fn);
}

// make_history(params bytes, fp8 cache, C function address, device index, splits, workspace bytes or -1, maker)
PyObject* make_history(PyObject*, PyObject* args) {
    const char* params;
    Py_ssize_t size;
    int fp8, dev, splits;
    unsigned long long fn;
    long long ws;
    PyObject* maker;
    if (!PyArg_ParseTuple(args, "y#pKiiLO", &params, &size, &fp8, &fn, &dev, &splits, &ws, &maker)) return nullptr;
    Call* c = new_call(vector<history, 8>, params, size, fp8, 0, fn);
    if (!c) return nullptr;
    c->dev = dev;
    c->n_split = splits;
    c->workspace = ws >= 0;
    c->ws_bytes = ws;
    Py_INCREF(maker);
    c->ws_maker = maker;
    return (PyObject*)c;
}

PyMethodDef methods[] = {
    {"make", make, METH_VARARGS, "A call of the current step, the cache writer or the page allocator."},
    {"make_history", make_history, METH_VARARGS, "A call of the history attention."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pcpa_fast_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__pcpa_fast_calls(void) {
    CallType.tp_name = "_pcpa_fast_calls.Call";
    CallType.tp_basicsize = sizeof(Call);
    CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL | Py_TPFLAGS_HAVE_GC;
    CallType.tp_vectorcall_offset = offsetof(Call, call);
    CallType.tp_call = PyVectorcall_Call;
    CallType.tp_dealloc = call_dealloc;
    CallType.tp_traverse = call_traverse;
    CallType.tp_clear = call_clear;
    CallType.tp_methods = call_methods;
    if (PyType_Ready(&CallType) < 0) return nullptr;
    PyObject* c = PyImport_ImportModule("torch._C");
    if (!c) return nullptr;
    g_raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
    g_device = PyObject_GetAttrString(c, "_cuda_getDevice");
    Py_DECREF(c);
    if (!g_raw_stream || !g_device) return nullptr;
    PyObject* const m = PyModule_Create(&module);
    if (!m) return nullptr;
    if (PyModule_AddIntConstant(m, "version", kVersion) < 0 ||
        PyModule_AddStringConstant(m, "torch_version", PCPA_TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
