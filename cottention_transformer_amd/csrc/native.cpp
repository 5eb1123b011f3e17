// The host side of the hot operators in native code: for ordinary calls (plain contiguous tensors of one type on the current
// device, shapes that agree) the tensors' pointers, the outputs, the workspace and the launch in one step each.  Anything
// else is answered with None, and the Python of ops.py, which knows all forms and their errors, takes the call; so is every call
// while a function or dispatch mode is on (torch.set_default_device is one).  A call costs
// about 6 us instead of 11, of which the launch is 3.5 (one launch; 128 positions of 2 heads).
// Nothing is kept between calls but the library's entry points.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

// dtype codes of include/cottention.h
constexpr int kF32 = 0, kF64 = 1, kF16 = 2, kBf16 = 3;

#define COTT_ENTRY(name, ...) int (*name)(__VA_ARGS__) = nullptr
struct Library {
    const char *(*cott_last_error)() = nullptr;
    size_t (*cott_causal_workspace_bytes)(int, int, int, int, int, int) = nullptr;
    size_t (*cott_causal_bwd_workspace_bytes)(int, int, int, int, int, int) = nullptr;
    size_t (*cott_noncausal_workspace_bytes)(int, int, int, int, int, int) = nullptr;
    COTT_ENTRY(cott_causal_fwd, const void *, const void *, const void *, void *, int, int, int, int, int, int, int, void *, size_t, void *);
    COTT_ENTRY(cott_causal_fwd_f32in_supported, int, int, int, int, int);
    COTT_ENTRY(cott_causal_fwd_f32in, const void *, const void *, const void *, void *, int, int, int, int, int, void *);
    COTT_ENTRY(cott_causal_saved_plan, int, int, int, int, int, int, int *, int *, int *, size_t *);
    COTT_ENTRY(cott_causal_fwd_save, const void *, const void *, const void *, void *, void *, int, int, int, int, int, int, int, int, void *,
               size_t, void *);
    COTT_ENTRY(cott_causal_bwd, const void *, const void *, const void *, const void *, void *, void *, void *, int, int, int, int, int, int,
               void *, size_t, void *);
    COTT_ENTRY(cott_causal_bwd_saved, const void *, const void *, const void *, const void *, void *, void *, void *, const void *, int, int,
               int, int, int, int, int, int, void *, size_t, void *);
    COTT_ENTRY(cott_causal_bwd_g16_supported, int, int, int, int, int);
    COTT_ENTRY(cott_causal_bwd_g16, const void *, const void *, const void *, const void *, void *, void *, void *, int, int, int, int, int,
               void *, size_t, void *);
    COTT_ENTRY(cott_noncausal_fwd, const void *, const void *, const void *, void *, int, int, int, int, int, int, void *, size_t, void *);
    COTT_ENTRY(cott_noncausal_bwd, const void *, const void *, const void *, const void *, void *, void *, void *, int, int, int, int, int,
               int, void *, size_t, void *);
    COTT_ENTRY(cott_decode_block_norm, const void *, const void *, const void *, const void *, const void *, void *, void *, const void *, int,
               float, const void *, long long, int, int, int, int, int, int, void *, size_t, void *);
} L;
PyObject *raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return kF32;
        case at::kDouble: return kF64;
        case at::kHalf: return kF16;
        case at::kBFloat16: return kBf16;
        default: return -1;
    }
}

// An ordinary dense tensor on GPU `device`: not a subclass, not a wrapper of a transform (vmap, grad, functionalization), no
// lazy conjugate or negative.
const at::Tensor *plain(PyObject *o, int device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::Batched, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                            c10::DispatchKey::ZeroTensor});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_nested() || t.key_set().has_any(other) || !t.has_storage() ||
        t.device().index() != device)
        return nullptr;
    return &t;
}
const at::Tensor *plain_contiguous(PyObject *o, int device) {
    const at::Tensor *t = plain(o, device);
    return t && t->is_contiguous() ? t : nullptr;
}

// The current device, or -1 when the first operand is no GPU tensor or a dispatch or function mode wants to see the operations.
int current_device(PyObject *first) {
    if (!THPVariable_CheckExact(first) || !THPVariable_Unpack(first).is_cuda()) return -1;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) return -1;
    return c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index();
}

struct Shape {
    int b, h, n, dk, dv;
};
// (B,H,N,D) tensors of one type that agree
bool shapes(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v, Shape *s) {
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || q.scalar_type() != k.scalar_type() || q.scalar_type() != v.scalar_type())
        return false;
    const auto a = q.sizes(), c = v.sizes();
    if (k.sizes() != a || a[0] != c[0] || a[1] != c[1] || a[2] != c[2]) return false;
    for (int64_t x : {a[0], a[1], a[2], a[3], c[3]})
        if (x < 1 || x > INT_MAX) return false;
    *s = Shape{(int)a[0], (int)a[1], (int)a[2], (int)a[3], (int)c[3]};
    return true;
}

bool stream_of(int device, void **stream) {
    PyObject *index = PyLong_FromLong(device);
    if (!index) return false;
    PyObject *r = PyObject_CallOneArg(raw_stream, index);
    Py_DECREF(index);
    if (!r) return false;
    *stream = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return !PyErr_Occurred();
}

struct Workspace {
    at::Tensor t;
    void *ptr = nullptr;
    size_t bytes;
    Workspace(size_t n, const at::Tensor &like) : bytes(n) {
        if (n == 0) return;
        t = at::empty({(int64_t)n}, like.options().dtype(at::kByte));
        ptr = t.data_ptr();
    }
};

PyObject *failed() {
    const char *msg = L.cott_last_error();
    PyErr_SetString(PyExc_RuntimeError, msg && *msg ? msg : "a call into the library failed");
    return nullptr;
}

PyObject *three(at::Tensor &a, at::Tensor &b, at::Tensor &c) {
    PyObject *x = THPVariable_Wrap(std::move(a)), *y = THPVariable_Wrap(std::move(b)), *z = THPVariable_Wrap(std::move(c));
    PyObject *r = x && y && z ? PyTuple_Pack(3, x, y, z) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    Py_XDECREF(z);
    return r;
}

bool wants(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "%zd arguments, %zd given", want, n);
    return false;
}

// causal_dot_product(q, k, v, reversed)
PyObject *causal(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 4)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev);
    Shape s;
    if (dev < 0 || !q || !k || !v || !shapes(*q, *k, *v, &s)) Py_RETURN_NONE;
    const int code = dtype_code(q->scalar_type()), reversed = PyObject_IsTrue(a[3]);
    void *stream;
    if (reversed < 0 || !stream_of(dev, &stream)) return nullptr;
    if (code < 0) Py_RETURN_NONE;
    at::Tensor o = at::empty({s.b, s.h, s.n, s.dv}, q->options());
    const Workspace ws(L.cott_causal_workspace_bytes(s.b, s.h, s.n, s.dk, s.dv, code), *q);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = L.cott_causal_fwd(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), s.b, s.h, s.n, s.dk, s.dv, code, reversed, ws.ptr,
                           ws.bytes, stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

// causal_dot_product_saving(q, k, v) of 16-bit tensors
PyObject *causal_saving(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 3)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev);
    Shape s;
    if (dev < 0 || !q || !k || !v || !shapes(*q, *k, *v, &s)) Py_RETURN_NONE;
    const int code = dtype_code(q->scalar_type());
    if (code != kF16 && code != kBf16) Py_RETURN_NONE;
    void *stream;
    if (!stream_of(dev, &stream)) return nullptr;
    int cpc = 0, cuts = 0, slot = 0, rc;
    size_t unused = 0;
    if (L.cott_causal_saved_plan(s.b, s.h, s.n, s.dk, s.dv, code, &cpc, &cuts, &slot, &unused)) return failed();
    at::Tensor o = at::empty({s.b, s.h, s.n, s.dv}, q->options()), saved;
    if (cuts > 0) saved = at::empty({s.b, s.h, cuts, slot}, q->options().dtype(at::kFloat));
    const Workspace ws(L.cott_causal_workspace_bytes(s.b, s.h, s.n, s.dk, s.dv, code), *q);
    Py_BEGIN_ALLOW_THREADS
    if (cuts > 0)
        rc = L.cott_causal_fwd_save(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), saved.data_ptr(), cpc, cuts, s.b, s.h, s.n,
                                    s.dk, s.dv, code, ws.ptr, ws.bytes, stream);
    else
        rc = L.cott_causal_fwd(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), s.b, s.h, s.n, s.dk, s.dv, code, 0, ws.ptr,
                               ws.bytes, stream);
    Py_END_ALLOW_THREADS
    if (rc) return failed();
    PyObject *po = THPVariable_Wrap(std::move(o));
    PyObject *ps = cuts > 0 ? THPVariable_Wrap(std::move(saved)) : Py_NewRef(Py_None);
    PyObject *r = po && ps ? PyTuple_Pack(2, po, ps) : nullptr;
    Py_XDECREF(po);
    Py_XDECREF(ps);
    return r;
    END_HANDLE_TH_ERRORS
}

// fp32 q, k, v rounded to bf16 inside the forward kernel (causal_dot_product_as)
PyObject *causal_f32in(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 3)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev);
    Shape s;
    if (dev < 0 || !q || !k || !v || q->scalar_type() != at::kFloat || !shapes(*q, *k, *v, &s)) Py_RETURN_NONE;
    if (((uintptr_t)q->data_ptr() | (uintptr_t)k->data_ptr() | (uintptr_t)v->data_ptr()) & 15) Py_RETURN_NONE;
    if (!L.cott_causal_fwd_f32in_supported(s.b, s.h, s.n, s.dk, s.dv)) Py_RETURN_NONE;
    void *stream;
    if (!stream_of(dev, &stream)) return nullptr;
    at::Tensor o = at::empty({s.b, s.h, s.n, s.dv}, q->options().dtype(at::kBFloat16));
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = L.cott_causal_fwd_f32in(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), s.b, s.h, s.n, s.dk, s.dv, stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

// causal_backward(q, k, v, grad_out, saved or None); an fp32 call may have a bf16 grad_out where the library reads it
PyObject *causal_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 5)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev),
                     *g = plain_contiguous(a[3], dev);
    const bool with_states = a[4] != Py_None;
    const at::Tensor *saved = with_states ? plain_contiguous(a[4], dev) : nullptr;
    Shape s;
    if (dev < 0 || !q || !k || !v || !g || (with_states && !saved) || !shapes(*q, *k, *v, &s) || g->sizes() != v->sizes()) Py_RETURN_NONE;
    const int code = dtype_code(q->scalar_type());
    const bool g16 = code == kF32 && g->scalar_type() == at::kBFloat16 && !with_states;
    if (code < 0 || !(g16 || g->scalar_type() == q->scalar_type())) Py_RETURN_NONE;
    if (g16 && ((((uintptr_t)q->data_ptr() | (uintptr_t)k->data_ptr() | (uintptr_t)v->data_ptr() | (uintptr_t)g->data_ptr()) & 15) ||
                !L.cott_causal_bwd_g16_supported(s.b, s.h, s.n, s.dk, s.dv)))
        Py_RETURN_NONE;
    int cpc = 0, cuts = 0, slot = 0, rc;
    size_t bytes = 0;
    if (with_states) {
        if (L.cott_causal_saved_plan(s.b, s.h, s.n, s.dk, s.dv, code, &cpc, &cuts, &slot, &bytes)) return failed();
        if (cuts < 1 || saved->scalar_type() != at::kFloat || saved->sizes() != at::IntArrayRef({s.b, s.h, cuts, slot})) Py_RETURN_NONE;
    } else {
        bytes = L.cott_causal_bwd_workspace_bytes(s.b, s.h, s.n, s.dk, s.dv, code);
    }
    void *stream;
    if (!stream_of(dev, &stream)) return nullptr;
    at::Tensor dq = at::empty(q->sizes(), q->options()), dk = at::empty(k->sizes(), q->options()), dv = at::empty(v->sizes(), q->options());
    const Workspace ws(bytes, *q);
    Py_BEGIN_ALLOW_THREADS
    if (with_states)
        rc = L.cott_causal_bwd_saved(q->data_ptr(), k->data_ptr(), v->data_ptr(), g->data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                     saved->data_ptr(), cpc, cuts, s.b, s.h, s.n, s.dk, s.dv, code, ws.ptr, ws.bytes, stream);
    else if (g16)
        rc = L.cott_causal_bwd_g16(q->data_ptr(), k->data_ptr(), v->data_ptr(), g->data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                   s.b, s.h, s.n, s.dk, s.dv, ws.ptr, ws.bytes, stream);
    else
        rc = L.cott_causal_bwd(q->data_ptr(), k->data_ptr(), v->data_ptr(), g->data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), s.b,
                               s.h, s.n, s.dk, s.dv, code, ws.ptr, ws.bytes, stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : three(dq, dk, dv);
    END_HANDLE_TH_ERRORS
}

// noncausal_dot_product(q, k, v)
PyObject *noncausal(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 3)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev);
    Shape s;
    if (dev < 0 || !q || !k || !v || !shapes(*q, *k, *v, &s)) Py_RETURN_NONE;
    const int code = dtype_code(q->scalar_type());
    if (code < 0) Py_RETURN_NONE;
    void *stream;
    if (!stream_of(dev, &stream)) return nullptr;
    at::Tensor o = at::empty({s.b, s.h, s.n, s.dv}, q->options());
    const Workspace ws(L.cott_noncausal_workspace_bytes(s.b, s.h, s.n, s.dk, s.dv, code), *q);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = L.cott_noncausal_fwd(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), s.b, s.h, s.n, s.dk, s.dv, code, ws.ptr, ws.bytes,
                              stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

// noncausal_backward(q, k, v, grad_out)
PyObject *noncausal_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 4)) return nullptr;
    const int dev = current_device(a[0]);
    const at::Tensor *q = plain_contiguous(a[0], dev), *k = plain_contiguous(a[1], dev), *v = plain_contiguous(a[2], dev),
                     *g = plain_contiguous(a[3], dev);
    Shape s;
    if (dev < 0 || !q || !k || !v || !g || !shapes(*q, *k, *v, &s) || g->sizes() != v->sizes() || g->scalar_type() != q->scalar_type())
        Py_RETURN_NONE;
    const int code = dtype_code(q->scalar_type());
    if (code < 0) Py_RETURN_NONE;
    void *stream;
    if (!stream_of(dev, &stream)) return nullptr;
    at::Tensor dq = at::empty(q->sizes(), q->options()), dk = at::empty(k->sizes(), q->options()), dv = at::empty(v->sizes(), q->options());
    const Workspace ws(L.cott_noncausal_workspace_bytes(s.b, s.h, s.n, s.dk, s.dv, code), *q);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = L.cott_noncausal_bwd(q->data_ptr(), k->data_ptr(), v->data_ptr(), g->data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), s.b,
                              s.h, s.n, s.dk, s.dv, code, ws.ptr, ws.bytes, stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : three(dq, dk, dv);
    END_HANDLE_TH_ERRORS
}

// decode_block(x, wq, wk, wv, wo, state, norm_const, cnt, table, position)
PyObject *decode_block(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!wants(n, 10)) return nullptr;
    const int dev = current_device(a[0]);
    if (dev < 0) Py_RETURN_NONE;
    const at::Tensor *t[7];
    for (int i = 0; i < 7; ++i)
        if (!(t[i] = plain_contiguous(a[i], dev))) Py_RETURN_NONE;
    const at::Tensor *table = plain_contiguous(a[8], dev);
    const at::Tensor &x = *t[0], &state = *t[5], &norm = *t[6];
    const int code = dtype_code(x.scalar_type()), norm_code = dtype_code(norm.scalar_type());
    if (!table || (code != kF16 && code != kBf16) || norm_code < 0 || x.dim() != 2 || state.dim() != 4) Py_RETURN_NONE;
    const int64_t b = x.size(0), e = x.size(1), h = state.size(1), d = state.size(2);
    if (b < 1 || b > INT_MAX || e < 1 || e > INT_MAX || state.size(0) != b || state.size(3) != d || h * d != e ||
        state.scalar_type() != at::kFloat || norm.numel() != h || table->dim() != 2 || table->scalar_type() != at::kFloat ||
        table->size(0) > INT_MAX)
        Py_RETURN_NONE;
    for (int i = 1; i < 5; ++i)
        if (t[i]->dim() != 2 || t[i]->size(0) != e || t[i]->size(1) != e || t[i]->scalar_type() != x.scalar_type()) Py_RETURN_NONE;
    const double cnt = PyFloat_AsDouble(a[7]);
    const long long pos = PyLong_AsLongLong(a[9]);
    void *stream;
    if (PyErr_Occurred() || !stream_of(dev, &stream)) return nullptr;
    at::Tensor scratch = at::empty({4, b, e}, x.options()), y = at::empty({b, e}, x.options());
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = L.cott_decode_block_norm(x.data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), t[3]->data_ptr(), t[4]->data_ptr(), state.data_ptr(),
                                  y.data_ptr(), norm.data_ptr(), norm_code, (float)cnt, table->data_ptr(), pos, (int)table->size(1),
                                  (int)table->size(0), (int)b, (int)h, (int)d, code, scratch.data_ptr(), (size_t)(8 * b * e), stream);
    Py_END_ALLOW_THREADS
    return rc ? failed() : THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// bind(addresses of the library's entry points by name, torch._C._cuda_getCurrentRawStream)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (!wants(n, 2)) return nullptr;
    struct {
        const char *name;
        void **to;
    } entries[] = {
#define COTT_BIND(name) {#name, reinterpret_cast<void **>(&L.name)}
        COTT_BIND(cott_last_error), COTT_BIND(cott_causal_workspace_bytes), COTT_BIND(cott_causal_bwd_workspace_bytes),
        COTT_BIND(cott_noncausal_workspace_bytes), COTT_BIND(cott_causal_fwd), COTT_BIND(cott_causal_fwd_f32in_supported),
        COTT_BIND(cott_causal_fwd_f32in), COTT_BIND(cott_causal_saved_plan), COTT_BIND(cott_causal_fwd_save), COTT_BIND(cott_causal_bwd),
        COTT_BIND(cott_causal_bwd_saved), COTT_BIND(cott_causal_bwd_g16_supported), COTT_BIND(cott_causal_bwd_g16),
        COTT_BIND(cott_noncausal_fwd), COTT_BIND(cott_noncausal_bwd), COTT_BIND(cott_decode_block_norm),
    };
    for (const auto &e : entries) {
        PyObject *address = PyDict_GetItemString(a[0], e.name);
        if (!address) return PyErr_Format(PyExc_KeyError, "%s", e.name);
        *e.to = PyLong_AsVoidPtr(address);
        if (PyErr_Occurred()) return nullptr;
    }
    Py_INCREF(a[1]);
    Py_XSETREF(raw_stream, a[1]);
    Py_RETURN_NONE;
}

#define COTT_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {COTT_METHOD(bind), COTT_METHOD(causal), COTT_METHOD(causal_saving), COTT_METHOD(causal_f32in),
                         COTT_METHOD(causal_backward), COTT_METHOD(noncausal), COTT_METHOD(noncausal_backward), COTT_METHOD(decode_block),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
