// CPython module `_oxq_torch`: the per-call half of the torch binding in native code.
//
// A decode step makes one library call per projection, and each call's kernel takes 3 - 10 us.  Building
// the tensor descriptors field by field in Python, allocating the output through torch.empty and crossing
// ctypes took 8 - 10 us of host time per call and was what bounded every eager call below about 13 us of
// GPU time; here the same steps (unpack the tensors, allocate the output, take the current stream, call the
// C ABI) are native.  Figures beside `layer_call` below.
//
// The module links against torch only.  The library's entry points are looked up in the handle that the ctypes
// loader opened (`bind`), so both bindings always talk to the same copy of it.
// OXQ_TORCH_HIP is 0 for a torch without GPU support: there plan-only contexts work, and nothing else could.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#if OXQ_TORCH_HIP
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#endif
#include <torch/csrc/Device.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "oxq.h"

namespace {

// ---------------------------------------------------------------- the library's entry points
#define OXQ_BOUND(X)                                                                                              \
    X(oxq_last_error) X(oxq_packed_quant_linear_forward) X(oxq_qlinear_forward) X(oxq_mxfp4_linear_forward)       \
    X(oxq_mlp_forward) X(oxq_mlp_scratch_elems) X(oxq_w4a16_matmul) X(oxq_w8a16_matmul) X(oxq_gptq_matmul)        \
    X(oxq_mpp_quant_matmul) X(oxq_f8_gemv) X(oxq_f8_matmul) X(oxq_gguf_quant_matmul) X(oxq_gguf_quant_mul_mm)     \
    X(oxq_mxfp4_matmul) X(oxq_mxfp4_moe_matmul) X(oxq_mxfp4_moe_gate_up_swiglu) X(oxq_mxfp4_experts_matmul)       \
    X(oxq_mxfp4_experts_gate_up_swiglu) X(oxq_moe_route) X(oxq_moe_group) X(oxq_moe_route_group)                  \
    X(oxq_gated_activation) X(oxq_activation_mul) X(oxq_moe_combine)

struct Api {
#define OXQ_FIELD(f) decltype(&::f) f = nullptr;
    OXQ_BOUND(OXQ_FIELD)
#undef OXQ_FIELD
};
Api api;
PyObject *error_class = nullptr;   // OxqError(status, message)
PyObject *tensor_struct = nullptr; // the ctypes descriptor class, accepted wherever a tensor is
PyObject *torch_empty = nullptr;   // torch.empty and torch.empty_like, for the modes that watch Python calls
PyObject *torch_empty_like = nullptr;

struct Failed {};  // a Python error is set

[[noreturn]] void raise(int status, const char *msg) {
    if (PyObject *e = PyObject_CallFunction(error_class, "is", status, msg)) {
        PyErr_SetObject(error_class, e);
        Py_DECREF(e);
    }
    throw Failed();
}

void check(int rc) {
    if (rc == OXQ_OK) return;
    const char *msg = api.oxq_last_error();
    raise(rc, msg ? msg : "");
}

// A library call with the GIL released: a launch may block while the queue is full, and other engine threads must run.
template <typename F> void call(F &&f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    check(rc);
}

// ---------------------------------------------------------------- arguments
int dtype_of(const at::Tensor &t) {
    switch (t.scalar_type()) {
    case at::kFloat: return OXQ_F32;
    case at::kHalf: return OXQ_F16;
    case at::kBFloat16: return OXQ_BF16;
    case at::kByte: return OXQ_U8;
    case at::kInt: return OXQ_I32;
    case at::kUInt32: return OXQ_U32;
    case at::kLong: return OXQ_I64;
    default: break;
    }
    raise(OXQ_ERR_DTYPE, (std::string("unsupported torch dtype ") + c10::toString(t.scalar_type())).c_str());
}

void fill(const at::Tensor &t, oxq_tensor &d) {
    const int64_t rank = t.dim();
    const int dtype = dtype_of(t);
    if (rank < 1 || rank > OXQ_MAX_RANK)
        raise(OXQ_ERR_SHAPE, ("rank " + std::to_string(rank) + " out of [1, " + std::to_string(OXQ_MAX_RANK) + "]").c_str());
    d.data = t.data_ptr();
    d.dtype = dtype;
    d.rank = (int32_t)rank;
    for (int i = 0; i < OXQ_MAX_RANK; ++i) d.dims[i] = i < rank ? t.size(i) : 0;
    d.contiguous = t.is_contiguous() ? 1 : 0;
    d.device = t.is_cuda() ? (int32_t)t.get_device() : OXQ_DEVICE_HOST;
}

const at::Tensor &tensor(PyObject *o) {
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
        throw Failed();
    }
    return THPVariable_Unpack(o);
}

// One tensor argument: None, a torch tensor or a ready-made descriptor.
struct Desc {
    oxq_tensor d;
    const oxq_tensor *p = nullptr;
    explicit Desc(PyObject *o) {
        if (o == Py_None) return;
        if (THPVariable_Check(o)) {
            fill(THPVariable_Unpack(o), d);
        } else if (PyObject_IsInstance(o, tensor_struct) == 1) {
            Py_buffer b;
            if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) throw Failed();
            memcpy(&d, b.buf, sizeof d);
            PyBuffer_Release(&b);
        } else {
            tensor(o);  // raises
        }
        p = &d;
    }
    explicit Desc(const at::Tensor &t) {
        fill(t, d);
        p = &d;
    }
    Desc(const Desc &o) : d(o.d), p(o.p ? &d : nullptr) {}
    Desc &operator=(const Desc &) = delete;
    operator const oxq_tensor *() const { return p; }
};

int64_t integer(PyObject *o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Failed();
    return v;
}

double real(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Failed();
    return v;
}

// An owned reference, dropped at the end of the scope.
struct Ref {
    PyObject *o;
    explicit Ref(PyObject *p) : o(p) {
        if (!o) throw Failed();
    }
    Ref(const Ref &) = delete;
    ~Ref() { Py_DECREF(o); }
};

at::Tensor unpacked(const Ref &r) { return THPVariable_Unpack(r.o); }

// Outputs are what torch.empty makes: allocated through the dispatcher, so that dispatch modes see them and they are
// filled under deterministic algorithms (0.25 us more than asking the allocator), and through the Python function itself
// while a torch function mode is active.
at::Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const at::Device &dev) {
    if (at::impl::torch_function_mode_enabled()) {
        const Ref size(PyTuple_New((Py_ssize_t)shape.size()));
        for (size_t i = 0; i < shape.size(); ++i) {
            PyObject *n = PyLong_FromLongLong(shape[i]);
            if (!n) throw Failed();
            PyTuple_SET_ITEM(size.o, (Py_ssize_t)i, n);
        }
        const Ref args(PyTuple_Pack(1, size.o)), device(THPDevice_New(dev));
        const Ref kwargs(Py_BuildValue("{sOsO}", "dtype", (PyObject *)torch::getTHPDtype(dtype), "device", device.o));
        return unpacked(Ref(PyObject_Call(torch_empty, args.o, kwargs.o)));
    }
    return at::empty(shape, at::TensorOptions().dtype(dtype).device(dev));
}
at::Tensor empty_like(PyObject *x) {
    const at::Tensor &t = tensor(x);
    if (at::impl::torch_function_mode_enabled()) return unpacked(Ref(PyObject_CallOneArg(torch_empty_like, x)));
    return at::empty_like(t);
}

// The output of a call: the caller's tensor (or descriptor), or a new one.
class Out {
    PyObject *given_;
    at::Tensor made_;
    Desc desc_;

  public:
    template <typename Make>
    Out(PyObject *o, Make &&make)
        : given_(o == Py_None ? nullptr : o), made_(given_ ? at::Tensor() : make()),
          desc_(given_ ? Desc(given_) : Desc(made_)) {}
    operator const oxq_tensor *() const { return desc_; }
    PyObject *get() {
        if (!given_) return THPVariable_Wrap(std::move(made_));
        Py_INCREF(given_);
        return given_;
    }
};

#define OXQ_BODY_BEGIN \
    HANDLE_TH_ERRORS   \
    try {
#define OXQ_BODY_END           \
    } catch (const Failed &) { \
        return nullptr;        \
    }                          \
    END_HANDLE_TH_ERRORS

void want(Py_ssize_t got, Py_ssize_t n) {
    if (got == n) return;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", n, got);
    throw Failed();
}

// ---------------------------------------------------------------- handles
enum { KIND_MLP = OXQ_LINEAR_MXFP4 + 1, KIND_PLAIN };  // beyond oxq_linear_kind: a FeedForward; a ctx or an expert set

#if OXQ_TORCH_HIP
int device() { return c10::hip::current_device(); }
void *current_stream() { return c10::hip::getCurrentHIPStream().stream(); }
#else
[[noreturn]] int device() {
    PyErr_SetString(PyExc_RuntimeError, "this torch has no GPU support: only plan-only contexts work");
    throw Failed();
}
void *current_stream() { device(); }
#endif

// A C handle: a ctx, an expert set, or a layer, which is called as `layer(x, out)` (a FeedForward: `(x, out, scratch)`).
struct Handle {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    void *ptr;
    int64_t width;  // columns of the output
    int kind;
    bool plan_only;  // validates and plans only: there may be no GPU to ask for a stream
    void *stream() const { return plan_only ? nullptr : current_stream(); }
};

// [.., k] -> [.., width]
at::Tensor empty_rows(const at::Tensor &x, int64_t width) {
    c10::SmallVector<int64_t, OXQ_MAX_RANK> shape(x.sizes().begin(), x.sizes().end());
    if (!shape.empty()) shape.back() = width;
    return empty(shape, x.scalar_type(), x.device());
}

// One resident 4096 x 4096 4-bit layer at one row of f16, called back to back without waiting: 12.2 us through
// Python-built descriptors, 4.5 us here (3.7 with the caller's output tensor; the kernel alone takes 3.6 us, torch's
// own zero_() 3.8 us a call).  The six outputs and one launch of moe_route_group: 27.8 -> 8.5 us.
PyObject *layer_call(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
    OXQ_BODY_BEGIN
    Handle *h = (Handle *)self;
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    want(n + (kwnames ? PyTuple_GET_SIZE(kwnames) : 0), h->kind == KIND_MLP ? 3 : 2);
    want(n, h->kind == KIND_MLP ? 3 : 2);
    const Desc x(args[0]);
    Out out(args[1], [&] { return empty_rows(tensor(args[0]), h->width); });
    void *const s = h->stream();
    switch (h->kind) {
    case OXQ_LINEAR_PACKED_QUANT:
        call([&] { return api.oxq_packed_quant_linear_forward((oxq_packed_quant_linear *)h->ptr, s, x, out); });
        break;
    case OXQ_LINEAR_GGUF:
        call([&] { return api.oxq_qlinear_forward((oxq_qlinear *)h->ptr, s, x, out); });
        break;
    case OXQ_LINEAR_MXFP4:
        call([&] { return api.oxq_mxfp4_linear_forward((oxq_mxfp4_linear *)h->ptr, s, x, out); });
        break;
    case KIND_MLP: {
        Out scratch(args[2], [&] {
            const at::Tensor &t = tensor(args[0]);
            const int64_t cols = t.dim() ? t.size(-1) : 1;
            int64_t elems = 0;
            check(api.oxq_mlp_scratch_elems((oxq_mlp *)h->ptr, t.numel() / std::max<int64_t>(cols, 1), &elems));
            return empty({std::max<int64_t>(elems, 1)}, t.scalar_type(), t.device());
        });
        call([&] { return api.oxq_mlp_forward((oxq_mlp *)h->ptr, s, x, scratch, out); });
        break;
    }
    default:
        PyErr_SetString(PyExc_TypeError, "this handle is not callable");
        throw Failed();
    }
    return out.get();
    OXQ_BODY_END
}

PyObject *handle_new(PyTypeObject *type, PyObject *args, PyObject *) {
    unsigned long long ptr;
    int kind, plan_only;
    long long width;
    if (!PyArg_ParseTuple(args, "KiLp", &ptr, &kind, &width, &plan_only)) return nullptr;
    Handle *h = (Handle *)type->tp_alloc(type, 0);
    if (!h) return nullptr;
    h->vectorcall = layer_call;
    h->ptr = (void *)(uintptr_t)ptr;
    h->width = width;
    h->kind = kind;
    h->plan_only = plan_only != 0;
    return (PyObject *)h;
}

PyTypeObject HandleType = {PyVarObject_HEAD_INIT(nullptr, 0)};

const Handle &handle(PyObject *o) {
    if (Py_TYPE(o) == &HandleType) return *(const Handle *)o;
    PyErr_SetString(PyExc_TypeError, "expected a native handle");
    throw Failed();
}
oxq_ctx *ctx_of(const Handle &h) { return (oxq_ctx *)h.ptr; }

// ---------------------------------------------------------------- products of checkpoint tensors
// `f(ctx, x, out, columns, operands ..)`: out [rows of x, columns] in x's type, or the caller's.
template <typename F> PyObject *rows_op(PyObject *const *a, F &&f) {
    const Handle &h = handle(a[0]);
    const Desc x(a[1]);
    const int64_t columns = integer(a[3]);
    Out out(a[2], [&] {
        const at::Tensor &t = tensor(a[1]);
        return empty({t.dim() ? t.size(0) : 1, columns}, t.scalar_type(), t.device());
    });
    void *const s = h.stream();
    f(ctx_of(h), s, x, out);
    return out.get();
}

template <auto Api::*Field> PyObject *packed_op(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 7);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc q(a[4]), z(a[5]), sc(a[6]);
        call([&] { return (api.*Field)(c, s, x, q, z, sc, out); });
    });
    OXQ_BODY_END
}

PyObject *gptq_matmul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 8);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc q(a[4]), z(a[5]), sc(a[6]);
        const uint32_t bits = (uint32_t)integer(a[7]);
        call([&] { return api.oxq_gptq_matmul(c, s, x, q, z, sc, bits, out); });
    });
    OXQ_BODY_END
}

PyObject *mpp_quant_matmul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 9);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc q(a[4]), z(a[5]), sc(a[6]);
        const uint32_t bits = (uint32_t)integer(a[7]);
        const int pack = (int)integer(a[8]);
        call([&] { return api.oxq_mpp_quant_matmul(c, s, x, q, z, sc, bits, pack, out); });
    });
    OXQ_BODY_END
}

template <auto Api::*Field> PyObject *f8_op(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 6);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc w(a[4]), sc(a[5]);
        call([&] { return (api.*Field)(c, s, x, w, sc, out); });
    });
    OXQ_BODY_END
}

template <auto Api::*Field> PyObject *gguf_op(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 7);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc w(a[4]);
        const int64_t k = integer(a[5]), cols = integer(a[3]);
        const int quant = (int)integer(a[6]);
        call([&] { return (api.*Field)(c, s, x, w, k, cols, quant, out); });
    });
    OXQ_BODY_END
}

PyObject *mxfp4_matmul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 7);
    return rows_op(a, [&](oxq_ctx *c, void *s, const oxq_tensor *x, const oxq_tensor *out) {
        const Desc w(a[4]), sc(a[5]);
        const int64_t k = integer(a[6]), cols = integer(a[3]);
        call([&] { return api.oxq_mxfp4_matmul(c, s, x, w, sc, k, cols, out); });
    });
    OXQ_BODY_END
}

// ---------------------------------------------------------------- experts
// [pairs, columns]: one row per (token, expert) pair, which token_ids lists or x already holds
at::Tensor empty_pairs(PyObject *x, PyObject *token_ids, int64_t columns) {
    const at::Tensor &t = tensor(x);
    const int64_t pairs = token_ids != Py_None ? tensor(token_ids).numel() : t.size(0);
    return empty({pairs, columns}, t.scalar_type(), t.device());
}

// (experts, x, out, expert_offsets, token_ids)
PyObject *experts_matmul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 5);
    const Handle &h = handle(a[0]);
    const Desc x(a[1]), off(a[3]), ids(a[4]);
    Out out(a[2], [&] { return empty_pairs(a[1], a[4], h.width); });
    void *const s = h.stream();
    const int gather = a[4] != Py_None;
    call([&] { return api.oxq_mxfp4_experts_matmul((oxq_mxfp4_experts *)h.ptr, s, x, off, ids, gather, out); });
    return out.get();
    OXQ_BODY_END
}

// -> (out, whether the fused launch was enqueued)
PyObject *with_flag(Out &out, int flag) {
    PyObject *o = out.get();
    if (!o) return nullptr;
    PyObject *r = PyTuple_Pack(2, o, flag ? Py_True : Py_False);
    Py_DECREF(o);
    return r;
}

PyObject *experts_gate_up_swiglu(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 6);
    const Handle &h = handle(a[0]);
    const Desc x(a[1]), off(a[3]), ids(a[4]);
    Out out(a[2], [&] { return empty_pairs(a[1], a[4], h.width / 2); });
    void *const s = h.stream();
    const int gather = a[4] != Py_None;
    const float limit = (float)real(a[5]);
    int fused = 0;
    call([&] {
        return api.oxq_mxfp4_experts_gate_up_swiglu((oxq_mxfp4_experts *)h.ptr, s, x, off, ids, gather, limit, out, &fused);
    });
    return with_flag(out, fused);
    OXQ_BODY_END
}

PyObject *moe_matmul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 10);
    const Handle &h = handle(a[0]);
    const int64_t k = integer(a[8]), cols = integer(a[9]);
    const Desc x(a[1]), w(a[3]), sc(a[4]), bias(a[5]), off(a[6]), ids(a[7]);
    Out out(a[2], [&] { return empty_pairs(a[1], a[7], cols); });
    void *const s = h.stream();
    const int gather = a[7] != Py_None;
    call([&] { return api.oxq_mxfp4_moe_matmul(ctx_of(h), s, x, w, sc, bias, off, ids, gather, k, cols, out); });
    return out.get();
    OXQ_BODY_END
}

PyObject *moe_gate_up_swiglu(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 11);
    const Handle &h = handle(a[0]);
    const int64_t k = integer(a[8]), cols = integer(a[9]);
    const float limit = (float)real(a[10]);
    const Desc x(a[1]), w(a[3]), sc(a[4]), bias(a[5]), off(a[6]), ids(a[7]);
    Out out(a[2], [&] { return empty_pairs(a[1], a[7], cols / 2); });
    void *const s = h.stream();
    const int gather = a[7] != Py_None;
    int fused = 0;
    call([&] {
        return api.oxq_mxfp4_moe_gate_up_swiglu(ctx_of(h), s, x, w, sc, bias, off, ids, gather, k, cols, limit, out, &fused);
    });
    return with_flag(out, fused);
    OXQ_BODY_END
}

// ---------------------------------------------------------------- mixture-of-experts glue
template <size_t N> PyObject *pack(at::Tensor (&t)[N]) {
    PyObject *r = PyTuple_New(N);
    if (!r) return nullptr;
    for (size_t i = 0; i < N; ++i) {
        PyObject *o = THPVariable_Wrap(std::move(t[i]));
        if (!o) {
            Py_DECREF(r);
            return nullptr;
        }
        PyTuple_SET_ITEM(r, i, o);
    }
    return r;
}

const at::Tensor &matrix(PyObject *o) {
    const at::Tensor &t = tensor(o);
    if (t.dim() != 2) raise(OXQ_ERR_SHAPE, ("expected two dimensions, got " + std::to_string(t.dim())).c_str());
    return t;
}

// (ctx, logits, top_k, norm) -> top_idx, top_vals
PyObject *moe_route(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 4);
    const Handle &h = handle(a[0]);
    const Desc logits(a[1]);
    const at::Tensor &t = tensor(a[1]);
    const int64_t T = t.size(0), k = integer(a[2]);
    const int norm = (int)integer(a[3]);
    at::Tensor r[2] = {empty({T, k}, at::kInt, t.device()), empty({T, k}, at::kFloat, t.device())};
    const Desc idx(r[0]), vals(r[1]);
    void *const s = h.stream();
    call([&] { return api.oxq_moe_route(ctx_of(h), s, logits, k, norm, idx, vals); });
    return pack(r);
    OXQ_BODY_END
}

// (ctx, top_idx, top_vals, n_experts) -> offsets, tokens, weights, pos
PyObject *moe_group(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 4);
    const Handle &h = handle(a[0]);
    const Desc idx(a[1]), vals(a[2]);
    const at::Tensor &t = matrix(a[1]);
    const int64_t T = t.size(0), k = t.size(1), E = integer(a[3]);
    const auto dev = t.device();
    at::Tensor r[4] = {empty({E + 1}, at::kInt, dev), empty({T * k}, at::kInt, dev), empty({T * k}, at::kFloat, dev),
                       empty({T, k}, at::kInt, dev)};
    const Desc off(r[0]), tok(r[1]), w(r[2]), pos(r[3]);
    void *const s = h.stream();
    call([&] { return api.oxq_moe_group(ctx_of(h), s, idx, vals, E, off, tok, w, pos); });
    return pack(r);
    OXQ_BODY_END
}

// (ctx, logits, top_k, norm) -> top_idx, top_vals, offsets, tokens, weights, pos
PyObject *moe_route_group(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 4);
    const Handle &h = handle(a[0]);
    const Desc logits(a[1]);
    const at::Tensor &t = matrix(a[1]);
    const int64_t T = t.size(0), E = t.size(1), k = integer(a[2]);
    const int norm = (int)integer(a[3]);
    const auto dev = t.device();
    at::Tensor r[6] = {empty({T, k}, at::kInt, dev),   empty({T, k}, at::kFloat, dev), empty({E + 1}, at::kInt, dev),
                       empty({T * k}, at::kInt, dev),  empty({T * k}, at::kFloat, dev), empty({T, k}, at::kInt, dev)};
    const Desc idx(r[0]), vals(r[1]), off(r[2]), tok(r[3]), w(r[4]), pos(r[5]);
    void *const s = h.stream();
    call([&] { return api.oxq_moe_route_group(ctx_of(h), s, logits, k, norm, idx, vals, off, tok, w, pos); });
    return pack(r);
    OXQ_BODY_END
}

// (ctx, gate_up, out, kind, limit)
PyObject *gated_activation(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 5);
    const Handle &h = handle(a[0]);
    const Desc gu(a[1]);
    Out out(a[2], [&] {
        const at::Tensor &t = tensor(a[1]);
        return empty_rows(t, t.dim() ? t.size(-1) / 2 : 0);
    });
    const int kind = (int)integer(a[3]);
    const float limit = (float)real(a[4]);
    void *const s = h.stream();
    call([&] { return api.oxq_gated_activation(ctx_of(h), s, gu, kind, limit, out); });
    return out.get();
    OXQ_BODY_END
}

// (ctx, gate, up, out, kind)
PyObject *activation_mul(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 5);
    const Handle &h = handle(a[0]);
    const Desc gate(a[1]), up(a[2]);
    Out out(a[3], [&] { return empty_like(a[1]); });
    const int kind = (int)integer(a[4]);
    void *const s = h.stream();
    call([&] { return api.oxq_activation_mul(ctx_of(h), s, gate, up, kind, out); });
    return out.get();
    OXQ_BODY_END
}

// (ctx, expert_out, pair_pos, top_vals, out)
PyObject *moe_combine(PyObject *, PyObject *const *a, Py_ssize_t n) {
    OXQ_BODY_BEGIN
    want(n, 5);
    const Handle &h = handle(a[0]);
    const Desc y(a[1]), pos(a[2]), vals(a[3]);
    Out out(a[4], [&] {
        const at::Tensor &t = matrix(a[1]);
        return empty({tensor(a[2]).size(0), t.size(1)}, t.scalar_type(), t.device());
    });
    void *const s = h.stream();
    call([&] { return api.oxq_moe_combine(ctx_of(h), s, y, pos, vals, out); });
    return out.get();
    OXQ_BODY_END
}

// ---------------------------------------------------------------- module
PyObject *current_device(PyObject *, PyObject *) {
    OXQ_BODY_BEGIN
    return PyLong_FromLong(device());
    OXQ_BODY_END
}

// bind(dlopen handle, error class, descriptor class, torch.empty, torch.empty_like)
PyObject *bind(PyObject *, PyObject *args) {
    unsigned long long lib;
    PyObject *err, *st, *make, *like;
    if (!PyArg_ParseTuple(args, "KOOOO", &lib, &err, &st, &make, &like)) return nullptr;
#define OXQ_RESOLVE(f)                                                                           \
    if (!(api.f = (decltype(&::f))dlsym((void *)(uintptr_t)lib, #f)))                            \
        return PyErr_Format(PyExc_ImportError, "the library does not export %s", #f);
    OXQ_BOUND(OXQ_RESOLVE)
#undef OXQ_RESOLVE
    Py_INCREF(err);
    Py_XSETREF(error_class, err);
    Py_INCREF(st);
    Py_XSETREF(tensor_struct, st);
    Py_INCREF(make);
    Py_XSETREF(torch_empty, make);
    Py_INCREF(like);
    Py_XSETREF(torch_empty_like, like);
    Py_RETURN_NONE;
}

#define OXQ_FAST(f) (PyCFunction)(void (*)(void))(f), METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"current_device", current_device, METH_NOARGS, nullptr},
    {"w4a16_matmul", OXQ_FAST((packed_op<&Api::oxq_w4a16_matmul>)), nullptr},
    {"w8a16_matmul", OXQ_FAST((packed_op<&Api::oxq_w8a16_matmul>)), nullptr},
    {"gptq_matmul", OXQ_FAST(gptq_matmul), nullptr},
    {"mpp_quant_matmul", OXQ_FAST(mpp_quant_matmul), nullptr},
    {"f8_gemv", OXQ_FAST((f8_op<&Api::oxq_f8_gemv>)), nullptr},
    {"f8_matmul", OXQ_FAST((f8_op<&Api::oxq_f8_matmul>)), nullptr},
    {"gguf_quant_matmul", OXQ_FAST((gguf_op<&Api::oxq_gguf_quant_matmul>)), nullptr},
    {"gguf_quant_mul_mm", OXQ_FAST((gguf_op<&Api::oxq_gguf_quant_mul_mm>)), nullptr},
    {"mxfp4_matmul", OXQ_FAST(mxfp4_matmul), nullptr},
    {"experts_matmul", OXQ_FAST(experts_matmul), nullptr},
    {"experts_gate_up_swiglu", OXQ_FAST(experts_gate_up_swiglu), nullptr},
    {"moe_matmul", OXQ_FAST(moe_matmul), nullptr},
    {"moe_gate_up_swiglu", OXQ_FAST(moe_gate_up_swiglu), nullptr},
    {"moe_route", OXQ_FAST(moe_route), nullptr},
    {"moe_group", OXQ_FAST(moe_group), nullptr},
    {"moe_route_group", OXQ_FAST(moe_route_group), nullptr},
    {"gated_activation", OXQ_FAST(gated_activation), nullptr},
    {"activation_mul", OXQ_FAST(activation_mul), nullptr},
    {"moe_combine", OXQ_FAST(moe_combine), nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_oxq_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__oxq_torch() {
    HandleType.tp_name = "oxydllm_amd._oxq_torch.Handle";
    HandleType.tp_basicsize = sizeof(Handle);
    HandleType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    HandleType.tp_vectorcall_offset = offsetof(Handle, vectorcall);
    HandleType.tp_call = PyVectorcall_Call;
    HandleType.tp_new = handle_new;
    if (PyType_Ready(&HandleType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&HandleType);
    if (PyModule_AddObject(m, "Handle", (PyObject *)&HandleType) < 0 || PyModule_AddIntConstant(m, "KIND_MLP", KIND_MLP) < 0 ||
        PyModule_AddIntConstant(m, "KIND_PLAIN", KIND_PLAIN) < 0)
        return nullptr;
    return m;
}
