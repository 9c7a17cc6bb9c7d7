// CPython module over the C ABI (include/kernl_hip.h): the per-call host work of the operators.
//
// Bounds a call on small inputs: the kernels there take 2 to 10 us, while the Python route to them — an autograd
// function, its autocast decorator, three tensor allocations, a device context and a ctypes call with 20 converted
// arguments — took 18 to 20 us per call.  Here one call reads the tensors' metadata, allocates the result and launches.
//
// Two kinds of functions:
//   *_fwd        what kernl_amd/_lib.py exposes under the same name: tensors in, one launch, no checks beyond the ABI's;
//   op_*, plan_* the whole operator for plain inputs (strided GPU tensors of one device, no autocast, nothing that autograd,
//                a tracer or a transform records).  Everything else — and every error — is answered with None: the caller then takes the Python
//                route, which casts, copies or raises as it always did.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/kernl_hip.h"

namespace {

PyObject *g_error = nullptr;  // KernlLibraryError of kernl_amd/_lib.py

// ---- arguments

struct BadArgument {};

const at::Tensor *tensor_or_null(PyObject *o) {
    if (o == Py_None) return nullptr;
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a tensor or None, got %s", Py_TYPE(o)->tp_name);
        throw BadArgument();
    }
    return &THPVariable_Unpack(o);
}

const at::Tensor &tensor(PyObject *o) {
    const at::Tensor *t = tensor_or_null(o);
    if (t == nullptr) {
        PyErr_SetString(PyExc_TypeError, "expected a tensor, got None");
        throw BadArgument();
    }
    return *t;
}

double number(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw BadArgument();
    return v;
}

int64_t integer(PyObject *o) {  // int(o): a float is cut off, a 0-d tensor is read
    PyObject *whole = PyLong_Check(o) ? (Py_INCREF(o), o) : PyNumber_Long(o);
    const int64_t v = whole == nullptr ? -1 : PyLong_AsLongLong(whole);
    Py_XDECREF(whole);
    if (v == -1 && PyErr_Occurred()) throw BadArgument();
    return v;
}

bool truth(PyObject *o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw BadArgument();
    return v != 0;
}

void count(Py_ssize_t got, Py_ssize_t want) {
    if (got != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
        throw BadArgument();
    }
}

int dtype_code(const at::Tensor &t) {
    switch (t.scalar_type()) {
        case at::kHalf: return KERNL_F16;
        case at::kBFloat16: return KERNL_BF16;
        case at::kFloat: return KERNL_F32;
        default: PyErr_SetString(PyExc_KeyError, "unsupported dtype"); throw BadArgument();
    }
}

void *data(const at::Tensor *t) { return t == nullptr ? nullptr : t->data_ptr(); }

void require_gpu(std::initializer_list<const at::Tensor *> tensors) {
    for (const at::Tensor *t : tensors)
        if (t != nullptr && !t->is_cuda()) {
            PyErr_SetString(g_error, "kernl_amd kernels need tensors on a GPU device (there is no CPU path)");
            throw BadArgument();
        }
}

void require_dims(const at::Tensor &t, int64_t dims) {
    if (t.dim() != dims) {
        PyErr_Format(PyExc_ValueError, "expected %lld dimensions, got %lld", (long long)dims, (long long)t.dim());
        throw BadArgument();
    }
}

// Calls `launch(stream)` with the tensor's device current and the GIL released, and raises what the library reports.
template <typename F>
PyObject *launched(const at::Tensor &on, const char *what, F &&launch) {
    const c10::DeviceGuard guard(on.device());
    void *stream = c10::hip::getCurrentHIPStream(on.device().index()).stream();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = launch(stream);
    Py_END_ALLOW_THREADS
    if (status != 0) {
        PyErr_Format(g_error, "%s failed with status %d: %s", what, status, kernl_last_error_string());
        throw BadArgument();
    }
    Py_RETURN_NONE;
}

template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *, PyObject *const *args, Py_ssize_t n) {
    // (PyTorch's own translation: a failed allocation is torch.OutOfMemoryError, which callers catch to try less)
    HANDLE_TH_ERRORS
    try {
        return F(args, n);
    } catch (const BadArgument &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// ---- the ABI's entry points on tensors

struct MaskArgs {
    const at::Tensor *mask;
    const int64_t *sizes = nullptr, *strides = nullptr;
    int dtype = KERNL_F32;
    explicit MaskArgs(const at::Tensor *m) : mask(m) {
        if (m == nullptr) return;
        require_dims(*m, 4);
        sizes = m->sizes().data();
        strides = m->strides().data();
        dtype = dtype_code(*m);
    }
};

PyObject *run_attention(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v, const at::Tensor &out, const at::Tensor *mask,
                        float scale, bool causal, int64_t start, float clamp) {
    const MaskArgs m(mask);
    const int dt = dtype_code(q);
    return launched(q, "kernl_attention_fwd", [&](void *stream) {
        if (causal && start != 0)
            return kernl_attention_cached_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), data(mask), q.size(0), q.size(1),
                                              q.size(2), k.size(2), q.size(3), q.strides().data(), k.strides().data(),
                                              v.strides().data(), out.strides().data(), m.sizes, m.strides, m.dtype, scale, start,
                                              clamp, dt, stream);
        return kernl_attention_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), data(mask), q.size(0), q.size(1), q.size(2),
                                   k.size(2), q.size(3), q.strides().data(), k.strides().data(), v.strides().data(),
                                   out.strides().data(), m.sizes, m.strides, m.dtype, scale, causal ? 1 : 0, clamp, dt, stream);
    });
}

PyObject *attention_fwd(PyObject *const *a, Py_ssize_t n) {  // q k v out mask scale causal clamp
    count(n, 8);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &out = tensor(a[3]), *mask = tensor_or_null(a[4]);
    require_gpu({&q, &k, &v, &out, mask});
    for (const at::Tensor *t : {&q, &k, &v, &out}) require_dims(*t, 4);
    return run_attention(q, k, v, out, mask, (float)number(a[5]), truth(a[6]), 0, (float)number(a[7]));
}

PyObject *attention_cached_fwd(PyObject *const *a, Py_ssize_t n) {  // q k v out mask scale start clamp
    count(n, 8);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &out = tensor(a[3]), *mask = tensor_or_null(a[4]);
    require_gpu({&q, &k, &v, &out, mask});
    for (const at::Tensor *t : {&q, &k, &v, &out}) require_dims(*t, 4);
    const MaskArgs m(mask);
    const int dt = dtype_code(q);
    const float scale = (float)number(a[5]), clamp = (float)number(a[7]);
    const int64_t start = integer(a[6]);
    return launched(q, "kernl_attention_cached_fwd", [&](void *stream) {
        return kernl_attention_cached_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), data(mask), q.size(0), q.size(1),
                                          q.size(2), k.size(2), q.size(3), q.strides().data(), k.strides().data(), v.strides().data(),
                                          out.strides().data(), m.sizes, m.strides, m.dtype, scale, start, clamp, dt, stream);
    });
}

PyObject *run_skinny(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v, const at::Tensor &out, const at::Tensor *mask,
                     const at::Tensor *ws, float scale, bool causal, float clamp) {
    const MaskArgs m(mask);
    const int dt = dtype_code(q);
    const auto entry = k.element_size() == 1 ? kernl_attention_skinny_kv8_fwd : kernl_attention_skinny_fwd;
    const int64_t ws_bytes = ws == nullptr ? 0 : (int64_t)ws->nbytes();
    return launched(q, "kernl_attention_skinny_fwd", [&](void *stream) {
        return entry(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), data(mask), data(ws), ws_bytes, q.size(0), q.size(1),
                     q.size(2), k.size(2), q.size(3), q.strides().data(), k.strides().data(), v.strides().data(), out.strides().data(),
                     m.sizes, m.strides, m.dtype, scale, causal ? 1 : 0, clamp, dt, stream);
    });
}

PyObject *attention_skinny_fwd(PyObject *const *a, Py_ssize_t n) {  // q k v out mask workspace scale causal clamp
    count(n, 9);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &out = tensor(a[3]);
    const at::Tensor *mask = tensor_or_null(a[4]), *ws = tensor_or_null(a[5]);
    require_gpu({&q, &k, &v, &out, mask, ws});
    for (const at::Tensor *t : {&q, &k, &v, &out}) require_dims(*t, 4);
    return run_skinny(q, k, v, out, mask, ws, (float)number(a[6]), truth(a[7]), (float)number(a[8]));
}

PyObject *run_linear(const at::Tensor &x, const at::Tensor &w, const at::Tensor *bias, const at::Tensor &out, const at::Tensor *act_in,
                     int act, int64_t M, int64_t N, int64_t K, const int64_t *xs, const int64_t *os) {
    const int dt = dtype_code(x);
    return launched(x, "kernl_linear_fwd", [&](void *stream) {
        return kernl_linear_fwd(x.data_ptr(), w.data_ptr(), data(bias), out.data_ptr(), data(act_in), M, N, K, xs, os,
                                act_in == nullptr ? nullptr : act_in->strides().data(), act, dt, stream);
    });
}

PyObject *linear_fwd(PyObject *const *a, Py_ssize_t n) {  // x2d w bias out2d act_in2d activation
    count(n, 6);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[3]);
    const at::Tensor *bias = tensor_or_null(a[2]), *act_in = tensor_or_null(a[4]);
    require_gpu({&x, &w, bias, &out, act_in});
    require_dims(x, 2);
    require_dims(out, 2);
    if (act_in != nullptr) require_dims(*act_in, 2);
    return run_linear(x, w, bias, out, act_in, (int)integer(a[5]), x.size(0), w.size(0), x.size(1), x.strides().data(),
                      out.strides().data());
}

PyObject *linear_rms_fwd(PyObject *const *a, Py_ssize_t n) {  // x2d rms_weight eps w bias out2d activation gated
    count(n, 8);
    const at::Tensor &x = tensor(a[0]), &g = tensor(a[1]), &w = tensor(a[3]), &out = tensor(a[5]), *bias = tensor_or_null(a[4]);
    require_gpu({&x, &g, &w, bias, &out});
    require_dims(x, 2);
    require_dims(out, 2);
    const float eps = (float)number(a[2]);
    const int act = (int)integer(a[6]), gated = truth(a[7]) ? 1 : 0, dt = dtype_code(x);
    return launched(x, "kernl_linear_rms_fwd", [&](void *stream) {
        return kernl_linear_rms_fwd(x.data_ptr(), g.data_ptr(), eps, w.data_ptr(), data(bias), out.data_ptr(), x.size(0), out.size(1),
                                    x.size(1), x.strides().data(), out.strides().data(), act, gated, dt, stream);
    });
}

// cos / sin [batch | 1, positions, head_dim]: a table of one batch entry is read with batch stride 0
struct TableArgs {
    const at::Tensor *cos, *sin;
    int64_t strides[3] = {0, 0, 0};
    int dtype = KERNL_F32;
    TableArgs(const at::Tensor *c, const at::Tensor *s) : cos(c), sin(s) {
        if (c == nullptr) return;
        if (s == nullptr) {
            PyErr_SetString(PyExc_ValueError, "cos and sin come together");
            throw BadArgument();
        }
        require_dims(*c, 3);
        require_dims(*s, 3);
        strides[0] = c->size(0) == 1 ? 0 : c->stride(0);
        strides[1] = c->stride(1);
        strides[2] = c->stride(2);
        dtype = dtype_code(*c);
    }
    const int64_t *table_strides() const { return cos == nullptr ? nullptr : strides; }
};

PyObject *linear_decode_fwd(PyObject *const *a, Py_ssize_t n) {
    // x2d rms_weight eps w bias residual2d out2d cos sin head_dim rope_cols rows_per_batch
    count(n, 12);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[3]), &out = tensor(a[6]);
    const at::Tensor *g = tensor_or_null(a[1]), *bias = tensor_or_null(a[4]), *res = tensor_or_null(a[5]);
    const TableArgs table(tensor_or_null(a[7]), tensor_or_null(a[8]));
    require_gpu({&x, g, &w, bias, res, &out, table.cos, table.sin});
    require_dims(x, 2);
    require_dims(out, 2);
    if (res != nullptr) require_dims(*res, 2);
    const float eps = (float)number(a[2]);
    const int64_t head_dim = integer(a[9]), rope_cols = integer(a[10]), rows_per_batch = integer(a[11]);
    const int dt = dtype_code(x);
    return launched(x, "kernl_linear_decode_fwd", [&](void *stream) {
        return kernl_linear_decode_fwd(x.data_ptr(), data(g), eps, w.data_ptr(), data(bias), data(res), out.data_ptr(), x.size(0),
                                       out.size(1), x.size(1), x.strides().data(), out.strides().data(),
                                       res == nullptr ? nullptr : res->strides().data(), data(table.cos), data(table.sin), head_dim,
                                       rope_cols, rows_per_batch, table.table_strides(), table.dtype, dt, stream);
    });
}

PyObject *linear_fewrow_fwd(PyObject *const *a, Py_ssize_t n) {
    // x2d w bias residual2d out2d activation workspace rms_weight eps gated cos sin head_dim rope_cols rows_per_batch
    count(n, 15);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[4]);
    const at::Tensor *bias = tensor_or_null(a[2]), *res = tensor_or_null(a[3]), *ws = tensor_or_null(a[6]), *g = tensor_or_null(a[7]);
    const TableArgs table(tensor_or_null(a[10]), tensor_or_null(a[11]));
    require_gpu({&x, &w, bias, res, &out, ws, g, table.cos, table.sin});
    require_dims(x, 2);
    require_dims(out, 2);
    if (res != nullptr) require_dims(*res, 2);
    const int act = (int)integer(a[5]), gated = truth(a[9]) ? 1 : 0, dt = dtype_code(x);
    const float eps = (float)number(a[8]);
    const int64_t head_dim = integer(a[12]), rope_cols = integer(a[13]), rows_per_batch = integer(a[14]);
    const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
    at::Tensor own;  // a fresh allocation per call: stream-ordered, so calls on different streams never share one
    if (ws == nullptr) {
        const int64_t need = kernl_linear_fewrow_workspace_bytes(M, N, K, gated, table.cos != nullptr ? 1 : 0);
        if (need > 0) {
            own = at::empty({need}, x.options().dtype(at::kByte));
            ws = &own;
        }
    }
    const int64_t ws_bytes = ws == nullptr ? 0 : (int64_t)ws->nbytes();
    const auto entry = w.element_size() == 2 ? kernl_linear_fewrow_fwd : kernl_linear_fewrow_w8_fwd;
    return launched(x, "kernl_linear_fewrow_fwd", [&](void *stream) {
        return entry(x.data_ptr(), data(g), eps, w.data_ptr(), data(bias), data(res), out.data_ptr(), data(ws), ws_bytes, M, N, K,
                     x.strides().data(), out.strides().data(), res == nullptr ? nullptr : res->strides().data(), data(table.cos),
                     data(table.sin), head_dim, rope_cols, rows_per_batch, table.table_strides(), table.dtype, act, gated, dt, stream);
    });
}

PyObject *run_layernorm(const at::Tensor &x, const at::Tensor &w, const at::Tensor *bias, const at::Tensor &out, const at::Tensor *mean,
                        const at::Tensor *rstd, float eps, bool rms, const at::Tensor *res, int64_t M, int64_t N, const int64_t *xs,
                        const int64_t *os, const int64_t *rs) {
    const int dt = dtype_code(x);
    float *mean_p = static_cast<float *>(data(mean)), *rstd_p = static_cast<float *>(data(rstd));
    return launched(x, res == nullptr ? "kernl_layernorm_fwd" : "kernl_add_layernorm_fwd", [&](void *stream) {
        if (res == nullptr)
            return kernl_layernorm_fwd(x.data_ptr(), w.data_ptr(), data(bias), out.data_ptr(), mean_p, rstd_p, M, N, xs[0], xs[1],
                                       os[0], os[1], eps, rms ? 1 : 0, dt, stream);
        return kernl_add_layernorm_fwd(x.data_ptr(), res->data_ptr(), w.data_ptr(), data(bias), out.data_ptr(), mean_p, rstd_p, M, N,
                                       xs[0], xs[1], rs[0], rs[1], os[0], os[1], eps, rms ? 1 : 0, dt, stream);
    });
}

PyObject *layernorm_fwd(PyObject *const *a, Py_ssize_t n) {  // x2d w bias out2d mean rstd eps rms residual2d
    count(n, 9);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[3]);
    const at::Tensor *bias = tensor_or_null(a[2]), *mean = tensor_or_null(a[4]), *rstd = tensor_or_null(a[5]), *res = tensor_or_null(a[8]);
    require_gpu({&x, &w, bias, &out, mean, rstd, res});
    require_dims(x, 2);
    require_dims(out, 2);
    if (res != nullptr) require_dims(*res, 2);
    return run_layernorm(x, w, bias, out, mean, rstd, (float)number(a[6]), truth(a[7]), res, x.size(0), x.size(1), x.strides().data(),
                         out.strides().data(), res == nullptr ? nullptr : res->strides().data());
}

// ---- whole operators

// What an operator runs right here: plain tensors on one GPU, outside autocast, with nothing for autograd to record — and
// nothing for anyone else who watches the operators go by: a launch made here is seen by no tracer, dispatch mode or
// functorch transform (vmap, jvp, grad), which the autograd functions of the Python route record or refuse.
bool plain_call() {
    static const c10::DispatchKeySet watchers({c10::DispatchKey::Tracer, c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                               c10::DispatchKey::FuncTorchDynamicLayerFrontMode});
    return !at::autocast::is_autocast_enabled(at::kCUDA) && !c10::impl::tls_local_dispatch_key_set().included_.has_any(watchers);
}

PyObject *takes_call(PyObject *const *, Py_ssize_t n) {  // whether plain tensors would be taken where this is called
    count(n, 0);
    return PyBool_FromLong(plain_call());
}

const at::Tensor *plain(PyObject *o, const c10::Device *device = nullptr) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
    if (device != nullptr && t.device() != *device) return nullptr;
    if (at::GradMode::is_enabled() && t.requires_grad()) return nullptr;
    if (t._fw_grad(0).defined()) return nullptr;  // a tangent (forward mode), with or without grad mode
    return &t;
}

// `o` may be None (then *out is null); false: not a plain tensor.
bool plain_or_none(PyObject *o, const c10::Device &device, const at::Tensor **out) {
    *out = nullptr;
    if (o == Py_None) return true;
    *out = plain(o, &device);
    return *out != nullptr;
}

bool sixteen_bit(const at::Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool aligned16(const at::Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
bool vector_of(const at::Tensor *t, const at::Tensor &like, int64_t n) {  // null, or a contiguous vector of n
    return t == nullptr || (t->scalar_type() == like.scalar_type() && t->dim() == 1 && t->size(0) == n && t->is_contiguous());
}

PyObject *op_layer_norm(PyObject *const *a, Py_ssize_t n) {  // x weight bias eps rms residual -> out | None
    count(n, 6);
    if (!plain_call()) Py_RETURN_NONE;
    const at::Tensor *x = plain(a[0]), *w, *bias, *res;
    if (x == nullptr || x->dim() == 0 || x->numel() == 0 || !x->is_contiguous()) Py_RETURN_NONE;
    const c10::Device device = x->device();
    w = plain(a[1], &device);
    if (w == nullptr || !plain_or_none(a[2], device, &bias) || !plain_or_none(a[5], device, &res)) Py_RETURN_NONE;
    const int64_t N = x->size(-1), M = x->numel() / N;
    if (!(sixteen_bit(*x) || x->scalar_type() == at::kFloat) || !vector_of(w, *x, N) || !vector_of(bias, *x, N)) Py_RETURN_NONE;
    if (res != nullptr && (res->sizes() != x->sizes() || res->scalar_type() != x->scalar_type() || !res->is_contiguous())) Py_RETURN_NONE;
    double eps = number(a[3]);
    if (x->scalar_type() == at::kHalf) eps = std::max(eps, 1.6e-5);  // the fp16 policy of the operator
    const at::Tensor out = at::empty(x->sizes(), x->options());
    const int64_t rows[2] = {N, 1};
    Py_XDECREF(run_layernorm(*x, *w, bias, out, nullptr, nullptr, (float)eps, truth(a[4]), res, M, N, rows, rows, rows));
    return THPVariable_Wrap(out);
}

// Shapes, types and mask of an attention call as implementations/attention.py asserts them.
bool attention_arguments(PyObject *const *a, const at::Tensor **q, const at::Tensor **k, const at::Tensor **v, const at::Tensor **out,
                         const at::Tensor **mask, float *clamp) {
    *q = plain(a[0]);
    if (*q == nullptr || (*q)->dim() != 4 || !sixteen_bit(**q)) return false;
    const c10::Device device = (*q)->device();
    *k = plain(a[1], &device);
    *v = plain(a[2], &device);
    *out = plain(a[3], &device);
    if (*k == nullptr || *v == nullptr || *out == nullptr || !plain_or_none(a[4], device, mask)) return false;
    const at::Tensor &Q = **q, &K = **k, &V = **v, &O = **out;
    if (K.scalar_type() != Q.scalar_type() || V.scalar_type() != Q.scalar_type() || O.scalar_type() != Q.scalar_type()) return false;
    if (K.dim() != 4 || K.sizes() != V.sizes() || O.sizes() != Q.sizes()) return false;
    if (K.size(0) != Q.size(0) || K.size(1) != Q.size(1) || K.size(3) != Q.size(3)) return false;
    *clamp = 0.0f;
    if (*mask != nullptr) {
        const at::Tensor &m = **mask;
        if (m.dim() != 4 || (m.size(0) != Q.size(0) && m.size(0) != 1) || (m.size(1) != Q.size(1) && m.size(1) != 1) ||
            (m.size(2) != Q.size(2) && m.size(2) != 1) || m.size(3) != K.size(2))
            return false;
        switch (m.scalar_type()) {  // smallest finite value of the mask's type
            case at::kHalf: *clamp = -65504.0f; break;
            case at::kBFloat16: *clamp = -3.3895313892515355e38f; break;
            case at::kFloat: *clamp = -3.4028234663852886e38f; break;
            default: return false;
        }
    }
    return true;
}

PyObject *op_attention(PyObject *const *a, Py_ssize_t n) {  // q k v out mask scale causal start -> out | None
    count(n, 8);
    if (!plain_call()) Py_RETURN_NONE;
    const at::Tensor *q, *k, *v, *out, *mask;
    float clamp;
    if (!attention_arguments(a, &q, &k, &v, &out, &mask, &clamp)) Py_RETURN_NONE;
    const bool causal = truth(a[6]);
    const int64_t start = causal && truth(a[7]) ? integer(a[7]) : 0;  // (looked at where it is used: None is as good as 0)
    Py_XDECREF(run_attention(*q, *k, *v, *out, mask, (float)number(a[5]), causal, start, clamp));
    Py_INCREF(a[3]);
    return a[3];
}

PyObject *op_skinny_attention(PyObject *const *a, Py_ssize_t n) {  // q k v out mask scale causal -> out | None
    count(n, 7);
    if (!plain_call()) Py_RETURN_NONE;
    const at::Tensor *q, *k, *v, *out, *mask;
    float clamp;
    if (!attention_arguments(a, &q, &k, &v, &out, &mask, &clamp)) Py_RETURN_NONE;
    const int64_t need = kernl_attention_skinny_workspace_bytes(q->size(0), q->size(1), q->size(2), k->size(2), q->size(3));
    at::Tensor ws;
    if (need > 0) ws = at::empty({need}, q->options().dtype(at::kByte));
    Py_XDECREF(run_skinny(*q, *k, *v, *out, mask, need > 0 ? &ws : nullptr, (float)number(a[5]), truth(a[6]), clamp));
    Py_INCREF(a[3]);
    return a[3];
}

// Rows that stream a weight on the stream-K kernel: `few_row_rule` of implementations/linear_layer.py (which says what was
// measured) with what `kernl_linear_fewrow_fwd` takes.
constexpr int64_t kFewRowMin = 17, kFewRowMax = 128, kFewRowMinWeight = 1 << 22, kFewRowLongK = 1536, kSplitKMaxRows = 2048, kFewRowLargeWeight = 24 << 20;

bool few_row_rule(int64_t rows, int64_t n, int64_t k, bool normed) {
    if (rows > 4 && rows < kFewRowMin && k % 64 == 0 && k >= 256)
        return n * k >= kFewRowLargeWeight && (normed ? rows >= 8 || k <= 8192 : rows >= 12 && k >= 5120);
    if (rows < kFewRowMin || rows > kFewRowMax || k < 256 || k % 64 != 0) return false;
    return n * k >= kFewRowMinWeight || (k >= kFewRowLongK && rows > 32);
}

// The rows of x: its shape seen as [M, K] with a row stride; false unless the features are contiguous.
struct Rows {
    int64_t M = 0, K = 0, strides[2] = {0, 1};
    bool of(const at::Tensor &x) {
        if (x.dim() < 1 || x.numel() == 0) return false;
        K = x.size(-1);
        M = x.numel() / K;
        if (x.dim() == 2) {
            strides[0] = x.stride(0);
            strides[1] = x.stride(1);
            return strides[1] == 1;
        }
        strides[0] = K;
        return x.is_contiguous();
    }
    bool vectors() const { return strides[0] % 8 == 0; }
};

at::Tensor rows_view(const at::Tensor &x, const Rows &r) { return x.dim() == 2 ? x : x.view({r.M, r.K}); }

at::Tensor output_for(const at::Tensor &x, int64_t N) {
    at::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    return at::empty(shape, x.options());
}

// x weight bias activation act_inputs small_kernels -> out, (x2d, out2d, out) for the stream-K kernel, or None
PyObject *op_linear(PyObject *const *a, Py_ssize_t n) {
    count(n, 6);
    if (!plain_call()) Py_RETURN_NONE;
    const at::Tensor *x = plain(a[0]), *w, *bias, *act_in;
    Rows r;
    if (x == nullptr || !sixteen_bit(*x) || !r.of(*x)) Py_RETURN_NONE;
    const c10::Device device = x->device();
    w = plain(a[1], &device);
    if (w == nullptr || !plain_or_none(a[2], device, &bias) || !plain_or_none(a[4], device, &act_in)) Py_RETURN_NONE;
    if (w->dim() != 2 || w->scalar_type() != x->scalar_type() || w->size(1) != r.K || w->size(0) == 0 || !w->is_contiguous()) Py_RETURN_NONE;
    const int64_t M = r.M, K = r.K, N = w->size(0);
    if (!vector_of(bias, *x, N)) Py_RETURN_NONE;
    if (act_in != nullptr && (act_in->dim() != 2 || act_in->size(0) != M || act_in->size(1) != N || act_in->scalar_type() != x->scalar_type()))
        Py_RETURN_NONE;
    const int act = (int)integer(a[3]);
    const bool vectors = r.vectors() && aligned16(*x) && aligned16(*w);
    if (vectors && K % 64 == 0 && M > 64 && r.strides[0] < (1 << 22)) {
        const int64_t need = kernl_linear_split_workspace_bytes(M, N, K, 0);
        if (need > 0) {  // too few tiles to occupy the chip: ranges of K per tile, added by a second launch
            const at::Tensor out = output_for(*x, N);
            const int64_t os[2] = {N, 1};
            const at::Tensor ws = at::empty({need}, x->options().dtype(at::kByte));
            const int dt = dtype_code(*x);
            Py_XDECREF(launched(*x, "kernl_linear_splitk_fwd", [&](void *stream) {
                return kernl_linear_splitk_fwd(x->data_ptr(), w->data_ptr(), data(bias), out.data_ptr(), data(act_in), ws.data_ptr(), need, M, N, K,
                                               r.strides, os, act_in == nullptr ? nullptr : act_in->strides().data(), act, dt, stream);
            }));
            return THPVariable_Wrap(out);
        }
    }
    const bool small = vectors && ((truth(a[5]) && kernl_linear_small_kind(M, N, K) != 0) ||
                                   (M > 64 && r.strides[0] < (1 << 22) && kernl_linear_mid_kind(M, N, K, 0) != 0));
    const at::Tensor out = output_for(*x, N);
    const int64_t os[2] = {N, 1};
    if (!small && vectors && K % 64 == 0 && act_in == nullptr && few_row_rule(M, N, K, false)) {
        PyObject *x2d = x->dim() == 2 ? (Py_INCREF(a[0]), a[0]) : THPVariable_Wrap(rows_view(*x, r));
        PyObject *y = THPVariable_Wrap(out);
        PyObject *y2d = out.dim() == 2 ? (Py_INCREF(y), y) : THPVariable_Wrap(out.view({M, N}));
        return Py_BuildValue("(NNN)", x2d, y2d, y);
    }
    Py_XDECREF(run_linear(*x, *w, bias, out, act_in, act, M, N, K, r.strides, os));
    return THPVariable_Wrap(out);
}

// What a projection of few rows needs before its launch, for the callers in implementations/linear_layer.py:
//   x weight bias rms_weight residual gated cos sin head_dim rope_cols
//   -> (x2d, residual2d | None, out2d, out, stream_k, rows_per_batch), or None where a check of the Python route fails
PyObject *plan_few_rows(PyObject *const *a, Py_ssize_t n) {
    count(n, 10);
    if (!plain_call()) Py_RETURN_NONE;
    const at::Tensor *x = plain(a[0]), *w, *bias, *g, *res, *cos, *sin;
    Rows r;
    if (x == nullptr || !sixteen_bit(*x) || !r.of(*x)) Py_RETURN_NONE;
    const c10::Device device = x->device();
    w = plain(a[1], &device);
    if (w == nullptr || !plain_or_none(a[2], device, &bias) || !plain_or_none(a[3], device, &g) || !plain_or_none(a[4], device, &res) ||
        !plain_or_none(a[6], device, &cos) || !plain_or_none(a[7], device, &sin))
        Py_RETURN_NONE;
    const bool gated = truth(a[5]);
    const int64_t head_dim = integer(a[8]), rope_cols = integer(a[9]);
    const int64_t M = r.M, K = r.K, rows = w->dim() == 2 ? w->size(0) : 0, N = gated ? rows / 2 : rows;
    if (w->dim() != 2 || w->scalar_type() != x->scalar_type() || w->size(1) != K || N == 0 || !w->is_contiguous() || !aligned16(*w))
        Py_RETURN_NONE;
    if (K % 64 != 0 || !r.vectors() || !aligned16(*x) || (gated && rows % 64 != 0)) Py_RETURN_NONE;
    if (!vector_of(bias, *x, rows) || !vector_of(g, *x, K)) Py_RETURN_NONE;
    const bool stream_k = few_row_rule(M, rows, K, g != nullptr) && (cos == nullptr || head_dim == 32 || head_dim == 64 || head_dim == 128);
    if (!stream_k && M > 64) Py_RETURN_NONE;
    const int64_t per_batch = x->dim() == 3 ? x->size(1) : M;
    if ((cos == nullptr) != (sin == nullptr)) Py_RETURN_NONE;
    if (cos != nullptr) {
        if (g == nullptr || cos->dim() != 3 || cos->sizes() != sin->sizes() || cos->strides() != sin->strides() ||
            cos->scalar_type() != sin->scalar_type() || cos->size(2) != head_dim || cos->size(1) != per_batch || cos->stride(2) != 1 ||
            (cos->size(0) != 1 && cos->size(0) != M / per_batch) || !(sixteen_bit(*cos) || cos->scalar_type() == at::kFloat))
            Py_RETURN_NONE;
        if (head_dim <= 0 || head_dim % 32 != 0 || N % head_dim != 0 || rope_cols < 0 || rope_cols > N || rope_cols % head_dim != 0)
            Py_RETURN_NONE;
    }
    if (res != nullptr && (res->scalar_type() != x->scalar_type() || res->numel() != M * N || !res->is_contiguous())) Py_RETURN_NONE;
    PyObject *x2d = x->dim() == 2 ? (Py_INCREF(a[0]), a[0]) : THPVariable_Wrap(rows_view(*x, r));
    const bool as_given = res == nullptr || (res->dim() == 2 && res->size(1) == N);
    PyObject *res2d = as_given ? (Py_INCREF(a[4]), a[4]) : THPVariable_Wrap(res->view({M, N}));
    const at::Tensor out = output_for(*x, N);
    PyObject *y = THPVariable_Wrap(out);
    PyObject *y2d = out.dim() == 2 ? (Py_INCREF(y), y) : THPVariable_Wrap(out.view({M, N}));
    return Py_BuildValue("(NNNNOL)", x2d, res2d, y2d, y, stream_k ? Py_True : Py_False, (long long)per_batch);
}

// Copies src[i] into dst[i] (lists of tensors of equal shapes and dtypes), all in one launch; None where some pair needs torch's copy.
PyObject *copy_many(PyObject *const *a, Py_ssize_t n) {
    count(n, 2);
    if (!PyList_Check(a[0]) || !PyList_Check(a[1])) Py_RETURN_NONE;
    const Py_ssize_t pairs = PyList_GET_SIZE(a[0]);
    if (pairs == 0 || pairs > 8 || PyList_GET_SIZE(a[1]) != pairs) Py_RETURN_NONE;
    void *dst[8];
    const void *src[8];
    int64_t bytes[8];
    const at::Tensor *first = nullptr;
    for (Py_ssize_t i = 0; i < pairs; ++i) {
        PyObject *d = PyList_GET_ITEM(a[0], i), *s = PyList_GET_ITEM(a[1], i);
        if (!THPVariable_CheckExact(d) || !THPVariable_CheckExact(s)) Py_RETURN_NONE;
        const at::Tensor &D = THPVariable_Unpack(d), &S = THPVariable_Unpack(s);
        if (first == nullptr) first = &D;
        if (!D.is_cuda() || D.device() != first->device() || S.device() != D.device() || S.scalar_type() != D.scalar_type() || S.sizes() != D.sizes() ||
            !S.is_contiguous() || !D.is_contiguous() || !aligned16(S) || !aligned16(D) || S.is_conj() || S.is_neg())
            Py_RETURN_NONE;
        dst[i] = D.data_ptr();
        src[i] = S.data_ptr();
        bytes[i] = (int64_t)S.nbytes();
    }
    for (Py_ssize_t i = 0; i < pairs; ++i)  // one after the other where one's source is another's destination
        for (Py_ssize_t j = 0; j < pairs; ++j) {
            const char *s = static_cast<const char *>(src[i]), *d = static_cast<const char *>(dst[j]);
            if (!(i == j && s == d) && s < d + bytes[j] && d < s + bytes[i]) Py_RETURN_NONE;
        }
    Py_DECREF(launched(*first, "kernl_copy_many", [&](void *stream) { return kernl_copy_many((int)pairs, src, dst, bytes, stream); }));
    Py_RETURN_TRUE;
}

PyObject *set_error_type(PyObject *, PyObject *type) {
    Py_XINCREF(type);
    Py_XSETREF(g_error, type);
    Py_RETURN_NONE;
}

#define ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<name>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ENTRY(attention_fwd), ENTRY(attention_cached_fwd), ENTRY(attention_skinny_fwd), ENTRY(linear_fwd), ENTRY(linear_rms_fwd),
    ENTRY(linear_decode_fwd), ENTRY(linear_fewrow_fwd), ENTRY(layernorm_fwd), ENTRY(op_layer_norm), ENTRY(op_attention),
    ENTRY(op_skinny_attention), ENTRY(op_linear), ENTRY(plan_few_rows), ENTRY(copy_many), ENTRY(takes_call),
    {"set_error_type", set_error_type, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Host side of the kernel library's calls.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject *m = PyModule_Create(&kModule);
    if (m == nullptr) return nullptr;
    g_error = PyExc_RuntimeError;
    Py_INCREF(g_error);
    PyObject *rule = Py_BuildValue("(LLLLL)", (long long)kFewRowMin, (long long)kFewRowMax, (long long)kFewRowMinWeight,
                                   (long long)kFewRowLongK, (long long)kSplitKMaxRows);
    if (rule == nullptr || PyModule_AddObject(m, "FEW_ROW_RULE", rule) < 0) return nullptr;
    return m;
}
