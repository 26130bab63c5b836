// sage_torch.cpp — the host side of the common calls, native (CPython extension _sage_host).
//
// attention_sage.py states the call surface: names, checks, error texts.  This module does the same work for
// calls that meet every check — allocate the outputs, carve the workspace, call the C ABI on the current
// stream — without the interpreter in between: a call of [1,64,4,64] takes 16.4 us of host time from Python and
// ctypes and 8.4 here, of which two launches are 5.  Anything it does not take (another dtype, a shape that must be
// refused, a tensor of a subclass, a tracer or a transform, a non-zero return code) comes back as None, and the
// Python function goes its own way and raises.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <map>
#include <mutex>
#include <utility>

#include "../../include/mi355_sage.h"

namespace {

// The C ABI's entry points, handed over by the ctypes loader: one library instance whatever its path.
struct Api {
    decltype(&mi355_sage_workspace_bytes) workspace_bytes;
    decltype(&mi355_sage_bwd_workspace_bytes) bwd_workspace_bytes;
    decltype(&mi355_sage_sdpa_bf16) sdpa;
    decltype(&mi355_sage_sdpa_bf16_train_fwd) train_fwd;
    decltype(&mi355_sage_sdpa_bf16_keymask) keymask;
    decltype(&mi355_sage_sdpa_bf16_mask_any) mask_any;
    decltype(&mi355_sage_sdpa_bf16_norm_rope) norm_rope;
    decltype(&mi355_sage_sdpa_bf16_norm_rope_train_fwd) norm_rope_train;
    decltype(&mi355_sage_sdpa_bwd_bf16) bwd;
    decltype(&mi355_sage_sdpa_bwd_f32_grads) bwd_f32;
    decltype(&mi355_sage_cast) cast;
} api;
constexpr int kApiEntries = sizeof(Api) / sizeof(void*);
static_assert(sizeof(Api) == kApiEntries * sizeof(void*), "one pointer per entry");

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// One growing buffer per (device, stream): steady-state calls allocate nothing and calls on different streams
// never share scratch memory.  A replaced buffer stays valid for the work queued on its stream: the
// allocator hands its memory out again only to that stream.  (Never destroyed: the device may be gone by then.)
// Order of locks: g_ws_mutex is taken without the interpreter's lock, because what happens under it — an
// allocation, the end of a tensor that Python has seen — may wait for that one.
std::mutex g_ws_mutex;
auto& g_ws = *new std::map<std::pair<int, void*>, at::Tensor>;

at::Tensor workspace(size_t nbytes, const at::Device& dev, void* stream) {
    at::Tensor replaced;                // (dies after the lock is released)
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    // (plain memory also when a mode is on for this thread: the buffer outlives it)
    c10::impl::ForceDispatchKeyGuard no_modes(c10::default_included_set, c10::default_excluded_set);
    at::Tensor& ws = g_ws[{dev.index(), stream}];
    if (!ws.defined() || (size_t)ws.numel() < nbytes) {
        at::Tensor grown = at::empty({(int64_t)nbytes}, at::TensorOptions().dtype(at::kByte).device(dev));
        replaced = std::exchange(ws, std::move(grown));
    }
    return ws;
}
size_t at_least(size_t n) { return n < 256 ? 256 : n; }

// Dense device memory and nothing else.  Every other kind of tensor — fake, functional, batched or wrapped by a
// transform, dual — carries a dispatch key or a tangent of its own; its sizes may be symbolic and it may have no
// memory to point to.
bool plain(const at::Tensor& t) {
    static const uint64_t keys = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
                                                      c10::DispatchKey::ADInplaceOrView}).raw_repr();
    return t.defined() && (t.key_set().raw_repr() & ~keys) == 0 && !t._fw_grad(0).defined();
}

struct Strides { int64_t s[4]; };
Strides bshd(const at::Tensor& t) { return Strides{{t.size(1) * t.size(2) * t.size(3), t.size(3), t.size(2) * t.size(3), 1}}; }

bool device_bhsd(const at::Tensor& t) { return t.dim() == 4 && t.is_cuda() && t.is_contiguous(); }
at::Tensor like(const at::Tensor& t, at::ScalarType dt) { return at::empty(t.sizes(), t.options().dtype(dt).requires_grad(false)); }

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// q [B,Sq,H,D], k and v [B,Skv,H,D], contiguous on one device, one dtype.
bool shapes_ok(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool square) {
    if (!device_bhsd(q) || !device_bhsd(k) || !device_bhsd(v) || k.sizes() != v.sizes()) return false;
    if (q.scalar_type() != k.scalar_type() || q.scalar_type() != v.scalar_type()) return false;
    if (q.device() != k.device() || q.device() != v.device()) return false;
    if (q.size(0) != k.size(0) || q.size(2) != k.size(2) || q.size(3) != k.size(3)) return false;
    return q.numel() > 0 && k.numel() > 0 && (!square || q.size(1) == k.size(1));
}

int cast(int n, const at::Tensor* const* src, at::Tensor* dst, bool to_bf16) {
    const void* s[4];
    void* d[4];
    int64_t len[4];
    for (int i = 0; i < n; i++) {
        dst[i] = like(*src[i], to_bf16 ? at::kBFloat16 : at::kFloat);
        s[i] = src[i]->data_ptr(); d[i] = dst[i].data_ptr(); len[i] = src[i]->numel();
    }
    return api.cast(n, s, d, len, to_bf16, stream_of(*src[0]));
}

enum Kind { kPlain = 0, kTrain = 1, kKeyMask = 2 };

// BF16 in, O (and Stats for kTrain) out; lo / hi: the masked key range, or hi = real_N_kv for kTrain.
int forward(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scale, int variant, int kind, int lo, int hi,
            at::Tensor& o, at::Tensor& stats) {
    const int B = q.size(0), Sq = q.size(1), H = q.size(2), D = q.size(3), Skv = k.size(1);
    const size_t need = api.workspace_bytes(B, H, Sq, Skv, D, variant);
    if (need == 0) return MI355_SAGE_EUNSUPPORTED;
    void* st = stream_of(q);
    o = like(q, at::kBFloat16);
    if (kind == kTrain) stats = at::empty({B, H, Sq, 1}, q.options().dtype(at::kFloat).requires_grad(false));
    const at::Tensor ws = workspace(at_least(need), q.device(), st);
    const Strides qs = bshd(q), ks = bshd(k);
    const void *pq = q.data_ptr(), *pk = k.data_ptr(), *pv = v.data_ptr();
    void *po = o.data_ptr(), *pw = ws.data_ptr();
    const size_t nw = (size_t)ws.numel();
    if (kind == kTrain)
        return api.train_fwd(pq, pk, pv, po, stats.data_ptr(), B, H, Sq, Skv, D, (float)scale, qs.s, ks.s, ks.s, qs.s, 0, 0, 0, 0, 0, 0,
                             Sq, hi, st, variant, pw, nw);
    if (kind == kKeyMask)
        return api.keymask(pq, pk, pv, po, nullptr, B, H, Sq, Skv, D, (float)scale, qs.s, ks.s, ks.s, qs.s, 0, 0, 0, 0, 0, lo, hi, st,
                           variant, pw, nw);
    return api.sdpa(pq, pk, pv, po, B, H, Sq, Skv, D, (float)scale, qs.s, ks.s, ks.s, qs.s, 0, 0, 0, 0, 0, st, variant, pw, nw);
}

// What the backward kernels read: shapes, types and devices of the saved set and the upstream gradient.
bool bwd_set_ok(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const at::Tensor& d, const at::Tensor& st,
                bool f32_ok) {
    if (!shapes_ok(q, k, v, false) || q.scalar_type() != at::kBFloat16) return false;
    for (const at::Tensor* t : {&o, &d})
        if (!device_bhsd(*t) || t->sizes() != q.sizes() || t->device() != q.device()) return false;
    if (o.scalar_type() != at::kBFloat16 || (d.scalar_type() != at::kBFloat16 && !(f32_ok && d.scalar_type() == at::kFloat))) return false;
    return st.scalar_type() == at::kFloat && st.is_cuda() && st.is_contiguous() && st.device() == q.device() &&
           st.numel() == q.size(0) * q.size(1) * q.size(2);
}

// Gradients of d_out's type, BF16 or F32.
int backward(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const at::Tensor& d_out,
             const at::Tensor& stats, double scale, int real_q, int real_kv, at::Tensor (&g)[3]) {
    const int B = q.size(0), Sq = q.size(1), H = q.size(2), D = q.size(3), Skv = k.size(1);
    const size_t need = api.bwd_workspace_bytes(B, H, Sq, Skv, D);
    if (need == 0) return MI355_SAGE_EUNSUPPORTED;
    void* st = stream_of(q);
    const at::ScalarType type = d_out.scalar_type();
    g[0] = like(q, type); g[1] = like(k, type); g[2] = like(v, type);
    const at::Tensor ws = workspace(at_least(need), q.device(), st);
    const Strides qs = bshd(q), ks = bshd(k);
    if (type == at::kFloat) {
        const at::Tensor d16 = like(d_out, at::kBFloat16);
        return api.bwd_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_out.data_ptr(), d16.data_ptr(), stats.data_ptr(),
                           g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr(), B, H, Sq, Skv, D, (float)scale, qs.s, ks.s, ks.s, qs.s, qs.s, qs.s,
                           ks.s, ks.s, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, real_q, real_kv, st, ws.data_ptr(), (size_t)ws.numel());
    }
    return api.bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_out.data_ptr(), stats.data_ptr(), g[0].data_ptr(),
                   g[1].data_ptr(), g[2].data_ptr(), B, H, Sq, Skv, D, (float)scale, qs.s, ks.s, ks.s, qs.s, qs.s, qs.s, ks.s, ks.s, 0, 0,
                   0, 0, 0, 0, 0, 0, 0, 0, real_q, real_kv, st, ws.data_ptr(), (size_t)ws.numel());
}

// The recorded attention node (attention_sage._SdpaNode): forward set saved, gradients by the flash backward,
// F32 activations cast at the boundary.
struct SdpaNode : torch::autograd::Function<SdpaNode> {
    static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                              double scale, int64_t variant) {
        at::Tensor b[3] = {q, k, v}, o, stats, out;
        const bool f32 = q.scalar_type() == at::kFloat;
        if (f32) {
            const at::Tensor* src[3] = {&q, &k, &v};
            TORCH_CHECK(cast(3, src, b, true) == 0, "record_sdpa: cast failed");
        }
        const int rc = ::forward(b[0], b[1], b[2], scale, (int)variant, kTrain, 0, k.size(1), o, stats);
        TORCH_CHECK(rc == 0, "sdpa_flash_train_fwd: shim rc=", rc);
        out = o;
        if (f32) {
            const at::Tensor* src[1] = {&o};
            TORCH_CHECK(cast(1, src, &out, false) == 0, "record_sdpa: cast failed");
        }
        ctx->save_for_backward({b[0], b[1], b[2], o, stats});
        ctx->saved_data["scale"] = scale;
        return out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble();
        const at::Tensor& g = grads[0];
        const at::Tensor& q = saved[0];
        at::Tensor d = g.is_contiguous() && aligned16(g) ? g : g.clone(at::MemoryFormat::Contiguous), out[3];
        if (d.scalar_type() != at::kFloat) d = d.to(at::kBFloat16);
        // (saved-tensor hooks may hand back anything)
        for (const at::Tensor& t : saved) TORCH_CHECK(plain(t), "sdpa_flash_backward_raw: a saved tensor came back without device memory");
        TORCH_CHECK(bwd_set_ok(q, saved[1], saved[2], saved[3], d, saved[4], true),
                    "sdpa_flash_backward_raw: a saved tensor came back with another shape, type, layout or device");
        const int rc = ::backward(q, saved[1], saved[2], saved[3], d, saved[4], scale, q.size(1), saved[1].size(1), out);
        TORCH_CHECK(rc == 0, "sdpa_flash_backward_raw: shim rc=", rc);
        if (g.scalar_type() != out[0].scalar_type())
            for (at::Tensor& t : out) t = t.to(g.scalar_type());
        return {out[0], out[1], out[2], at::Tensor(), at::Tensor()};
    }
};

// ---- argument access -----------------------------------------------------------------------------
// Taken: a plain torch.Tensor or Parameter (a subclass's results are of its type: left to the Python path).
bool tensor_arg(PyObject* o, const at::Tensor*& t) {
    if (!THPVariable_CheckExact(o)) return false;
    t = &THPVariable_Unpack(o);
    return plain(*t);
}
// A mode or transform is on for this thread (its allocations would not be plain tensors either).
bool intercepted() {
    return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~c10::default_included_set.raw_repr()) != 0;
}
bool double_arg(PyObject* o, double& x) {
    x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
bool int_arg(PyObject* o, int& x) {
    if (!PyLong_Check(o)) return false;
    const long n = PyLong_AsLong(o);
    if (n == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    x = (int)n;
    return x == n;
}
template <class F> int without_gil(F f) {
    PyThreadState* s = PyEval_SaveThread();
    int rc;
    try {
        rc = f();
    } catch (...) {
        PyEval_RestoreThread(s);
        throw;
    }
    PyEval_RestoreThread(s);
    return rc;
}

// What the interpreter calls: no C++ exception crosses its frames.  Out of memory, errors of the device and
// exceptions of Python hooks arrive as the Python exceptions torch raises for them.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)> PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
    try {
        return F(a, n);
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// fwd(q, k, v, scale, variant, kind, lo, hi, square) -> o, (o, stats) for kind 1, or None.  BF16; for the kinds
// without Stats also F32, cast at the boundary.
PyObject* py_fwd(PyObject* const* a, Py_ssize_t n) {
    const at::Tensor *q, *k, *v;
    double scale;
    int variant, kind, lo, hi, square;
    if (intercepted() || n != 9 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !double_arg(a[3], scale) || !int_arg(a[4], variant) ||
        !int_arg(a[5], kind) || !int_arg(a[6], lo) || !int_arg(a[7], hi) || !int_arg(a[8], square))
        Py_RETURN_NONE;
    if (!shapes_ok(*q, *k, *v, square != 0)) Py_RETURN_NONE;
    const bool f32 = q->scalar_type() == at::kFloat;
    if (q->scalar_type() != at::kBFloat16 && !(f32 && kind != kTrain)) Py_RETURN_NONE;
    at::Tensor o, stats;
    const int rc = without_gil([&] {
        if (!f32) return forward(*q, *k, *v, scale, variant, kind, lo, hi, o, stats);
        at::Tensor b[3], ob;
        const at::Tensor* src[3] = {q, k, v};
        int r = cast(3, src, b, true);
        if (r == 0) r = forward(b[0], b[1], b[2], scale, variant, kind, lo, hi, ob, stats);
        if (r != 0) return r;
        const at::Tensor* back[1] = {&ob};
        return cast(1, back, &o, false);
    });
    if (rc != 0) Py_RETURN_NONE;
    if (kind != kTrain) return THPVariable_Wrap(std::move(o));
    PyObject* t = PyTuple_New(2);
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(o)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(stats)));
    return t;
}

// bias(q, k, v, mask, scale, variant, square) -> o or None.  BF16, mask [B,H,Sq,Skv] with contiguous rows.
PyObject* py_bias(PyObject* const* a, Py_ssize_t n) {
    const at::Tensor *q, *k, *v, *m;
    double scale;
    int variant, square;
    if (intercepted() || n != 7 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !tensor_arg(a[3], m) || !double_arg(a[4], scale) ||
        !int_arg(a[5], variant) || !int_arg(a[6], square))
        Py_RETURN_NONE;
    if (!shapes_ok(*q, *k, *v, square != 0) || q->scalar_type() != at::kBFloat16 || m->scalar_type() != at::kBFloat16) Py_RETURN_NONE;
    const int B = q->size(0), Sq = q->size(1), H = q->size(2), D = q->size(3), Skv = k->size(1);
    if (m->dim() != 4 || m->device() != q->device() || m->size(0) != B || m->size(1) != H || m->size(2) != Sq || m->size(3) != Skv || m->stride(3) != 1)
        Py_RETURN_NONE;
    at::Tensor o;
    const int rc = without_gil([&] {
        const size_t need = api.workspace_bytes(B, H, Sq, Skv, D, variant);
        if (need == 0) return MI355_SAGE_EUNSUPPORTED;
        void* st = stream_of(*q);
        o = like(*q, at::kBFloat16);
        const at::Tensor ws = workspace(at_least(need), q->device(), st);
        const Strides qs = bshd(*q), ks = bshd(*k), ms{{m->stride(0), m->stride(1), m->stride(2), 1}};
        return api.mask_any(q->data_ptr(), k->data_ptr(), v->data_ptr(), m->data_ptr(), o.data_ptr(), B, H, Sq, Skv, D, (float)scale, qs.s,
                            ks.s, ks.s, ms.s, qs.s, 0, 0, 0, 0, 0, st, variant, ws.data_ptr(), (size_t)ws.numel());
    });
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(o));
}

// norm_rope(q, k, v, q_gain, k_gain, eps, cos, sin, scale, variant, blkq, blkk, k_flags, layout, train)
//   -> o, (o, stats) with train, or None.  BF16 with BF16 gains; layout as in the C ABI, without the table bit.
PyObject* py_norm_rope(PyObject* const* a, Py_ssize_t n) {
    const at::Tensor *q, *k, *v, *gq, *gk, *cs = nullptr, *sn = nullptr;
    double eps, scale;
    int variant, blkq, blkk, k_flags, layout, train;
    if (intercepted() || n != 15 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !tensor_arg(a[3], gq) || !tensor_arg(a[4], gk) ||
        !double_arg(a[5], eps) || !double_arg(a[8], scale) || !int_arg(a[9], variant) || !int_arg(a[10], blkq) || !int_arg(a[11], blkk) ||
        !int_arg(a[12], k_flags) || !int_arg(a[13], layout) || !int_arg(a[14], train))
        Py_RETURN_NONE;
    if ((a[6] == Py_None) != (a[7] == Py_None)) Py_RETURN_NONE;
    if (a[6] != Py_None && (!tensor_arg(a[6], cs) || !tensor_arg(a[7], sn))) Py_RETURN_NONE;
    if (!shapes_ok(*q, *k, *v, true) || q->scalar_type() != at::kBFloat16) Py_RETURN_NONE;
    const int B = q->size(0), S = q->size(1), H = q->size(2), D = q->size(3);
    const int64_t cols = (layout & MI355_SAGE_NORM_FULL_ROW) ? (int64_t)H * D : D;
    for (const at::Tensor* g : {gq, gk})
        if (g->scalar_type() != at::kBFloat16 || g->device() != q->device() || !g->is_contiguous() || g->numel() != cols) Py_RETURN_NONE;
    int64_t batch_rows = 0;
    if (cs) {
        if (cs->scalar_type() != sn->scalar_type() || (cs->scalar_type() != at::kFloat && cs->scalar_type() != at::kBFloat16)) Py_RETURN_NONE;
        if (cs->dim() != 2 || cs->sizes() != sn->sizes() || cs->size(1) != D / 2 || !cs->is_contiguous() || !sn->is_contiguous() ||
            cs->device() != q->device() || sn->device() != q->device())
            Py_RETURN_NONE;
        if (cs->scalar_type() == at::kBFloat16) layout |= MI355_SAGE_ROPE_TABLES_BF16;
        if (cs->size(0) == (int64_t)B * S * H && B > 1) batch_rows = (int64_t)S * H;
        else if (cs->size(0) != (int64_t)S * H) Py_RETURN_NONE;
    }
    at::Tensor o, stats;
    const int rc = without_gil([&] {
        const size_t need = api.workspace_bytes(B, H, S, S, D, variant);
        if (need == 0) return MI355_SAGE_EUNSUPPORTED;
        void* st = stream_of(*q);
        o = like(*q, at::kBFloat16);
        if (train) stats = at::empty({B, H, S, 1}, q->options().dtype(at::kFloat).requires_grad(false));
        const at::Tensor ws = workspace(at_least(need), q->device(), st);
        const Strides s = bshd(*q);
        const void *pc = cs ? cs->data_ptr() : nullptr, *ps = sn ? sn->data_ptr() : nullptr;
        if (train)
            return api.norm_rope_train(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), stats.data_ptr(), B, H, S, S, D, (float)scale,
                                       s.s, s.s, s.s, s.s, 0, 0, 0, 0, 0, 0, S, S, st, variant, gq->data_ptr(), gk->data_ptr(), (float)eps, pc,
                                       ps, batch_rows, layout, ws.data_ptr(), (size_t)ws.numel());
        return api.norm_rope(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), B, H, S, S, D, (float)scale, s.s, s.s, s.s, s.s, 0, 0, 0,
                             0, 0, st, variant, blkq, blkk, k_flags, gq->data_ptr(), gk->data_ptr(), (float)eps, pc, ps, batch_rows, layout,
                             ws.data_ptr(), (size_t)ws.numel());
    });
    if (rc != 0) Py_RETURN_NONE;
    if (!train) return THPVariable_Wrap(std::move(o));
    PyObject* t = PyTuple_New(2);
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(o)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(stats)));
    return t;
}

// bwd(q, k, v, o, d_out, stats, scale, real_q, real_kv) -> (d_q, d_k, d_v) or None.  BF16, Stats F32 contiguous.
PyObject* py_bwd(PyObject* const* a, Py_ssize_t n) {
    const at::Tensor *q, *k, *v, *o, *d, *st;
    double scale;
    int rq, rk;
    if (intercepted() || n != 9 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !tensor_arg(a[3], o) || !tensor_arg(a[4], d) ||
        !tensor_arg(a[5], st) || !double_arg(a[6], scale) || !int_arg(a[7], rq) || !int_arg(a[8], rk))
        Py_RETURN_NONE;
    if (!bwd_set_ok(*q, *k, *v, *o, *d, *st, false)) Py_RETURN_NONE;
    at::Tensor g[3];
    if (without_gil([&] { return backward(*q, *k, *v, *o, *d, *st, scale, rq, rk, g); }) != 0) Py_RETURN_NONE;
    PyObject* t = PyTuple_New(3);
    for (int i = 0; i < 3; i++) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(std::move(g[i])));
    return t;
}

// record(q, k, v, scale, variant) -> att with its node, or None.
PyObject* py_record(PyObject* const* a, Py_ssize_t n) {
    const at::Tensor *q, *k, *v;
    double scale;
    int variant;
    if (intercepted() || n != 5 || !tensor_arg(a[0], q) || !tensor_arg(a[1], k) || !tensor_arg(a[2], v) || !double_arg(a[3], scale) || !int_arg(a[4], variant))
        Py_RETURN_NONE;
    if (!shapes_ok(*q, *k, *v, true) || (q->scalar_type() != at::kBFloat16 && q->scalar_type() != at::kFloat)) Py_RETURN_NONE;
    // (what the kernels would refuse is left to the Python path, so that nothing can fail inside the node)
    if ((q->size(3) != 64 && q->size(3) != 128) || (variant != 0 && variant != 1) || !aligned16(*q) || !aligned16(*k) || !aligned16(*v)) Py_RETURN_NONE;
    at::Tensor out;
    without_gil([&] { out = SdpaNode::apply(*q, *k, *v, scale, (int64_t)variant); return 0; });
    return THPVariable_Wrap(std::move(out));
}

// workspace(nbytes, tensor) -> this (device, stream)'s buffer
PyObject* py_workspace(PyObject* const* a, Py_ssize_t n) {
    if (n != 2 || !PyLong_Check(a[0]) || !THPVariable_Check(a[1])) {
        PyErr_SetString(PyExc_TypeError, "workspace(nbytes, tensor)");
        return nullptr;
    }
    const at::Tensor* t = &THPVariable_Unpack(a[1]);
    TORCH_CHECK(plain(*t), "workspace: not a tensor with device memory");
    const size_t nbytes = PyLong_AsSize_t(a[0]);
    if (PyErr_Occurred()) return nullptr;
    at::Tensor ws;
    without_gil([&] { ws = workspace(nbytes, t->device(), stream_of(*t)); return 0; });
    return THPVariable_Wrap(std::move(ws));
}

// bind(addresses): the C ABI entry points, in the order of Api
PyObject* py_bind(PyObject* const* a, Py_ssize_t n) {
    if (n != kApiEntries) {
        PyErr_Format(PyExc_TypeError, "bind: %d addresses expected", kApiEntries);
        return nullptr;
    }
    void* p[kApiEntries];
    for (int i = 0; i < kApiEntries; i++) {
        p[i] = PyLong_AsVoidPtr(a[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    std::memcpy(&api, p, sizeof(api));
    Py_RETURN_NONE;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(entry<py_##name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(fwd), METHOD(bias), METHOD(norm_rope), METHOD(bwd), METHOD(record), METHOD(workspace), METHOD(bind), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_sage_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sage_host(void) { return PyModule_Create(&module_def); }
