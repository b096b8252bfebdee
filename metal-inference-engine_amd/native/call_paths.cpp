// The decode step's calls from Python, with their checks in C++: for a batch of a few rows a kernel runs for 5-15 us,
// which is what the checks, allocations and the ctypes call of kernels.py take in Python. Each function here takes the
// arguments of its counterpart in kernels.py, and answers only where that counterpart would pass every tensor on as it
// is: plain torch tensors on one device with the types, shapes, strides and alignments the kernel reads. Then it makes
// the output and launches through the same C ABI entry point (addresses handed over once, by init). Anything else
// returns None and goes the general way, which converts, copies or refuses as it always did. Nothing is kept between
// calls: workspaces and counters are kernels.py's, passed in. C++ exceptions become Python's as torch's own bindings
// make them (an allocation that fails is torch.OutOfMemoryError, as from torch.empty).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include "../../include/rk_path.h"

namespace {

#define ENTRIES(X)                                                                                                  \
    X(rk_linear_workspace_bytes) X(rk_linear_rows_ex2) X(rk_swiglu_rows) X(rk_rms_norm) X(rk_layer_norm)             \
    X(rk_paged_decode_workspace_bytes) X(rk_paged_decode) X(rk_paged_decode_planned) X(rk_deltanet_decode)           \
    X(rk_attn_prep)
#define DECLARE(f) decltype(&::f) p_##f = nullptr;
ENTRIES(DECLARE)
#undef DECLARE
PyObject* on_error = nullptr;                      // on_error(entry, status) raises

// init({name: address}, on_error): the addresses of one library, whose interface must be the one compiled in here
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2 || !PyDict_Check(a[0])) return PyErr_Format(PyExc_TypeError, "init(dict, callable)");
    auto address = [&](const char* name) -> void* {
        PyObject* v = PyDict_GetItemString(a[0], name);
        return v ? PyLong_AsVoidPtr(v) : nullptr;
    };
    bool ok = true;
#define CHECK(f) ok = ok && address(#f);
    CHECK(rk_abi_version) ENTRIES(CHECK)
#undef CHECK
    if (!ok) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_KeyError, "init: an entry point is missing");
    const int version = reinterpret_cast<decltype(&::rk_abi_version)>(address("rk_abi_version"))();
    if (version != RK_ABI_VERSION)
        return PyErr_Format(PyExc_ImportError, "rk_calls.so was built for ABI version %d, the library has %d: build both again",
                            RK_ABI_VERSION, version);
#define FETCH(f) p_##f = reinterpret_cast<decltype(&::f)>(address(#f));
    ENTRIES(FETCH)
#undef FETCH
    Py_XINCREF(a[1]);
    Py_XSETREF(on_error, a[1]);
    Py_RETURN_NONE;
}

// a plain torch tensor (no subclass, no wrapper of a transform) on a ROCm device, or null
const at::Tensor* tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.has_storage() || !t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg() ||
        t.key_set().has_any(c10::functorch_transforms_ks))
        return nullptr;
    return &t;
}
bool is(const at::Tensor& t, at::ScalarType ty) { return t.scalar_type() == ty; }
bool at_(const at::Tensor& t, uintptr_t align) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % align == 0; }
bool same(const at::Tensor& a, const at::Tensor& b) { return a.device() == b.device(); }
void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
// The output's allocation and the launch run without the GIL, as torch.empty and a ctypes call do: either may wait (for
// memory to come free, for room in the device's queue), and other Python threads go on meanwhile. Whole statements: the
// scope ends before anything of Python's is touched.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
at::Tensor make(at::IntArrayRef sizes, const at::Tensor& like) { return at::empty(sizes, like.options().dtype(at::kFloat)); }

// fp32, contiguous, on x's device, of `n` values in the given shape; None gives true and null
bool plain(PyObject* o, const at::Tensor& x, at::IntArrayRef shape, const at::Tensor*& out) {
    out = nullptr;
    if (o == Py_None) return true;
    const at::Tensor* t = tensor(o);
    if (!t || !same(*t, x) || !is(*t, at::kFloat) || !t->is_contiguous() || t->sizes() != shape) return false;
    out = t;
    return true;
}

PyObject* finish(const char* entry, int rc, PyObject* result) {
    if (rc == RK_OK) return result;
    Py_XDECREF(result);
    PyObject* r = PyObject_CallFunction(on_error, "si", entry, rc);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s: status %d", entry, rc);
    return nullptr;
}

// a prepared weight: type code and its parts, of the shapes _weight_args asks for
struct Weight {
    const at::Tensor *data, *scales = nullptr, *mins = nullptr;
    long long N, K;
};
bool weight(PyObject* const* a, int wt, Weight& w) {   // data, scales, mins
    w.data = tensor(a[0]);
    if (!w.data || w.data->dim() != 2 || !w.data->is_contiguous() || !at_(*w.data, 16)) return false;
    w.N = w.data->size(0);
    w.K = w.data->size(1) * (wt == RK_W_INT4 ? 2 : 1);
    if (w.N < 1 || w.N > INT_MAX || w.K < 32 || w.K > INT_MAX || w.K % 32) return false;
    if (wt == RK_W_BF16) return is(*w.data, at::kBFloat16);
    if (!is(*w.data, wt == RK_W_INT8 ? at::kChar : at::kByte)) return false;
    for (int i = 0; i < (wt == RK_W_INT4 ? 2 : 1); ++i) {
        const at::Tensor* t = tensor(a[1 + i]);
        if (!t || !same(*t, *w.data) || !is(*t, at::kHalf) || !t->is_contiguous() || t->dim() != 2 || t->size(0) != w.N ||
            t->size(1) != w.K / 32)
            return false;
        (i ? w.mins : w.scales) = t;
    }
    return true;
}

// rows of K fp32 values with unit stride at a stride >= K of 4n, 16-byte aligned
bool rows_k(const at::Tensor& x, long long K, long long& ld) {
    const long long M = x.size(0);
    if (x.stride(1) != 1 || !at_(x, 16) || (M > 1 && (x.stride(0) % 4 || x.stride(0) < K))) return false;
    ld = M > 1 ? x.stride(0) : K;
    return true;
}

// linear(x, wt, data, scales, mins, N, K, bias, residual, ss, norm_w, eps, want_ss, glu, workspace, counters, stream)
//   -> y, or (y, tile sums of squares) with want_ss; ss given: the RMSNorm of x is applied; glu: y = silu * up
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 17) return PyErr_Format(PyExc_TypeError, "linear: 17 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor* x = tensor(a[0]);
        const int wt = (int)PyLong_AsLong(a[1]);
        Weight w;
        if (!x || x->dim() != 2 || !is(*x, at::kFloat) || !weight(a + 2, wt, w) || !same(*x, *w.data) ||
            PyLong_AsLongLong(a[5]) != w.N || PyLong_AsLongLong(a[6]) != w.K)
            Py_RETURN_NONE;
        const long long M = x->size(0), N = w.N, K = w.K;
        const bool want_ss = a[12] == Py_True, glu = a[13] == Py_True, norm = a[9] != Py_None;
        long long ld = 0, ss_ld = 0;
        if (M < 1 || M > 16 || x->size(1) != K || !rows_k(*x, K, ld) || (glu && N % 16)) Py_RETURN_NONE;
        const at::Tensor *bias, *res, *ss = nullptr, *nw = nullptr;
        if (!plain(a[7], *x, {N}, bias) || !plain(a[8], *x, {M, N}, res)) Py_RETURN_NONE;
        if (norm) {
            // the shapes rms_norm_linear and rms_norm_swiglu send to the fused norm
            const bool long_int8 = !glu && wt == RK_W_INT8 && N >= 65536 && K % 1024 == 0;
            if (M > 8 || K % 256 || K > 2048 || (N > 16384 && !long_int8)) Py_RETURN_NONE;
            if (!plain(a[9], *x, {M, K / 16}, ss) || !plain(a[10], *x, {K}, nw) || !nw || !at_(*nw, 16)) Py_RETURN_NONE;
            ss_ld = ss->stride(0);
        }
        const at::Tensor *ws = a[14] == Py_None ? nullptr : tensor(a[14]), *cnt = a[15] == Py_None ? nullptr : tensor(a[15]);
        const size_t need = p_rk_linear_workspace_bytes((int)M, (int)N, (int)K, wt);
        if (!cnt || !same(*cnt, *x) || cnt->numel() < (N + 15) / 16 ||
            (need && (!ws || !same(*ws, *x) || (size_t)ws->numel() < need)))
            Py_RETURN_NONE;
        void* stream = PyLong_AsVoidPtr(a[16]);
        const float eps = (float)PyFloat_AsDouble(a[11]);
        if (PyErr_Occurred()) return nullptr;
        at::Tensor y, sums;
        int rc;
        const int op = norm ? RK_X_RMS_NORM : RK_X_PLAIN;
        float* part = need ? static_cast<float*>(ws->data_ptr()) : nullptr;
        const size_t pb = need ? (size_t)ws->numel() : 0;
        {
            Unlocked scope;
            y = make({M, glu ? N / 2 : N}, *x);
            if (want_ss) sums = make({M, (N + 15) / 16}, *x);
            if (glu)
                rc = p_rk_swiglu_rows(y.data_ptr<float>(), x->data_ptr<float>(), ld, op, (const float*)ptr(ss), ss_ld,
                                      (const float*)ptr(nw), eps, (int)M, (int)(N / 2), (int)K, ptr(w.data), wt,
                                      ptr(w.scales), ptr(w.mins), part, pb, (uint32_t*)ptr(cnt), (int)cnt->numel(), stream);
            else
                rc = p_rk_linear_rows_ex2(y.data_ptr<float>(), want_ss ? sums.data_ptr<float>() : nullptr,
                                          x->data_ptr<float>(), ld, op, (const float*)ptr(ss), ss_ld, (const float*)ptr(nw),
                                          eps, (int)M, (int)N, (int)K, ptr(w.data), wt, ptr(w.scales), ptr(w.mins),
                                          (const float*)ptr(bias), (const float*)ptr(res), part, pb, (uint32_t*)ptr(cnt),
                                          (int)cnt->numel(), stream);
        }
        PyObject* out = THPVariable_Wrap(y);
        if (want_ss && out) {
            PyObject* s = THPVariable_Wrap(sums);
            PyObject* t = s ? PyTuple_Pack(2, out, s) : nullptr;
            Py_DECREF(out);
            Py_XDECREF(s);
            out = t;
        }
        return finish(glu ? "rk_swiglu_rows" : "rk_linear_rows_ex2", rc, out);
    END_HANDLE_TH_ERRORS
}

// norm(layer, x, w, eps, stream): rk_layer_norm (layer True) or rk_rms_norm of 2-D fp32 rows, fp32 weights
PyObject* norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) return PyErr_Format(PyExc_TypeError, "norm: 5 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor* x = tensor(a[1]);
        const at::Tensor* w;
        if (!x || x->dim() != 2 || !is(*x, at::kFloat) || x->size(0) < 1 || x->size(1) < 1 || x->size(0) > INT_MAX ||
            x->size(1) > INT_MAX || x->stride(1) != 1 || (x->size(0) > 1 && x->stride(0) < x->size(1)) ||
            a[2] == Py_None || !plain(a[2], *x, {x->size(1)}, w))
            Py_RETURN_NONE;
        void* stream = PyLong_AsVoidPtr(a[4]);
        const float eps = (float)PyFloat_AsDouble(a[3]);
        if (PyErr_Occurred()) return nullptr;
        at::Tensor y;
        const auto fn = a[0] == Py_True ? p_rk_layer_norm : p_rk_rms_norm;
        const long long ld = x->size(0) > 1 ? x->stride(0) : x->size(1);
        int rc;
        {
            Unlocked scope;
            y = make(x->sizes(), *x);
            rc = fn(y.data_ptr<float>(), x->data_ptr(), RK_F32, ld, w->data_ptr(), RK_F32, (int)x->size(0),
                    (int)x->size(1), eps, stream);
        }
        return finish(a[0] == Py_True ? "rk_layer_norm" : "rk_rms_norm", rc, THPVariable_Wrap(y));
    END_HANDLE_TH_ERRORS
}

int code(const at::Tensor& t) { return is(t, at::kFloat) ? RK_F32 : is(t, at::kBFloat16) ? RK_BF16 : -1; }

// a paged pool layer pair: [NB, bs, Hkv, d], one type, contiguous
bool pools(const at::Tensor* k, const at::Tensor* v) {
    return k && v && k->dim() == 4 && k->sizes() == v->sizes() && k->scalar_type() == v->scalar_type() && code(*k) >= 0 &&
           same(*k, *v) && k->is_contiguous() && v->is_contiguous() && k->size(0) <= INT_MAX && k->size(1) <= INT_MAX;
}

// paged_decode(q, k_pool, v_pool, tables, lens, block_size, window, gate, plan buffer, workspace, stream) -> [B, Hq, d]
PyObject* paged_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 11) return PyErr_Format(PyExc_TypeError, "paged_decode: 11 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]), *tb = tensor(a[3]), *ln = tensor(a[4]);
        if (!q || !tb || !ln || !pools(k, v) || q->dim() != 3 || !is(*q, at::kFloat) || !q->is_contiguous() ||
            !same(*q, *k) || !same(*q, *tb) || !same(*q, *ln) || !is(*tb, at::kInt) || !is(*ln, at::kInt) ||
            tb->dim() != 2 || ln->dim() != 1 || !tb->is_contiguous() || !ln->is_contiguous() || !at_(*q, 16))
            Py_RETURN_NONE;
        const long long B = q->size(0), Hq = q->size(1), d = q->size(2), bs = PyLong_AsLongLong(a[5]);
        const long long window = PyLong_AsLongLong(a[6]);
        if (PyErr_Occurred()) return nullptr;
        if (B < 1 || B > INT_MAX || k->size(3) != d || k->size(1) != bs || tb->size(0) != B || ln->size(0) != B ||
            tb->size(1) > INT_MAX || window < 0 || window > INT_MAX)
            Py_RETURN_NONE;
        const at::Tensor* gate = nullptr;
        if (a[7] != Py_None) {
            gate = tensor(a[7]);
            if (!gate || !same(*gate, *q) || !is(*gate, at::kFloat) || gate->dim() != 2 || gate->size(0) != B ||
                gate->size(1) != Hq * d || gate->stride(1) != 1 || gate->stride(0) % 4 || !at_(*gate, 16))
                Py_RETURN_NONE;
        }
        const at::Tensor *plan = a[8] == Py_None ? nullptr : tensor(a[8]), *ws = a[9] == Py_None ? nullptr : tensor(a[9]);
        const size_t need = p_rk_paged_decode_workspace_bytes((int)B, (int)Hq, (int)k->size(2), (int)d, (int)bs, (int)tb->size(1));
        if (!ws || !same(*ws, *q) || (size_t)ws->numel() < need || (a[8] != Py_None && !plan)) Py_RETURN_NONE;
        void* stream = PyLong_AsVoidPtr(a[10]);
        if (PyErr_Occurred()) return nullptr;
        at::Tensor out;
        const float* g = static_cast<const float*>(ptr(gate));
        const long long gld = gate ? gate->stride(0) : 0;
        int rc;
        {
            Unlocked scope;
            out = make({B, Hq, d}, *q);
            float* o = out.data_ptr<float>();
            rc = plan ? p_rk_paged_decode_planned(o, (const float*)ptr(q), ptr(k), ptr(v), code(*k), (const int32_t*)ptr(tb),
                                                  (const int32_t*)ptr(ln), (int)B, (int)Hq, (int)k->size(2), (int)d, (int)bs,
                                                  (int)tb->size(1), (int)k->size(0), (int)window, g, gld,
                                                  (int32_t*)ptr(plan), (size_t)plan->numel(), ws->data_ptr(),
                                                  (size_t)ws->numel(), stream)
                      : p_rk_paged_decode(o, (const float*)ptr(q), ptr(k), ptr(v), code(*k), (const int32_t*)ptr(tb),
                                          (const int32_t*)ptr(ln), (int)B, (int)Hq, (int)k->size(2), (int)d, (int)bs,
                                          (int)tb->size(1), (int)k->size(0), (int)window, g, gld, ws->data_ptr(),
                                          (size_t)ws->numel(), stream);
        }
        return finish(plan ? "rk_paged_decode_planned" : "rk_paged_decode", rc, THPVariable_Wrap(out));
    END_HANDLE_TH_ERRORS
}

// deltanet_decode(qkv, z, b, a, conv_state, S, seq_index, slot, conv_w, A_log, dt_bias, norm_w, eps, H, dk, dv, key_dim,
// stream) -> [B, H dv]
PyObject* deltanet_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 18) return PyErr_Format(PyExc_TypeError, "deltanet_decode: 18 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *qkv = tensor(a[0]), *z = tensor(a[1]), *b = tensor(a[2]), *aa = tensor(a[3]),
                         *conv = tensor(a[4]), *S = tensor(a[5]), *seq = tensor(a[6]);
        const at::Tensor *w = tensor(a[8]), *A = tensor(a[9]), *dt = tensor(a[10]), *nw = tensor(a[11]);
        for (const at::Tensor* t : {qkv, z, b, aa, conv, S, w, A, dt, nw})
            if (!t || !is(*t, at::kFloat) || !same(*t, *qkv)) Py_RETURN_NONE;
        if (!seq || !same(*seq, *qkv) || !is(*seq, at::kInt) || !seq->is_contiguous()) Py_RETURN_NONE;
        const long long slot = PyLong_AsLongLong(a[7]), H = PyLong_AsLongLong(a[13]), dk = PyLong_AsLongLong(a[14]),
                        dv = PyLong_AsLongLong(a[15]), key = PyLong_AsLongLong(a[16]);
        const float eps = (float)PyFloat_AsDouble(a[12]);
        void* stream = PyLong_AsVoidPtr(a[17]);
        if (PyErr_Occurred()) return nullptr;
        if (qkv->dim() != 2 || z->dim() != 2 || b->dim() != 2 || aa->dim() != 2 || S->dim() != 5 || conv->dim() != 4 ||
            w->dim() != 2 || key != H * dk)
            Py_RETURN_NONE;
        const long long B = qkv->size(0), C = qkv->size(1), nl = S->size(1), K = w->size(1);
        if (B < 1 || B > INT_MAX || C != 2 * key + H * dv || S->size(2) != H || S->size(3) != dk || S->size(4) != dv ||
            conv->size(3) != C || conv->size(1) != nl || conv->size(2) != K - 1 || slot < 0 || slot >= nl ||
            z->size(0) != B || z->size(1) != H * dv || b->size(0) != B || b->size(1) != H || aa->size(0) != B ||
            aa->size(1) != H || w->size(0) != C || A->numel() != H || dt->numel() != H || nw->numel() != dv ||
            seq->numel() != B || nl > INT_MAX)
            Py_RETURN_NONE;
        for (const at::Tensor* t : {conv, S, w, A, dt, nw})
            if (!t->is_contiguous()) Py_RETURN_NONE;
        for (const at::Tensor* t : {qkv, z, b, aa})
            if (t->stride(1) != 1) Py_RETURN_NONE;
        auto ld = [&](const at::Tensor* t) { return B > 1 ? t->stride(0) : t->size(1); };
        if (ld(b) != ld(aa)) Py_RETURN_NONE;
        at::Tensor out;
        auto f = [](const at::Tensor* t) { return static_cast<float*>(t->data_ptr()); };
        int rc;
        {
            Unlocked scope;
            out = make({B, H * dv}, *qkv);
            rc = p_rk_deltanet_decode(out.data_ptr<float>(), f(qkv), f(z), f(b), f(aa), ld(qkv), ld(z), ld(b), f(conv),
                                      f(S), f(w), f(A), f(dt), f(nw), static_cast<const int32_t*>(seq->data_ptr()),
                                      (int)B, (int)H, (int)dk, (int)dv, (int)K, (int)nl, (int)slot, eps, stream);
        }
        return finish("rk_deltanet_decode", rc, THPVariable_Wrap(out));
    END_HANDLE_TH_ERRORS
}

// attn_prep(y, q_w, k_w, eps, positions, inv_freq, rot, Hq, Hkv, d, k_pool, v_pool, slots, stream) -> q [N, Hq, d]:
// the decode form, which writes the pool
PyObject* attn_prep(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 14) return PyErr_Format(PyExc_TypeError, "attn_prep: 14 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *y = tensor(a[0]), *pos = tensor(a[4]), *k = tensor(a[10]), *v = tensor(a[11]), *sl = tensor(a[12]);
        const at::Tensor *inv = a[5] == Py_None ? nullptr : tensor(a[5]), *qw, *kw;
        const long long rot = PyLong_AsLongLong(a[6]), Hq = PyLong_AsLongLong(a[7]), Hkv = PyLong_AsLongLong(a[8]),
                        d = PyLong_AsLongLong(a[9]);
        const float eps = (float)PyFloat_AsDouble(a[3]);
        void* stream = PyLong_AsVoidPtr(a[13]);
        if (PyErr_Occurred()) return nullptr;
        if (!y || !pos || !sl || !pools(k, v) || (a[5] != Py_None && !inv) || y->dim() != 2 || !is(*y, at::kFloat) ||
            !same(*y, *pos) || !same(*y, *k) || !same(*y, *sl) || (inv && !same(*y, *inv)) || a[1] == Py_None ||
            a[2] == Py_None || !plain(a[1], *y, {d}, qw) || !plain(a[2], *y, {d}, kw) || d < 64 || d % 64 || rot < 0 ||
            rot > d || Hq < 1 || Hkv < 1)
            Py_RETURN_NONE;
        const long long N = y->size(0), per = d / 64;
        if (N < 1 || N > INT_MAX || y->size(1) < (Hq + 2 * Hkv) * d || y->stride(1) != 1 || y->stride(0) % per ||
            !at_(*y, per * 4) || !is(*pos, at::kInt) || pos->numel() != N || !pos->is_contiguous() || !is(*sl, at::kLong) ||
            sl->numel() != N || !sl->is_contiguous() || k->size(2) != Hkv || k->size(3) != d || (rot > 0) != (inv != nullptr) ||
            (inv && (!is(*inv, at::kFloat) || inv->numel() != rot / 2 || !inv->is_contiguous())))
            Py_RETURN_NONE;
        at::Tensor q;
        int rc;
        {
            Unlocked scope;
            q = make({N, Hq, d}, *y);
            rc = p_rk_attn_prep(q.data_ptr<float>(), nullptr, nullptr, ptr(k), ptr(v), code(*k),
                                static_cast<const int64_t*>(sl->data_ptr()), (int)k->size(0), (int)k->size(1),
                                y->data_ptr(), RK_F32, y->stride(0), (const float*)ptr(qw), (const float*)ptr(kw), eps,
                                static_cast<const int32_t*>(pos->data_ptr()), (const float*)ptr(inv), (int)rot, (int)N,
                                (int)Hq, (int)Hkv, (int)d, stream);
        }
        return finish("rk_attn_prep", rc, THPVariable_Wrap(q));
    END_HANDLE_TH_ERRORS
}

#define METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(init), METHOD(linear), METHOD(norm), METHOD(paged_decode), METHOD(deltanet_decode),
                         METHOD(attn_prep), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "rk_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_rk_calls(void) { return PyModule_Create(&module); }
