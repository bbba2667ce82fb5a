// Host side of the hot operators and of the modules' `forward`: argument checks, pointer and stride extraction, workspaces
// and the calls into libtrinity_hip.so, as a CPython extension over torch's C++ tensors.
//
// Why native: the decode-append step is 35 us of kernels behind some 60 us of Python -- nine tensors to check, two dozen
// attribute reads and a ctypes call per launch -- and every small operator is bound by that time alone (RMSNorm of 16 rows:
// 3 us of kernel, 14 us a call).  Measured with forwards back to back, us in Python / here: RMSNorm of 16 x 4096 13.5 /
// 3.6; LoRA on 16 tokens 35 / 8.2; decode-append with 16 new tokens on 1024 cached 59 / 35.5 (Llama3-8B widths), with
// KeyFormer's scores 70 / 39 (Falcon-7B widths) -- the last three are their kernels.  Host time of a forward 3 - 8 us.
//
// The functions take tensors by position (METH_FASTCALL).  Those named *_forward return True when they have enqueued the
// whole forward, and False -- having done nothing -- for tensors whose layout or type they do not cover; the caller then
// takes its general Python path.  Invalid arguments raise what that path raises: ValueError, or TrnError with the status.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <string>
#include <type_traits>
#include <vector>
#include "../../../include/trinity_hip.h"

namespace {

struct ValueErr { std::string msg; };
struct TrnErr { const char* fn; int status; };
struct PyErrSet {};      // a Python exception is already set
struct Declined { std::string why; };      // more than four dimensions: the general path may still flatten them

PyObject* g_trn_error = nullptr;      // triton_amd._lib.TrnError

std::string format(const char* f, ...) {
    char b[512];
    va_list ap;
    va_start(ap, f);
    vsnprintf(b, sizeof b, f, ap);
    va_end(ap);
    return b;
}
#define NEED(cond, ...) do { if (__builtin_expect(!(cond), 0)) throw ValueErr{format(__VA_ARGS__)}; } while (0)

// A call into libtrinity_hip.so without the interpreter lock, as ctypes makes it: a launch waits while its queue is full, and
// the process's other Python threads go on.  (The arguments are evaluated before, under the lock.)
template <class... P>
int unlocked(int (*fn)(P...), std::common_type_t<P>... args) {
    PyThreadState* const state = PyEval_SaveThread();
    const int status = fn(args...);
    PyEval_RestoreThread(state);
    return status;
}
#define CALL(fn, ...) do { const int st_ = unlocked(fn, __VA_ARGS__); if (__builtin_expect(st_ != 0, 0)) throw TrnErr{#fn, st_}; } while (0)

// A tensor as the C ABI needs it.
struct View {
    char* p = nullptr;
    int dim = 0;
    int64_t s[4] = {0, 0, 0, 0}, st[4] = {0, 0, 0, 0};
    c10::ScalarType dt = c10::ScalarType::Half;
    bool cuda = false;
    int dev = 0;
    bool half() const { return dt == c10::ScalarType::Half; }
    bool f32() const { return dt == c10::ScalarType::Float; }
    int64_t numel() const { int64_t n = 1; for (int i = 0; i < dim; ++i) n *= s[i]; return n; }
    bool unit() const { return dim == 0 || st[dim - 1] == 1; }
    bool contiguous() const {
        int64_t e = 1;
        for (int i = dim - 1; i >= 0; --i) {
            if (s[i] != 1 && st[i] != e) return false;
            e *= s[i];
        }
        return true;
    }
    std::string shape() const {
        std::string r = "(";
        for (int i = 0; i < dim; ++i) r += (i ? ", " : "") + std::to_string(s[i]);
        return r + (dim == 1 ? ",)" : ")");
    }
};

View view_of(const at::Tensor& t, const char* name) {
    View v;
    v.dim = (int)t.dim();
    if (v.dim > 4) throw Declined{format("%s: expected at most 4 dimensions, got %d", name, v.dim)};
    const auto sz = t.sizes();
    const auto sd = t.strides();
    for (int i = 0; i < v.dim; ++i) { v.s[i] = sz[i]; v.st[i] = sd[i]; }
    v.dt = t.scalar_type();
    v.cuda = t.is_cuda();
    v.dev = v.cuda ? t.get_device() : -1;
    v.p = static_cast<char*>(t.data_ptr());
    return v;
}
View arg(PyObject* o, const char* name) {
    NEED(THPVariable_Check(o), "%s: expected a tensor", name);
    return view_of(THPVariable_Unpack(o), name);
}
struct OptView { bool given = false; View v; void* p() const { return given ? v.p : nullptr; } };
OptView opt(PyObject* o, const char* name) { OptView r; if (o != Py_None) { r.given = true; r.v = arg(o, name); } return r; }
double num(PyObject* o) { const double d = PyFloat_AsDouble(o); if (d == -1.0 && PyErr_Occurred()) throw PyErrSet{}; return d; }
bool flag(PyObject* o) { const int r = PyObject_IsTrue(o); if (r < 0) throw PyErrSet{}; return r != 0; }
void count(Py_ssize_t n, Py_ssize_t want, const char* fn) {
    if (n != want) { PyErr_Format(PyExc_TypeError, "%s: expected %zd arguments, got %zd", fn, want, n); throw PyErrSet{}; }
}

void dev_half(const View& t, const char* n) {
    NEED(t.cuda, "%s: expected a GPU tensor", n);
    NEED(t.half(), "%s: expected float16, got %s", n, c10::toString(t.dt));
    NEED(t.unit(), "%s: innermost stride must be 1", n);
}
void dev_float(const View& t, const char* n) {
    NEED(t.cuda, "%s: expected a GPU tensor", n);
    NEED(t.f32(), "%s: expected float32, got %s", n, c10::toString(t.dt));
    NEED(t.unit(), "%s: innermost stride must be 1", n);
}
void* stream_of(const View& t) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)t.dev).stream(); }

// [H,S,D] as [1,H,S,D]; 4-D passes through.
View as4(const View& t, const char* n) {
    NEED(t.dim == 3 || t.dim == 4, "%s: expected [heads, seq, head_dim] or [batch, heads, seq, head_dim], got %s", n, t.shape().c_str());
    if (t.dim == 4) return t;
    View r = t;
    r.dim = 4;
    r.s[0] = 1; r.st[0] = t.s[0] * t.st[0];
    for (int i = 0; i < 3; ++i) { r.s[i + 1] = t.s[i]; r.st[i + 1] = t.st[i]; }
    return r;
}
View make(const View& like, char* p, std::initializer_list<int64_t> s, std::initializer_list<int64_t> st) {
    View r = like;
    r.p = p; r.dim = (int)s.size();
    int i = 0;
    for (int64_t x : s) r.s[i++] = x;
    i = 0;
    for (int64_t x : st) r.st[i++] = x;
    return r;
}
bool same_shape(const View& a, const View& b) {
    if (a.dim != b.dim) return false;
    for (int i = 0; i < a.dim; ++i) if (a.s[i] != b.s[i]) return false;
    return true;
}

// ---------------------------------------------------------------------------------------------- workspaces
// A module's workspaces by name, shape, type and device: found here under the interpreter lock, allocated -- on the first
// call that asks for one -- and owned by the module through `alloc(name, shape, dtype, device index, zeroed, optional)`, which
// refuses to under a graph capture, or for an optional one returns None: an undefined tensor here.  A forward holds the
// tensors it was given until it returns: between its launches another thread may release the module's.
struct Entry { std::string name; std::vector<int64_t> shape; c10::ScalarType dt; int dev; at::Tensor t; };
struct Workspaces { PyObject_HEAD std::vector<Entry>* e; PyObject* alloc; };

at::Tensor workspace(Workspaces* w, const char* name, at::IntArrayRef shape, c10::ScalarType dt, int dev, bool zeroed = false, bool optional = false) {
    for (const Entry& e : *w->e)
        if (e.dt == dt && e.dev == dev && at::IntArrayRef(e.shape) == shape && e.name == name) return e.t;
    PyObject* sh = PyTuple_New((Py_ssize_t)shape.size());
    if (!sh) throw PyErrSet{};
    for (size_t i = 0; i < shape.size(); ++i) PyTuple_SET_ITEM(sh, (Py_ssize_t)i, PyLong_FromLongLong(shape[i]));
    PyObject* t = PyObject_CallFunction(w->alloc, "sNsiii", name, sh, c10::toString(dt), dev, (int)zeroed, (int)optional);
    if (!t) throw PyErrSet{};
    at::Tensor r;
    if (t != Py_None) {
        r = THPVariable_Unpack(t);
        w->e->push_back(Entry{name, shape.vec(), dt, dev, r});
    }
    Py_DECREF(t);
    return r;
}
Workspaces* ws_arg(PyObject* o);
// Size at which a workspace of so many bytes is kept: the next power of two from 1 MB on, so that lengths share one (by exact
// size each length met would keep its own; all of them together are at most twice the largest).
int64_t kept_bytes(int64_t need) {
    int64_t n = (int64_t)1 << 20;
    while (n < need) n <<= 1;
    return n;
}

// ---------------------------------------------------------------------------------------------- operators
void rmsnorm_call(const View& x, const OptView& gamma, const View& y, double eps) {
    dev_half(x, "x"); dev_half(y, "y");
    NEED(x.dim == 2 && same_shape(x, y), "x %s / y %s: expected equal 2-D shapes", x.shape().c_str(), y.shape().c_str());
    if (gamma.given) {
        dev_half(gamma.v, "gamma");
        NEED(gamma.v.dim == 1 && gamma.v.s[0] == x.s[1], "gamma %s: expected (%lld,)", gamma.v.shape().c_str(), (long long)x.s[1]);
    }
    CALL(trn_rmsnorm_f16, x.p, gamma.p(), y.p, 1, x.s[0], x.s[1], 0, x.st[0], 0, y.st[0], 0, (float)eps, stream_of(x));
}
void head_rmsnorm_call(const View& x, const OptView& gamma, const View& y, double eps, int64_t row_start) {
    dev_half(x, "x"); dev_half(y, "y");
    NEED(x.dim == 3 && same_shape(x, y), "x, y: expected equal [heads, seq, head_dim] shapes");
    NEED(0 <= row_start && row_start <= x.s[1], "row_start out of range");
    if (gamma.given) {
        dev_half(gamma.v, "gamma");
        NEED(gamma.v.dim == 1 && gamma.v.s[0] == x.s[2], "gamma: expected (head_dim,)");
    }
    CALL(trn_rmsnorm_f16, x.p, gamma.p(), y.p, x.s[0], x.s[1] - row_start, x.s[2], x.st[0], x.st[1], y.st[0], y.st[1], row_start,
         (float)eps, stream_of(x));
}

trn_attn_desc attn_desc(const View& q, const View& k, const View& v, const View& o, double scale, bool causal) {
    dev_half(q, "q"); dev_half(k, "k");
    NEED(q.dim == 4, "q: expected [batch, heads, seq, head_dim], got %s", q.shape().c_str());
    NEED(k.dim == 4, "k: expected [batch, heads, seq, head_dim], got %s", k.shape().c_str());
    NEED(k.s[0] == q.s[0] && k.s[3] == q.s[3], "k %s does not match q %s", k.shape().c_str(), q.shape().c_str());
    dev_half(v, "v"); dev_half(o, "o");
    NEED(same_shape(v, k), "v %s must equal k %s", v.shape().c_str(), k.shape().c_str());
    NEED(same_shape(o, q), "o %s must equal q %s", o.shape().c_str(), q.shape().c_str());
    trn_attn_desc d{};
    d.batch = (int32_t)q.s[0]; d.n_q_heads = (int32_t)q.s[1]; d.n_kv_heads = (int32_t)k.s[1];
    d.seq_q = (int32_t)q.s[2]; d.seq_kv = (int32_t)k.s[2]; d.head_dim = (int32_t)q.s[3];
    d.q_stride_b = q.st[0]; d.q_stride_h = q.st[1]; d.q_stride_s = q.st[2];
    d.k_stride_b = k.st[0]; d.k_stride_h = k.st[1]; d.k_stride_s = k.st[2];
    d.v_stride_b = v.st[0]; d.v_stride_h = v.st[1]; d.v_stride_s = v.st[2];
    d.o_stride_b = o.st[0]; d.o_stride_h = o.st[1]; d.o_stride_s = o.st[2];
    d.scale = (float)scale; d.causal = causal ? 1 : 0; d.tau = 1.f;
    return d;
}
void add_noise(trn_attn_desc& d, const View& n, double tau) {
    NEED(n.cuda && n.unit() && (n.half() || n.f32()), "noise: expected a float32 or float16 GPU tensor with innermost stride 1");
    NEED(n.dim == 4 && n.s[0] == d.batch && n.s[1] == d.n_q_heads && n.s[2] == d.seq_q && n.s[3] == d.seq_kv,
         "noise %s: expected (%d, %d, %d, %d)", n.shape().c_str(), d.batch, d.n_q_heads, d.seq_q, d.seq_kv);
    d.noise_stride_b = n.st[0]; d.noise_stride_h = n.st[1]; d.noise_stride_s = n.st[2];
    d.tau = (float)tau;
}

void prenorm_qkv_call(const View& x, const OptView& gamma, const View (&w)[3], const View (&o)[3], double eps, bool norm) {
    static const char* wn[] = {"wq", "wk", "wv"};
    static const char* on[] = {"q_out", "k_out", "v_out"};
    dev_half(x, "x");
    NEED(x.dim == 2, "x: expected [tokens, hidden]");
    const int64_t T = x.s[0], K = x.s[1];
    for (int i = 0; i < 3; ++i) {
        dev_half(w[i], wn[i]);
        NEED(w[i].dim == 2 && w[i].s[0] == K, "%s: expected [hidden=%lld, n_out], got %s", wn[i], (long long)K, w[i].shape().c_str());
    }
    NEED(w[1].s[1] == w[2].s[1], "wk and wv must have the same number of columns");
    const int64_t D = o[0].dim > 0 ? o[0].s[o[0].dim - 1] : 0;
    for (int i = 0; i < 3; ++i) {
        dev_half(o[i], on[i]);
        NEED(o[i].dim == 3 && o[i].s[1] == T && o[i].s[2] == D && o[i].s[0] * D == w[i].s[1],
             "%s: expected [heads, %lld, %lld] with heads*%lld == %lld, got %s", on[i], (long long)T, (long long)D, (long long)D,
             (long long)w[i].s[1], o[i].shape().c_str());
    }
    if (gamma.given) {
        dev_half(gamma.v, "gamma");
        NEED(gamma.v.dim == 1 && gamma.v.s[0] == K, "gamma: expected (hidden,)");
    }
    CALL(trn_prenorm_qkv_f16, x.p, gamma.p(), w[0].p, w[1].p, w[2].p, o[0].p, o[1].p, o[2].p, T, K, w[0].s[1], w[1].s[1], D, x.st[0],
         w[0].st[0], w[1].st[0], w[2].st[0], o[0].st[0], o[0].st[1], o[1].st[0], o[1].st[1], o[2].st[0], o[2].st[1], (float)eps,
         norm ? 1 : 0, stream_of(x));
}

// ---------------------------------------------------------------------------------------------- functions
using Args = PyObject* const*;

bool f_rmsnorm(Args a, Py_ssize_t n) {                    // x, gamma | None, y, eps
    count(n, 4, "rmsnorm");
    rmsnorm_call(arg(a[0], "x"), opt(a[1], "gamma"), arg(a[2], "y"), num(a[3]));
    return true;
}

// RMSNorm.forward: X, X_norm of any shape whose leading axes flatten.
bool f_rmsnorm_forward(Args a, Py_ssize_t n) {            // eps, X, X_norm, gamma
    count(n, 4, "rmsnorm_forward");
    View x = arg(a[1], "X"), y = arg(a[2], "X_norm");
    // (an output of another shape is read as rows of X's width, and an empty one refused, by the general path)
    if (x.dim < 1 || y.dim < 1 || x.s[x.dim - 1] != y.s[y.dim - 1] || x.numel() == 0 || y.numel() == 0) return false;
    for (View* t : {&x, &y})
        if (t->dim != 2) {
            if (!t->contiguous()) return false;
            const int64_t c = t->s[t->dim - 1];
            *t = make(*t, t->p, {t->numel() / c, c}, {c, 1});
        }
    rmsnorm_call(x, opt(a[3], "gamma"), y, num(a[0]));
    return true;
}

// attention: q, k, v, o, scale, causal, lse | None, q_norm, gamma_q | None, q_eps, noise | None, tau, lse_pert | None, workspace | None
bool f_attention(Args a, Py_ssize_t n) {
    count(n, 14, "attention");
    const View q = arg(a[0], "q"), k = arg(a[1], "k"), v = arg(a[2], "v"), o = arg(a[3], "o");
    trn_attn_desc d = attn_desc(q, k, v, o, num(a[4]), flag(a[5]));
    d.q_norm = flag(a[7]) ? 1 : 0; d.q_norm_eps = (float)num(a[9]);
    const OptView noise = opt(a[10], "noise"), lse = opt(a[6], "lse"), lp = opt(a[12], "lse_pert"), g = opt(a[8], "gamma_q"), ws = opt(a[13], "workspace");
    if (noise.given) { dev_float(noise.v, "noise"); add_noise(d, noise.v, num(a[11])); }
    for (const OptView* r : {&lse, &lp}) {
        if (!r->given) continue;
        const char* nm = r == &lse ? "lse" : "lse_pert";
        dev_float(r->v, nm);
        NEED(r->v.dim == 3 && r->v.s[0] == d.batch && r->v.s[1] == d.n_q_heads && r->v.s[2] == d.seq_q && r->v.contiguous(),
             "%s: expected contiguous float32 (%d, %d, %d)", nm, d.batch, d.n_q_heads, d.seq_q);
    }
    if (g.given) {
        dev_half(g.v, "gamma_q");
        NEED(g.v.dim == 1 && g.v.s[0] == d.head_dim, "gamma_q: expected (head_dim,)");
    }
    NEED(!noise.given || lp.given, "noise given without lse_pert");
    if (ws.given) {
        NEED(ws.v.cuda && ws.v.contiguous() && ws.v.dt == c10::ScalarType::Byte, "workspace: expected a contiguous uint8 GPU tensor");
        CALL(trn_attn_fwd_ws_f16, &d, q.p, k.p, v.p, o.p, (float*)lse.p(), g.p(), (const float*)noise.p(), (float*)lp.p(), ws.v.p, ws.v.numel(), stream_of(q));
    } else {
        CALL(trn_attn_fwd_f16, &d, q.p, k.p, v.p, o.p, (float*)lse.p(), g.p(), (const float*)noise.p(), (float*)lp.p(), stream_of(q));
    }
    return true;
}

double scale_of(PyObject* o, int64_t head_dim) { return o == Py_None ? 1.0 / std::sqrt((double)head_dim) : num(o); }

bool f_attention_forward(Args a, Py_ssize_t n) {          // scale | None, causal, K, O, Q, V
    count(n, 6, "attention_forward");
    const View k = as4(arg(a[2], "K"), "K"), o = as4(arg(a[3], "O"), "O"), q = as4(arg(a[4], "Q"), "Q"), v = as4(arg(a[5], "V"), "V");
    const trn_attn_desc d = attn_desc(q, k, v, o, scale_of(a[0], q.s[3]), flag(a[1]));
    CALL(trn_attn_fwd_f16, &d, q.p, k.p, v.p, o.p, nullptr, nullptr, nullptr, nullptr, stream_of(q));
    return true;
}

bool f_qknorm_forward(Args a, Py_ssize_t n) {             // workspaces, scale | None, causal, eps, K, O, Q, V, gamma_k, gamma_q
    count(n, 10, "qknorm_forward");
    Workspaces* w = ws_arg(a[0]);
    View k = as4(arg(a[4], "K"), "K");
    const View o = as4(arg(a[5], "O"), "O"), q = as4(arg(a[6], "Q"), "Q"), v = as4(arg(a[7], "V"), "V");
    NEED(k.contiguous(), "K: expected a contiguous tensor");
    // (whose strides along axes of one element may be anything: a single KV head of a token-major tensor)
    k = make(k, k.p, {k.s[0], k.s[1], k.s[2], k.s[3]}, {k.s[1] * k.s[2] * k.s[3], k.s[2] * k.s[3], k.s[3], 1});
    NEED(k.cuda, "K: expected a GPU tensor");
    const double eps = num(a[3]);
    trn_attn_desc d = attn_desc(q, k, v, o, scale_of(a[1], k.s[3]), flag(a[2]));
    d.q_norm = 1; d.q_norm_eps = (float)eps;
    const OptView gq = opt(a[9], "gamma_q");
    if (gq.given) {
        dev_half(gq.v, "gamma_q");
        NEED(gq.v.dim == 1 && gq.v.s[0] == d.head_dim, "gamma_q: expected (head_dim,)");
    }
    const OptView gk = opt(a[8], "gamma_k");
    if (gk.given) {
        dev_half(gk.v, "gamma");
        NEED(gk.v.dim == 1 && gk.v.s[0] == d.head_dim, "gamma: expected (head_dim,)");
    }
    at::Tensor kn;
    if (trn_attn_qknorm_workspace_bytes(&d) > 0) kn = workspace(w, "k_norm", {k.s[0], k.s[1], k.s[2], k.s[3]}, k.dt, k.dev);
    CALL(trn_attn_qknorm_f16, &d, q.p, k.p, v.p, o.p, gq.p(), gk.p(), (float)eps, kn.defined() ? kn.data_ptr() : nullptr, stream_of(q));
    return true;
}

// Noise that the kernels read as it is.  fp16 rows and fp32 rows off the 16-byte grid that overlap (an expanded tensor) or lie
// too far apart for 32-bit offsets within a head -- by the bound of the statistics launch, the tighter one -- are copied by the
// general path; aligned fp32 has always been passed on.
bool direct_noise(const View& n) {
    if (!(n.half() || n.f32()) || !n.unit() || n.dim < 3) return false;
    bool aligned = n.f32() && reinterpret_cast<uintptr_t>(n.p) % 16 == 0;
    for (int i = 0; i < n.dim - 1; ++i) aligned = aligned && n.st[i] % 4 == 0;
    return aligned || (n.st[n.dim - 2] >= n.s[n.dim - 1] && (n.s[n.dim - 2] + TRN_STATS_SPARE_ROWS) * n.st[n.dim - 2] * 4 <= 0x7fffffffLL);
}

// the statistics tensors the kernels can write themselves
bool direct_outputs(const View& a, const View* b, int64_t numel) {
    if (!(a.half() || a.f32()) || !a.cuda || !a.contiguous() || a.numel() != numel) return false;
    return !b || (b->dt == a.dt && b->cuda && b->contiguous() && b->numel() == numel);
}

bool f_key_scores_forward(Args a, Py_ssize_t n) {         // workspaces, scale | None, causal, tau, mean_std, K, O, Q, V, C_out1, C_out2 | None, noise | None
    count(n, 12, "key_scores_forward");
    Workspaces* w = ws_arg(a[0]);
    const View k = as4(arg(a[5], "K"), "K"), o = as4(arg(a[6], "O"), "O"), q = as4(arg(a[7], "Q"), "Q"), v = as4(arg(a[8], "V"), "V");
    const View c1 = arg(a[9], "C_out");
    const OptView c2 = opt(a[10], "C_out2"), noise = opt(a[11], "noise");
    if (!q.cuda || !direct_outputs(c1, c2.given ? &c2.v : nullptr, q.s[0] * q.s[1] * k.s[2])) return false;
    if (noise.given && !direct_noise(noise.v)) return false;
    trn_attn_desc d = attn_desc(q, k, v, o, scale_of(a[1], q.s[3]), flag(a[2]));
    if (noise.given) add_noise(d, as4(noise.v, "noise"), num(a[3]));
    const at::Tensor rows = workspace(w, noise.given ? "lse_pert" : "lse", {q.s[0], q.s[1], q.s[2]}, c10::ScalarType::Float, q.dev);
    at::Tensor parts;
    int64_t need = noise.given ? trn_attn_key_scores_workspace_bytes(&d, noise.v.half() ? 2 : 3) : 0;
    if (need) {
        need = kept_bytes(need);
        parts = workspace(w, "key_parts", {need}, c10::ScalarType::Byte, q.dev, false, true);
        if (!parts.defined()) need = 0;             // (captured with noise of another type than the eager call's: without)
    }
    CALL(trn_attn_key_scores_f16, &d, q.p, k.p, v.p, o.p, noise.p(), noise.given && noise.v.half(), static_cast<float*>(rows.data_ptr()),
         c1.p, c2.p(), c1.half(), flag(a[4]), need ? parts.data_ptr() : nullptr, need, stream_of(q));
    return true;
}

bool f_prenorm_qkv(Args a, Py_ssize_t n) {                // x, gamma | None, wq, wk, wv, q_out, k_out, v_out, eps, norm
    count(n, 10, "prenorm_qkv");
    const View w[3] = {arg(a[2], "wq"), arg(a[3], "wk"), arg(a[4], "wv")}, o[3] = {arg(a[5], "q_out"), arg(a[6], "k_out"), arg(a[7], "v_out")};
    prenorm_qkv_call(arg(a[0], "x"), opt(a[1], "gamma"), w, o, num(a[8]), flag(a[9]));
    return true;
}

bool f_prenorm_forward(Args a, Py_ssize_t n) {            // workspaces, head_dim, scale | None, causal, eps, norm, O, WK, WQ, WV, X, gamma
    count(n, 12, "prenorm_forward");
    Workspaces* w = ws_arg(a[0]);
    const int64_t D = (int64_t)num(a[1]);
    const View O = arg(a[6], "O"), wk = arg(a[7], "WK"), wq = arg(a[8], "WQ"), wv = arg(a[9], "WV"), X = arg(a[10], "X");
    if (X.dim < 2 || X.dim > 3 || O.dim < 2 || O.dim > 3 || wq.dim != 2 || wk.dim != 2 || !X.cuda) return false;
    NEED(X.contiguous() && O.contiguous(), "X, O: expected contiguous tensors");
    const int64_t B = X.dim == 3 ? X.s[0] : 1, S = X.s[X.dim - 2], K = X.s[X.dim - 1], nq = wq.s[1], nkv = wk.s[1];
    if (D <= 0 || nq % D || nkv % D || O.numel() != B * S * nq) return false;
    const int64_t T = B * S, ld = nq + 2 * nkv;
    const at::Tensor qkv_ws = workspace(w, "qkv", {T, ld}, X.dt, X.dev);
    const View qkv = view_of(qkv_ws, "qkv");
    const View ws[3] = {wq, wk, wv};
    const int64_t off[3] = {0, nq, nq + nkv}, nn[3] = {nq, nkv, nkv};
    View hm[3], b4[3];
    for (int i = 0; i < 3; ++i) {
        hm[i] = make(qkv, qkv.p + 2 * off[i], {nn[i] / D, T, D}, {D, ld, 1});
        b4[i] = make(qkv, qkv.p + 2 * off[i], {B, nn[i] / D, S, D}, {S * ld, D, ld, 1});
    }
    const trn_attn_desc d = attn_desc(b4[0], b4[1], b4[2], make(O, O.p, {B, nq / D, S, D}, {S * nq, D, nq, 1}), scale_of(a[2], D), flag(a[3]));
    prenorm_qkv_call(make(X, X.p, {T, K}, {K, 1}), opt(a[11], "gamma"), ws, hm, num(a[4]), flag(a[5]));
    CALL(trn_attn_fwd_f16, &d, b4[0].p, b4[1].p, b4[2].p, O.p, nullptr, nullptr, nullptr, nullptr, stream_of(X));
    return true;
}

// The decode-append modules.
bool f_decode_forward(Args a, Py_ssize_t n) {
    // workspaces, head_dim, prenorm, scale, causal, head_major, q_norm, tau, K_cache, O2, V_cache, WK, WQ, WV, X, C_out1 | None,
    // C_out2 | None, noise | None
    count(n, 18, "decode_forward");
    Workspaces* w = ws_arg(a[0]);
    const int64_t D = (int64_t)num(a[1]);
    const bool prenorm = flag(a[2]), causal = flag(a[4]), head_major = flag(a[5]), q_norm = flag(a[6]);
    const double scale = num(a[3]);
    const View Kc = arg(a[8], "K_cache"), O2 = arg(a[9], "O2"), Vc = arg(a[10], "V_cache"), wk = arg(a[11], "WK"), wq = arg(a[12], "WQ"),
               wv = arg(a[13], "WV"), X = arg(a[14], "X");
    const OptView c1 = opt(a[15], "C_out"), c2 = opt(a[16], "C_out2"), noise = opt(a[17], "noise");
    if (X.dim != 2 || Kc.dim != 3 || !X.cuda || O2.dim != 2) return false;
    const int64_t M = X.s[0], N = X.s[1], H = Kc.s[0], PM = Kc.s[1], P = PM - M;
    NEED(H * D == N && P >= 0 && same_shape(Kc, Vc) && Kc.s[2] == D, "inconsistent shapes: X %s, caches %s, head_dim %lld", X.shape().c_str(),
         Kc.shape().c_str(), (long long)D);
    if (O2.s[0] != M || O2.s[1] != N || (head_major && !O2.contiguous())) return false;
    if (c1.given && !direct_outputs(c1.v, c2.given ? &c2.v : nullptr, H * PM)) return false;
    if (noise.given && !(noise.v.dim == 3 && direct_noise(noise.v))) return false;
    const at::Tensor q_ws = workspace(w, "q", {H, M, D}, X.dt, X.dev);
    const View q = view_of(q_ws, "q");
    const View q4 = as4(q, "q"), k4 = as4(Kc, "K_cache"), v4 = as4(Vc, "V_cache");
    const View o4 = head_major ? make(O2, O2.p, {1, H, M, D}, {H * M * D, M * D, D, 1}) : make(O2, O2.p, {1, H, M, D}, {M * O2.st[0], D, O2.st[0], 1});
    NEED(O2.unit(), "O2: innermost stride must be 1");
    trn_attn_desc d = attn_desc(q4, k4, v4, o4, scale, causal);
    d.q_norm = q_norm ? 1 : 0;
    if (noise.given) add_noise(d, as4(noise.v, "noise"), num(a[7]));
    int64_t need = c1.given ? 0 : trn_attn_workspace_bytes(&d);
    at::Tensor split;
    if (need) split = workspace(w, "attn_ws", {need}, c10::ScalarType::Byte, X.dev, true);
    else if ((need = c1.given ? trn_attn_key_scores_workspace_bytes(&d, noise.given) : trn_attn_chunk_workspace_bytes(&d)) > 0) {
        // one for chunks and caches of every length: by exact size each length would keep its own
        need = need <= TRN_ATTN_CHUNK_WORKSPACE_MAX(D) ? TRN_ATTN_CHUNK_WORKSPACE_MAX(D) : kept_bytes(need);
        split = workspace(w, "attn_shares", {need}, c10::ScalarType::Byte, X.dev, false, true);
        if (!split.defined()) need = 0;             // (captured, the cache grown long since the eager call: without)
    }
    void* const ws = need ? split.data_ptr() : nullptr;
    at::Tensor rows_ws;
    if (c1.given) rows_ws = workspace(w, noise.given ? "lse_pert" : "lse", {1, H, M}, c10::ScalarType::Float, X.dev);
    float* const rows = c1.given ? static_cast<float*>(rows_ws.data_ptr()) : nullptr;
    const View wts[3] = {wq, wk, wv};
    const View outs[3] = {q, make(Kc, Kc.p + 2 * P * Kc.st[1], {H, M, D}, {Kc.st[0], Kc.st[1], Kc.st[2]}),
                          make(Vc, Vc.p + 2 * P * Vc.st[1], {H, M, D}, {Vc.st[0], Vc.st[1], Vc.st[2]})};
    prenorm_qkv_call(X, OptView{}, wts, outs, 0.0, prenorm);
    if (q_norm) head_rmsnorm_call(Kc, OptView{}, Kc, 0.0, P);          // in place, the appended rows only
    if (c1.given)
        CALL(trn_attn_key_scores_f16, &d, q.p, Kc.p, Vc.p, o4.p, noise.p(), noise.given && noise.v.half(), rows, c1.v.p, c2.p(), c1.v.half(), 0,
             ws, need, stream_of(X));
    else
        CALL(trn_attn_fwd_ws_f16, &d, q.p, Kc.p, Vc.p, o4.p, nullptr, nullptr, nullptr, nullptr, ws, need, stream_of(X));
    return true;
}

bool f_lora_forward(Args a, Py_ssize_t n) {               // workspaces, A, B, O, W, X
    count(n, 6, "lora_forward");
    Workspaces* ws = ws_arg(a[0]);
    const View A = arg(a[1], "A"), B = arg(a[2], "B"), O = arg(a[3], "O"), W = arg(a[4], "W"), X = arg(a[5], "X");
    if (A.dim != 2 || B.dim != 2 || O.dim != 2 || W.dim != 2 || X.dim != 2 || !X.cuda) return false;
    const int64_t M = X.s[0], N = X.s[1], R = B.s[0], P = B.s[1];
    NEED(W.s[0] == N && W.s[1] == P && A.s[0] == N && A.s[1] == R && O.s[0] == M && O.s[1] == P,
         "inconsistent shapes: X %s, W %s, A %s, B %s, O %s", X.shape().c_str(), W.shape().c_str(), A.shape().c_str(), B.shape().c_str(), O.shape().c_str());
    const at::Tensor d_ws = workspace(ws, "D", {M, R}, X.dt, X.dev);
    const View d = view_of(d_ws, "D");
    dev_half(X, "x");
    for (const View* t : {&W, &A, &B}) dev_half(*t, "weights");
    dev_half(O, "outs"); dev_half(d, "outs");
    CALL(trn_lora_f16, X.p, M, N, X.st[0], W.p, P, W.st[0], A.p, R, A.st[0], B.p, B.st[0], O.p, O.st[0], d.p, d.st[0], stream_of(X));
    return true;
}

bool f_gmlp_forward(Args a, Py_ssize_t n) {               // workspaces, silu, O, W1, W2, X
    count(n, 6, "gmlp_forward");
    Workspaces* ws = ws_arg(a[0]);
    const View O = arg(a[2], "O"), W1 = arg(a[3], "W1"), W2 = arg(a[4], "W2"), X = arg(a[5], "X");
    if (O.dim != 2 || W1.dim != 2 || W2.dim != 2 || X.dim != 2 || !X.cuda) return false;
    NEED(W1.s[0] == X.s[1] && same_shape(W1, W2) && O.s[0] == X.s[0] && O.s[1] == W1.s[1], "inconsistent shapes: X %s, W1 %s, W2 %s, O %s",
         X.shape().c_str(), W1.shape().c_str(), W2.shape().c_str(), O.shape().c_str());
    const at::Tensor c2_ws = workspace(ws, "C2", {O.s[0], O.s[1]}, X.dt, X.dev);
    const View c2 = view_of(c2_ws, "C2");
    dev_half(X, "x"); dev_half(W1, "weights"); dev_half(W2, "weights"); dev_half(O, "outs"); dev_half(c2, "outs");
    CALL(trn_gated_mlp_f16, X.p, X.s[0], X.s[1], X.st[0], W1.p, W1.st[0], W2.p, W2.st[0], W1.s[1], O.p, O.st[0], c2.p, c2.st[0],
         flag(a[1]) ? 1 : 0, stream_of(X));
    return true;
}

// ---------------------------------------------------------------------------------------------- Python glue
PyObject* raise_trn(const char* fn, int status) {
    if (!g_trn_error) { PyErr_Format(PyExc_RuntimeError, "%s failed: %s (%d)", fn, trn_status_name(status), status); return nullptr; }
    PyObject* e = PyObject_CallFunction(g_trn_error, "sis", fn, status, trn_status_name(status));
    if (e) { PyErr_SetObject(g_trn_error, e); Py_DECREF(e); }
    return nullptr;
}
// OP: an operator of its own, which has no general path behind it.
template <bool (*F)(Args, Py_ssize_t), bool OP>
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
    try {
        if (F(a, n)) Py_RETURN_TRUE;
        Py_RETURN_FALSE;
    } catch (const ValueErr& e) {
        PyErr_SetString(PyExc_ValueError, e.msg.c_str());
    } catch (const Declined& e) {
        if (!OP) Py_RETURN_FALSE;
        PyErr_SetString(PyExc_ValueError, e.why.c_str());
    } catch (const TrnErr& e) {
        return raise_trn(e.fn, e.status);
    } catch (const PyErrSet&) {
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyObject* ws_new(PyTypeObject* t, PyObject* args, PyObject*) {
    PyObject* alloc;
    if (!PyArg_ParseTuple(args, "O", &alloc)) return nullptr;
    Workspaces* w = reinterpret_cast<Workspaces*>(t->tp_alloc(t, 0));
    if (!w) return nullptr;
    w->e = new std::vector<Entry>();
    Py_INCREF(alloc);
    w->alloc = alloc;
    return reinterpret_cast<PyObject*>(w);
}
void ws_dealloc(PyObject* o) {
    delete reinterpret_cast<Workspaces*>(o)->e;
    Py_XDECREF(reinterpret_cast<Workspaces*>(o)->alloc);
    Py_TYPE(o)->tp_free(o);
}
PyObject* ws_clear(PyObject* o, PyObject*) {
    reinterpret_cast<Workspaces*>(o)->e->clear();
    Py_RETURN_NONE;
}
Py_ssize_t ws_len(PyObject* o) { return (Py_ssize_t)reinterpret_cast<Workspaces*>(o)->e->size(); }
PyMethodDef ws_methods[] = {{"clear", ws_clear, METH_NOARGS, "forget every tensor"}, {nullptr, nullptr, 0, nullptr}};
PySequenceMethods ws_seq = {ws_len};
PyTypeObject ws_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
Workspaces* ws_arg(PyObject* o) {
    if (Py_TYPE(o) != &ws_type) { PyErr_SetString(PyExc_TypeError, "expected Workspaces"); throw PyErrSet{}; }
    return reinterpret_cast<Workspaces*>(o);
}

PyObject* set_error_class(PyObject*, PyObject* cls) {
    Py_XDECREF(g_trn_error);
    Py_INCREF(cls);
    g_trn_error = cls;
    Py_RETURN_NONE;
}

#define FN(name) {#name, (PyCFunction)(void (*)(void))entry<f_##name, false>, METH_FASTCALL, nullptr}
#define OPERATOR(name) {#name, (PyCFunction)(void (*)(void))entry<f_##name, true>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {OPERATOR(rmsnorm), OPERATOR(attention), OPERATOR(prenorm_qkv), FN(rmsnorm_forward), FN(attention_forward),
                         FN(qknorm_forward), FN(key_scores_forward), FN(prenorm_forward), FN(decode_forward), FN(lora_forward), FN(gmlp_forward),
                         {"set_error_class", set_error_class, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "host side of the modules' forward", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    ws_type.tp_name = "triton_amd._host.Workspaces";
    ws_type.tp_basicsize = sizeof(Workspaces);
    ws_type.tp_flags = Py_TPFLAGS_DEFAULT;
    ws_type.tp_new = ws_new;
    ws_type.tp_dealloc = ws_dealloc;
    ws_type.tp_methods = ws_methods;
    ws_type.tp_as_sequence = &ws_seq;
    if (PyType_Ready(&ws_type) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&ws_type);
    if (PyModule_AddObject(m, "Workspaces", reinterpret_cast<PyObject*>(&ws_type)) < 0) return nullptr;
    return m;
}
