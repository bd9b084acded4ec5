// The eager ops' argument checks and calls into liblfm2q as a CPython module (lfm2opt.kernels wraps it). A small op is
// bound by the host: checked and called from Python through ctypes, a GEMV of 4.3 us took 11.1 us a call and a quantize +
// GEMM pair of 14 us 34 (6.5 and 22 from here). The checks and messages are the ones the ops document; every function takes the op's arguments in
// the op's order, launches on torch's current stream of the first tensor's device and returns None.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdexcept>
#include <string>

#include "lfm2q.h"

namespace {

using at::Tensor;

[[noreturn]] void fail(const std::string &msg) { throw std::runtime_error(msg); }
void require(bool ok, const char *msg) {
    if (!ok) fail(msg);
}

// an argument that must be a tensor, and one that may be None (a null pointer then)
const Tensor &tensor(PyObject *o, const char *name) {
    if (!THPVariable_Check(o)) fail(std::string(name) + " must be a tensor");
    return THPVariable_Unpack(o);
}
const Tensor *optional(PyObject *o, const char *name) { return o == Py_None ? nullptr : &tensor(o, name); }

const char *dtype_name(at::ScalarType t) {
    switch (t) {
        case at::kChar: return "torch.int8";
        case at::kFloat: return "torch.float32";
        case at::kInt: return "torch.int32";
        default: return "dtype";
    }
}
const Tensor &bf16(PyObject *o, const char *name) {
    const Tensor &t = tensor(o, name);
    if (!(t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.is_contiguous()))
        fail(std::string(name) + " must be contiguous CUDA bf16");
    return t;
}
const Tensor &typed(PyObject *o, at::ScalarType dt, const char *name) {
    const Tensor &t = tensor(o, name);
    if (!(t.is_cuda() && t.scalar_type() == dt && t.is_contiguous()))
        fail(std::string(name) + " must be contiguous CUDA " + dtype_name(dt));
    return t;
}
const Tensor *opt_bf16(PyObject *o, const char *name) { return o == Py_None ? nullptr : &bf16(o, name); }

template <typename... T>
void same_device(const Tensor &a, const T *...rest) {
    const bool ok = ((rest == nullptr || rest->device() == a.device()) && ...);
    require(ok, "all tensors must be on the same device");
}

template <typename T>
T *ptr(const Tensor &t) {
    return static_cast<T *>(t.data_ptr());
}
template <typename T>
T *ptr(const Tensor *t) {
    return t ? static_cast<T *>(t->data_ptr()) : nullptr;
}
lfm2q_stream_t stream(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool truth(PyObject *o) {
    const int r = PyObject_IsTrue(o);
    if (r < 0) throw std::invalid_argument("");  // the Python error is set
    return r != 0;
}
long integer(PyObject *o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw std::invalid_argument("");
    return v;
}
float real(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw std::invalid_argument("");
    return (float)v;
}

// The interpreter lock released for a scope, and taken again however the scope is left
class Unlocked {
    PyThreadState *state = PyEval_SaveThread();

  public:
    Unlocked() = default;
    Unlocked(const Unlocked &) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// The library call f(a..., the current stream of on's device) without the interpreter lock; a non-zero status becomes
// RuntimeError with the library's message. The arguments, pointers among them, are values by now: reading the pointer of
// a tensor that has none (a vmap wrapper) throws, and must do so while the lock is held.
template <typename... P, typename... A>
void run(const Tensor &on, int (*f)(P...), A... a) {
    const lfm2q_stream_t st = stream(on);
    int status;
    {
        const Unlocked unlocked;
        status = f(a..., st);
    }
    if (status != LFM2Q_OK) fail(lfm2q_last_error());
}

// The GEMM workspace of t's device and current stream: the entry of lfm2opt._capi's table, made by its prepare_workspace
// when there is none.
PyObject *g_workspaces = nullptr, *g_prepare = nullptr;

Tensor workspace(const Tensor &t) {  // (held by the caller while it is in use)
    const lfm2q_stream_t st = stream(t);
    require(g_workspaces != nullptr, "lfm2q: the workspace table is not set");
    PyObject *key = Py_BuildValue("(iK)", (int)t.device().index(), (unsigned long long)(uintptr_t)st);
    if (!key) throw std::invalid_argument("");
    PyObject *w = PyDict_GetItemWithError(g_workspaces, key);
    Py_DECREF(key);
    if (!w && PyErr_Occurred()) throw std::invalid_argument("");
    if (w) return tensor(w, "workspace");
    PyObject *dev = PyUnicode_FromFormat("cuda:%d", (int)t.device().index());
    PyObject *made = dev ? PyObject_CallOneArg(g_prepare, dev) : nullptr;
    Py_XDECREF(dev);
    if (!made) throw std::invalid_argument("");
    const Tensor ws = tensor(made, "workspace");
    Py_DECREF(made);
    return ws;
}

typedef PyObject *const *Args;

// ------------------------------------------------------------------------------------------------ decode GEMVs
// (W, scale, x, y, rows)
void gemv(Args a) {
    const Tensor &x = bf16(a[2], "x"), &y = bf16(a[3], "y"), &W = tensor(a[0], "W");
    require(W.is_cuda() && W.is_contiguous() && W.dim() == 2, "W must be a contiguous CUDA matrix");
    const bool int8 = W.scalar_type() == at::kChar;
    require(int8 || W.scalar_type() == at::kBFloat16, "W must be bf16 or int8");
    const Tensor *scale = optional(a[1], "scale");
    require(!int8 || (scale && scale->scalar_type() == at::kFloat), "int8 W needs fp32 scale");
    const int64_t N = W.size(0), K = W.size(1), B = K ? x.numel() / K : 0;
    require(B >= 1 && x.numel() == B * K && y.numel() == B * N, "x [B, K], y [B, N]");
    if (scale) {
        typed(a[1], at::kFloat, "scale");
        require(scale->numel() == N, "scale must have N elements");
    }
    same_device(W, &x, &y, scale);
    const long rows = integer(a[4]);
    const float *s = ptr<float>(scale);
    if (int8)
        run(x, lfm2q_gemv_w8, ptr<int8_t>(W), s, ptr<lfm2q_bf16>(x), ptr<lfm2q_bf16>(y), B, N, K, rows);
    else
        run(x, lfm2q_gemv_bf16, ptr<lfm2q_bf16>(W), s, ptr<lfm2q_bf16>(x), ptr<lfm2q_bf16>(y), B, N, K, rows);
}

// the epilogue of an INT4 GEMV: 0, 1 or 2, as any number
long epilogue(PyObject *o) {
    if (!PyFloat_Check(o)) return integer(o);
    const double v = PyFloat_AS_DOUBLE(o);
    return v == 0.0 || v == 1.0 || v == 2.0 ? (long)v : -1;
}
// the group size of scales S [R, K / group], and the output width of x [B, K], y [B, N] under epilogue epi
int64_t w4_group(const Tensor &S, int64_t R, int64_t K) {
    require(S.dim() == 2 && S.size(0) == R && S.size(1) >= 1 && K % S.size(1) == 0, "S must be [N, K / group]");
    const int64_t group = K / S.size(1);
    require(group > 0 && group % 32 == 0, "group size must be a multiple of 32");  // (0: a weight without columns)
    return group;
}
void w4_run(int fmt, const Tensor &W, const Tensor &S, const Tensor *Z, const Tensor &x, const Tensor &y, int64_t R,
            int64_t K, int64_t group, long epi) {
    require(epi == 0 || epi == 1 || epi == 2, "epi 0 (none), 1 (swiglu) or 2 (residual)");
    const int64_t N = epi == 1 ? R / 2 : R, B = K ? x.numel() / K : 0;
    require((epi != 1 || R % 2 == 0) && B >= 1 && x.numel() == B * K && y.numel() == B * N, "x [B, K], y [B, N]");
    same_device(W, &S, Z, &x, &y);
    run(x, lfm2q_gemv_w4, fmt, W.data_ptr(), S.data_ptr(), ptr<int32_t>(Z), ptr<lfm2q_bf16>(x), ptr<lfm2q_bf16>(y), B, N, K,
        group, epi);
}
// (Wp, S, x, y, epi)
void gemv_w4(Args a) {
    const Tensor &x = bf16(a[2], "x"), &y = bf16(a[3], "y"), &W = tensor(a[0], "Wp"), &S = tensor(a[1], "S");
    require(W.is_cuda() && W.is_contiguous() && W.scalar_type() == at::kByte && W.dim() == 2,
            "Wp: contiguous uint8 [N, K/2]");
    require(S.is_cuda() && S.is_contiguous() && S.scalar_type() == at::kFloat, "S: contiguous fp32 [N, K/128]");
    const int64_t R = W.size(0), K = W.size(1) * 2;
    w4_run(0, W, S, nullptr, x, y, R, K, w4_group(S, R, K), epilogue(a[4]));
}
// (qweight, scales, qzeros, x, y, epi)
void gemv_w4z(Args a) {
    const Tensor &x = bf16(a[3], "x"), &y = bf16(a[4], "y"), &W = tensor(a[0], "qweight"), &S = tensor(a[1], "scales"),
                 &Z = tensor(a[2], "qzeros");
    require(W.is_cuda() && W.is_contiguous() && W.scalar_type() == at::kInt && W.dim() == 2,
            "qweight: contiguous int32 [N, K/8]");
    require(S.is_cuda() && S.is_contiguous() && S.scalar_type() == at::kHalf, "scales: contiguous fp16 [N, K/group]");
    const int64_t R = W.size(0), K = W.size(1) * 8, group = w4_group(S, R, K), G = K / group;
    require(Z.is_cuda() && Z.is_contiguous() && Z.scalar_type() == at::kInt && Z.dim() == 2 && Z.size(0) == R &&
                Z.size(1) == (G + 7) / 8,
            "qzeros: contiguous int32 [N, ceil(K/group/8)]");
    w4_run(1, W, S, &Z, x, y, R, K, group, epilogue(a[5]));
}
// (g, y)
void silu_mul(Args a) {
    const Tensor &g = bf16(a[0], "g"), &y = bf16(a[1], "y");
    const int64_t I2 = g.size(-1);
    require(I2 > 0, "g [B, 2I], y [B, I]");
    const int64_t B = g.numel() / I2;
    require(I2 % 2 == 0 && y.numel() == B * (I2 / 2), "g [B, 2I], y [B, I]");
    same_device(g, &y);
    run(g, lfm2q_silu_mul, ptr<lfm2q_bf16>(g), ptr<lfm2q_bf16>(y), B, I2 / 2);
}

// ------------------------------------------------------------------------------------------------ GEMMs
// w [N, K], sw [N], bias [N] or None, y [M, N]; returns N
int64_t common(PyObject *ow, PyObject *osw, PyObject *ob, PyObject *oy, int64_t M, int64_t K) {
    const Tensor &w = typed(ow, at::kChar, "w"), &sw = typed(osw, at::kFloat, "sw"), &y = bf16(oy, "y");
    require(w.dim() == 2 && w.size(1) == K, "w must be [N, K]");
    const int64_t N = w.size(0);
    require(K % 16 == 0, "need K % 16 == 0");
    require(sw.numel() == N && y.numel() == M * N, "sw / y shape");
    if (const Tensor *b = opt_bf16(ob, "bias")) require(b->numel() == N, "bias shape");
    return N;
}
// (xq, sx, w, sw, bias, y, gelu)
void gemm_i8(Args a) {
    const Tensor &xq = typed(a[0], at::kChar, "xq"), &sx = typed(a[1], at::kFloat, "sx");
    require(xq.dim() >= 1, "sx shape");
    const int64_t K = xq.size(-1), M = K ? xq.numel() / K : 0;
    const bool grouped = sx.dim() == 2;
    require(grouped ? K % 64 == 0 && sx.size(0) == K / 64 && sx.size(1) == M : sx.numel() == M, "sx shape");
    const int64_t N = common(a[2], a[3], a[4], a[5], M, K);
    const Tensor &w = tensor(a[2], "w"), &sw = tensor(a[3], "sw"), *b = optional(a[4], "bias"), &y = tensor(a[5], "y");
    same_device(xq, &sx, &w, &sw, b, &y);
    const int gelu = truth(a[6]);
    const int8_t *pq = ptr<int8_t>(xq), *pw = ptr<int8_t>(w);
    const float *ps = ptr<float>(sx), *psw = ptr<float>(sw);
    const lfm2q_bf16 *pb = ptr<lfm2q_bf16>(b);
    lfm2q_bf16 *py = ptr<lfm2q_bf16>(y);
    if (grouped) {
        run(xq, lfm2q_gemm_i8_grouped, pq, ps, pw, psw, pb, py, M, N, K, gelu);
    } else {  // per token: with the stream's workspace (the K split for shapes with fewer tiles than CUs)
        const Tensor ws = workspace(xq);
        run(xq, lfm2q_gemm_i8_ex, pq, ps, pw, psw, pb, py, M, N, K, gelu, ws.data_ptr(), (size_t)ws.numel());
    }
}
// (xq, sxT, w, sw, bias, yq, ysT, gelu)
void gemm_i8_q(Args a) {
    const Tensor &xq = typed(a[0], at::kChar, "xq"), &sxT = typed(a[1], at::kFloat, "sxT"), &w = typed(a[2], at::kChar, "w"),
                 &sw = typed(a[3], at::kFloat, "sw"), &yq = typed(a[5], at::kChar, "yq"),
                 &ysT = typed(a[6], at::kFloat, "ysT");
    require(xq.dim() >= 1, "sxT shape");
    const int64_t K = xq.size(-1), M = K ? xq.numel() / K : 0;
    require(w.dim() >= 1, "w [N, K] with N % 64 == 0");
    const int64_t N = w.size(0);
    require(sxT.dim() == 2 && K % 64 == 0 && sxT.size(0) == K / 64 && sxT.size(1) == M, "sxT shape");
    require(w.dim() == 2 && w.size(1) == K && N % 64 == 0 && sw.numel() == N, "w [N, K] with N % 64 == 0");
    require(yq.numel() == M * N && ysT.dim() == 2 && ysT.size(0) == N / 64 && ysT.size(1) == M, "yq / ysT shape");
    const Tensor *b = opt_bf16(a[4], "bias");
    if (b) require(b->numel() == N, "bias shape");
    same_device(xq, &sxT, &w, &sw, b, &yq, &ysT);
    const int gelu = truth(a[7]);
    run(xq, lfm2q_gemm_i8_q, ptr<int8_t>(xq), ptr<float>(sxT), ptr<int8_t>(w), ptr<float>(sw), ptr<lfm2q_bf16>(b),
        ptr<int8_t>(yq), ptr<float>(ysT), M, N, K, gelu);
}
// (x, w, sw, bias, y, gelu)
void gemm_w8(Args a) {
    const Tensor &x = bf16(a[0], "x");
    require(x.dim() >= 1, "w must be [N, K]");
    const int64_t K = x.size(-1), M = K ? x.numel() / K : 0, N = common(a[1], a[2], a[3], a[4], M, K);
    const Tensor &w = tensor(a[1], "w"), &sw = tensor(a[2], "sw"), *b = optional(a[3], "bias"), &y = tensor(a[4], "y");
    same_device(x, &w, &sw, b, &y);
    const int gelu = truth(a[5]);
    const lfm2q_bf16 *px = ptr<lfm2q_bf16>(x), *pb = ptr<lfm2q_bf16>(b);
    const int8_t *pw = ptr<int8_t>(w);
    const float *psw = ptr<float>(sw);
    lfm2q_bf16 *py = ptr<lfm2q_bf16>(y);
    const Tensor ws = workspace(x);  // the K split across workgroups for shapes with few tiles
    run(x, lfm2q_gemm_w8_ex, px, pw, psw, pb, py, M, N, K, gelu, ws.data_ptr(), (size_t)ws.numel());
}

// ------------------------------------------------------------------------------------------------ producers
// (x, q, s)
void quant_rows(Args a) {
    const Tensor &x = bf16(a[0], "x"), &q = typed(a[1], at::kChar, "q"), &s = typed(a[2], at::kFloat, "s");
    require(x.dim() >= 1, "K must be a multiple of 8");
    const int64_t K = x.size(-1), rows = K ? x.numel() / K : 0;
    if (s.dim() == 2) {
        require(K % 64 == 0 && K > 0 && s.size(0) == K / 64 && s.size(1) == rows && q.numel() == x.numel(),
                "grouped shapes");
        same_device(x, &q, &s);
        run(x, lfm2q_quant_groups, ptr<lfm2q_bf16>(x), ptr<int8_t>(q), ptr<float>(s), rows, K);
        return;
    }
    require(K % 8 == 0 && K != 0, "K must be a multiple of 8");
    require(q.numel() == x.numel() && s.numel() == rows, "q / s shape");
    same_device(x, &q, &s);
    run(x, lfm2q_quant_rows, ptr<lfm2q_bf16>(x), ptr<int8_t>(q), ptr<float>(s), rows, K);
}
// per row (1-D s) or per row and 64 columns (2-D s [L / 64, rows])
int check_qs(const Tensor &q, const Tensor &s, int64_t rows, int64_t L) {
    const bool grouped = s.dim() == 2;
    require(q.numel() == rows * L, "q shape");
    require(grouped ? s.size(0) == L / 64 && s.size(1) == rows && L % 64 == 0 : s.numel() == rows, "s shape");
    return grouped;
}
// (h, y, w, b, q, s, eps, x)
void add_layernorm_q(Args a) {
    const Tensor &h = bf16(a[0], "h"), &w = bf16(a[2], "w"), &b = bf16(a[3], "b"), *y = opt_bf16(a[1], "y");
    if (y) require(y->numel() == h.numel(), "y shape");
    const int64_t D = h.dim() ? h.size(-1) : 0, rows = D ? h.numel() / D : 0;
    require(D % 8 == 0 && 0 < D && D <= 8192 && w.numel() == D && b.numel() == D, "D must be a multiple of 8, <= 8192");
    const Tensor &q = typed(a[4], at::kChar, "q"), &s = typed(a[5], at::kFloat, "s");
    const int grouped = check_qs(q, s, rows, D);
    const Tensor *x = opt_bf16(a[7], "x");
    if (x) require(x->numel() == h.numel(), "x shape");
    same_device(h, y, &w, &b, &q, &s, x);
    const float eps = real(a[6]);
    run(h, lfm2q_add_layernorm_q, ptr<lfm2q_bf16>(h), ptr<lfm2q_bf16>(y), ptr<lfm2q_bf16>(w), ptr<lfm2q_bf16>(b),
        ptr<int8_t>(q), ptr<float>(s), ptr<lfm2q_bf16>(x), rows, D, eps, grouped);
}
// (h, y, w, q, s, eps, x)
void add_rmsnorm_q(Args a) {
    const Tensor &h = bf16(a[0], "h"), &w = bf16(a[2], "w"), *y = opt_bf16(a[1], "y");
    if (y) require(y->numel() == h.numel(), "y shape");
    const int64_t H = h.dim() ? h.size(-1) : 0, rows = H ? h.numel() / H : 0;
    require(w.numel() == H && H % 8 == 0 && 0 < H && H <= 8192, "w shape");
    const Tensor &q = typed(a[3], at::kChar, "q"), &s = typed(a[4], at::kFloat, "s");
    const int grouped = check_qs(q, s, rows, H);
    const Tensor *x = opt_bf16(a[6], "x");
    if (x) require(x->numel() == h.numel(), "x shape");
    same_device(h, y, &w, &q, &s, x);
    const float eps = real(a[5]);
    run(h, lfm2q_add_rmsnorm_q, ptr<lfm2q_bf16>(h), ptr<lfm2q_bf16>(y), ptr<lfm2q_bf16>(w), ptr<int8_t>(q), ptr<float>(s),
        ptr<lfm2q_bf16>(x), rows, H, eps, grouped);
}
// (g, q, s, x)
void silu_mul_q(Args a) {
    const Tensor &g = bf16(a[0], "g");
    const int64_t I = g.dim() ? g.size(-1) / 2 : 0, rows = I ? g.numel() / (2 * I) : 0;
    require(I % 8 == 0 && 0 < I && I <= 8192 && g.size(-1) == 2 * I, "I shape");
    const Tensor &q = typed(a[1], at::kChar, "q"), &s = typed(a[2], at::kFloat, "s");
    const int grouped = check_qs(q, s, rows, I);
    const Tensor *x = opt_bf16(a[3], "x");
    if (x) require(x->numel() == rows * I, "x shape");
    same_device(g, &q, &s, x);
    run(g, lfm2q_silu_mul_q, ptr<lfm2q_bf16>(g), ptr<int8_t>(q), ptr<float>(s), ptr<lfm2q_bf16>(x), rows, I, grouped);
}

// ------------------------------------------------------------------------------------------------ module
// set_workspaces(table {(device index, stream): tensor}, prepare(device) -> tensor)
void set_workspaces(Args a) {
    if (!PyDict_Check(a[0]) || !PyCallable_Check(a[1])) fail("set_workspaces: a dict and a callable");
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XSETREF(g_workspaces, a[0]);
    Py_XSETREF(g_prepare, a[1]);
}

// F with exactly N positional arguments; C++ exceptions become RuntimeError
template <void (*F)(Args), int N>
PyObject *entry(PyObject *, Args args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    try {
        F(args);
    } catch (const std::invalid_argument &) {  // the Python error is already set
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "invalid argument");
        return nullptr;
    } catch (const c10::Error &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown error");
        return nullptr;
    }
    Py_RETURN_NONE;
}
#define LFM2Q_ENTRY(F_, N_) {#F_, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(entry<F_, N_>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {LFM2Q_ENTRY(gemv, 5),          LFM2Q_ENTRY(gemv_w4, 5),       LFM2Q_ENTRY(gemv_w4z, 6),
                         LFM2Q_ENTRY(silu_mul, 2),      LFM2Q_ENTRY(gemm_i8, 7),       LFM2Q_ENTRY(gemm_i8_q, 8),
                         LFM2Q_ENTRY(gemm_w8, 6),       LFM2Q_ENTRY(quant_rows, 3),    LFM2Q_ENTRY(add_layernorm_q, 8),
                         LFM2Q_ENTRY(add_rmsnorm_q, 7), LFM2Q_ENTRY(silu_mul_q, 4),    LFM2Q_ENTRY(set_workspaces, 2),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lfm2q_native", "Eager ops of liblfm2q.", -1, methods,
                      nullptr,               nullptr,         nullptr,                  nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lfm2q_native(void) { return PyModule_Create(&module); }
