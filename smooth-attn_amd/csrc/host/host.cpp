// Native call path of the ordinary calls of the Python API.
//
// Every function here takes a call whose tensors the kernels can use as they
// are, allocates the results, launches through the C ABI
// (include/smooth_attn_amd.h) on torch's current stream and returns; for any
// other call (a wrong or unusual argument, a tensor that must be copied or
// padded first, a tensor subclass, a functorch transform, tracing, a dispatch
// or function mode, forward-mode gradients) it returns None and launches
// nothing, and the Python path of smooth_attn/kernels.py handles or refuses
// that call as it always did.
//
// Why: small calls are bound by the host.  Per pass, Python path -> this one,
// same kernels: causal normalisation forward [2,8,512,512] 9.2 -> 4.4 us,
// prefill [1,32/8,512,128] 18.0 -> 11.4, a decode step (append + attention) of
// 8 sequences 44 -> 22, training steps [2,16,1023,1023] normalisation 95 -> 48
// and [4,12,1024,64] attention 154 -> 89, each now bound by its kernels.  The
// autograd nodes are C++, so the backward needs no interpreter on the autograd
// thread.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>

#include "smooth_attn_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------
// The C ABI, bound once to the addresses of the loaded library.
// ---------------------------------------------------------------------------
struct Abi {
    decltype(&sa_status_string) status_string = nullptr;
    decltype(&sa_norm_fwd) norm_fwd = nullptr;
    decltype(&sa_norm_bwd) norm_bwd = nullptr;
    decltype(&sa_flash_fwd) flash_fwd = nullptr;
    decltype(&sa_flash_bwd_ws) flash_bwd_ws = nullptr;
    decltype(&sa_flash_bwd_workspace_size) flash_bwd_workspace_size = nullptr;
    decltype(&sa_paged_decode) paged_decode = nullptr;
    decltype(&sa_paged_decode_workspace_size) paged_decode_workspace_size = nullptr;
    decltype(&sa_paged_kv_append_lens) paged_kv_append_lens = nullptr;
} abi;

template <typename F>
bool bind_one(PyObject* table, const char* name, F& fn) {
    PyObject* v = PyDict_GetItemString(table, name);
    if (v == nullptr) {
        PyErr_Format(PyExc_KeyError, "no address for %s", name);
        return false;
    }
    fn = reinterpret_cast<F>(PyLong_AsVoidPtr(v));
    return !PyErr_Occurred();
}

// bind({name: address}): call once, before anything else.
PyObject* py_bind(PyObject*, PyObject* table) {
    if (!PyDict_Check(table)) {
        PyErr_SetString(PyExc_TypeError, "bind() takes a dict of addresses");
        return nullptr;
    }
    if (!bind_one(table, "sa_status_string", abi.status_string) || !bind_one(table, "sa_norm_fwd", abi.norm_fwd) ||
        !bind_one(table, "sa_norm_bwd", abi.norm_bwd) || !bind_one(table, "sa_flash_fwd", abi.flash_fwd) ||
        !bind_one(table, "sa_flash_bwd_ws", abi.flash_bwd_ws) ||
        !bind_one(table, "sa_flash_bwd_workspace_size", abi.flash_bwd_workspace_size) ||
        !bind_one(table, "sa_paged_decode", abi.paged_decode) ||
        !bind_one(table, "sa_paged_decode_workspace_size", abi.paged_decode_workspace_size) ||
        !bind_one(table, "sa_paged_kv_append_lens", abi.paged_kv_append_lens))
        return nullptr;
    Py_RETURN_NONE;
}

void check(int status, const char* what) {
    if (status != 0)
        throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(status) +
                                 "): " + abi.status_string(status));
}

// Lets other Python threads run while a call allocates and launches, which may
// wait: for a full queue, a first load of the kernel's code, an allocation that
// frees cached memory first.  Gives the interpreter back before an exception
// leaves its scope.
struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    NoGil() = default;
    NoGil(const NoGil&) = delete;
    NoGil& operator=(const NoGil&) = delete;
    ~NoGil() { PyEval_RestoreThread(state); }
};

// ---------------------------------------------------------------------------
// Which calls are ordinary.
// ---------------------------------------------------------------------------
// No interposer of any kind between this call and the device.
bool plain_mode() {
    return !torch::jit::tracer::isTracing() && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A dense tensor on a GPU, of exactly torch.Tensor or torch.nn.Parameter, and
// no wrapper or lazily conjugated / negated view.
const Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet wrappers(
        {c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
         c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::Fake,
         c10::DispatchKey::ZeroTensor, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
         c10::DispatchKey::Quantized});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
        t.key_set().has_any(wrappers) || t._fw_grad(0).defined())
        return nullptr;
    return &t;
}

int code_of(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return SA_F32;
        case at::kHalf: return SA_F16;
        case at::kBFloat16: return SA_BF16;
        case at::kFloat8_e4m3fn: return SA_FP8_E4M3FN;
        default: return -1;
    }
}
bool float_code(int c) { return c == SA_F32 || c == SA_F16 || c == SA_BF16; }

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// kernels.py's _flash_operand: (b, h, t) strides that are multiples of 16
// bytes, unit stride along D, a 16-byte aligned base, rows at most 16 MiB
// apart.
bool operand_ok(const Tensor& t) {
    const int64_t es = t.element_size(), a = 16 / es;
    const auto s = t.strides();
    if (s.back() != 1 || !aligned16(t) || s[s.size() - 2] * es > (int64_t(1) << 24)) return false;
    for (size_t i = 0; i + 1 < s.size(); ++i)
        if (s[i] % a != 0) return false;
    return true;
}

sa_stream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
const int64_t* strides(const Tensor& t) { return t.strides().data(); }

bool as_double(PyObject* o, double& v) {
    v = PyFloat_Check(o) ? PyFloat_AS_DOUBLE(o) : PyLong_CheckExact(o) ? PyLong_AsDouble(o) : NAN;
    if (PyErr_Occurred()) PyErr_Clear();
    return std::isfinite(v);
}
// A non-negative int (not a bool or an int-like object) below 2^31.
bool as_int(PyObject* o, int& v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long x = PyLong_AsLongAndOverflow(o, &over);
    if (over != 0 || x < 0 || x > INT32_MAX) return false;
    v = static_cast<int>(x);
    return true;
}

// ---------------------------------------------------------------------------
// Normalisation.
// ---------------------------------------------------------------------------
constexpr int64_t kMaxCols = 8192;  // kernels.py MAX_ROW_COLS

struct Family {
    double alpha, theta;
    int power;
    bool parse(PyObject* a, PyObject* t, PyObject* p) {
        return as_double(a, alpha) && as_double(t, theta) && as_int(p, power) && power >= 1 && power <= 3;
    }
};

// Rows of contiguous x into contiguous y.
void norm_fwd(const Tensor& x, const Tensor& y, bool causal, const Family& f) {
    const int64_t cols = x.size(-1);
    const c10::DeviceGuard guard(x.device());
    check(abi.norm_fwd(x.data_ptr(), y.data_ptr(), x.numel() / cols, cols, cols, cols, code_of(x.scalar_type()), causal,
                       static_cast<float>(f.alpha), static_cast<float>(f.theta), f.power, stream_of(x)),
          "sa_norm_fwd");
}

bool norm_input_ok(const Tensor& x, bool causal) {
    return float_code(code_of(x.scalar_type())) && (causal ? x.dim() >= 2 : x.dim() == 2) && x.numel() > 0 &&
           x.is_contiguous() && x.size(-1) <= kMaxCols && (!causal || x.size(-1) == x.size(-2));
}

// norm_out(out, x, causal, alpha, theta, power) -> bool: whether it ran.
PyObject* py_norm_out(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Family f;
    const Tensor *out, *x;
    if (n != 6 || !plain_mode() || !(out = plain(a[0])) || !(x = plain(a[1])) || !f.parse(a[3], a[4], a[5]))
        Py_RETURN_FALSE;
    const bool causal = a[2] == Py_True;
    if (!norm_input_ok(*x, causal) || out->scalar_type() != x->scalar_type() || out->device() != x->device() ||
        out->sizes() != x->sizes() || !out->is_contiguous())
        Py_RETURN_FALSE;
    {
        const NoGil released;
        norm_fwd(*x, *out, causal, f);
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

struct CausalNorm : public torch::autograd::Function<CausalNorm> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, double alpha, double theta, int64_t power) {
        const Family f{alpha, theta, static_cast<int>(power)};
        Tensor y = at::empty_like(x);
        norm_fwd(x, y, true, f);
        ctx->save_for_backward({x});
        ctx->saved_data["alpha"] = alpha;
        ctx->saved_data["theta"] = theta;
        ctx->saved_data["power"] = power;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        if (!ctx->needs_input_grad(0)) return {Tensor(), Tensor(), Tensor(), Tensor()};
        const Tensor saved = ctx->get_saved_variables()[0];
        Tensor g = grads[0];
        TORCH_CHECK_VALUE(g.is_cuda() && g.device() == saved.device(),
                          "grad_output must live on the same CUDA device as x");
        TORCH_CHECK_VALUE(float_code(code_of(saved.scalar_type())) && saved.sizes() == g.sizes(),
                          "the saved x must have grad_output's shape and a dtype of the fused kernels");
        const int64_t cols = saved.size(-1);
        // (unpack hooks may hand back another layout or type than forward saved)
        const bool as_saved = saved.is_contiguous();
        Tensor x = as_saved ? saved : saved.reshape({-1, cols});
        if (!as_saved && (x.stride(1) != 1 || x.stride(0) < cols)) x = x.contiguous();
        if (g.scalar_type() != at::kFloat && g.scalar_type() != x.scalar_type()) g = g.to(at::kFloat);
        g = g.contiguous();
        Tensor dx = at::empty_like(x);
        const c10::DeviceGuard guard(x.device());
        check(abi.norm_bwd(x.data_ptr(), g.data_ptr(), dx.data_ptr(), x.numel() / cols, cols, x.stride(-2), cols,
                           dx.stride(-2),
                           code_of(x.scalar_type()), code_of(g.scalar_type()), 1,
                           static_cast<float>(ctx->saved_data["alpha"].toDouble()),
                           static_cast<float>(ctx->saved_data["theta"].toDouble()),
                           static_cast<int>(ctx->saved_data["power"].toInt()), stream_of(x)),
              "sa_norm_bwd");
        return {as_saved ? dx : dx.view(saved.sizes()), Tensor(), Tensor(), Tensor()};
    }
};

// causal_norm(x, alpha, theta, power) -> y or None.
PyObject* py_causal_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Family f;
    const Tensor* x;
    if (n != 4 || !plain_mode() || !(x = plain(a[0])) || !f.parse(a[1], a[2], a[3]) || !norm_input_ok(*x, true))
        Py_RETURN_NONE;
    Tensor y;
    {
        const NoGil released;
        if (at::GradMode::is_enabled() && x->requires_grad()) {
            y = CausalNorm::apply(*x, f.alpha, f.theta, static_cast<int64_t>(f.power));
        } else {
            y = at::empty_like(*x);
            norm_fwd(*x, y, true, f);
        }
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------
// Fused attention.
// ---------------------------------------------------------------------------
struct FlashCall {
    double scale;
    int window;
    bool exact;
};

// Whether the kernels take q, k and v as they are (kernels.py's checks).
bool flash_ok(const Tensor& q, const Tensor& k, const Tensor& v) {
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || q.numel() == 0 || k.numel() == 0) return false;
    const int code = code_of(q.scalar_type());
    if (!float_code(code) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
    if (k.device() != q.device() || v.device() != q.device()) return false;
    const int64_t D = q.size(3), Hkv = k.size(1);
    if (k.size(0) != q.size(0) || k.size(2) != q.size(2) || k.size(3) != D || v.sizes() != k.sizes() ||
        q.size(1) % Hkv != 0)
        return false;
    if (D > 512 || D % (code == SA_F32 ? 4 : 8) != 0 || q.size(0) > INT32_MAX || q.size(1) > INT32_MAX ||
        q.size(2) > INT32_MAX)
        return false;
    return operand_ok(q) && operand_ok(k) && operand_ok(v);
}

int dim(const Tensor& t, int i) { return static_cast<int>(t.size(i)); }

void flash_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const FlashCall& c, Tensor& o, Tensor& row_sums) {
    o = at::empty_like(q);
    if (o.stride(-1) != 1) o = at::empty(q.sizes(), q.options());
    row_sums = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
    const c10::DeviceGuard guard(q.device());
    check(abi.flash_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), row_sums.data_ptr<float>(), dim(q, 0),
                        dim(q, 1), dim(k, 1), dim(q, 2), dim(q, 3), strides(q), strides(k), strides(v), strides(o),
                        static_cast<float>(c.scale), c.window, c.exact, code_of(q.scalar_type()), stream_of(q)),
          "sa_flash_fwd");
}

// What backward reads: q, k, v, o and the row sums as forward saved them, or
// as unpack hooks hand them back.
void check_saved(const variable_list& saved, const Tensor& grad) {
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &row_sums = saved[4];
    for (const Tensor* t : {&q, &k, &v, &o, &row_sums, &grad})
        TORCH_CHECK_VALUE(t->is_cuda() && t->device() == q.device(),
                          "attention tensors must live on the same CUDA device as q");
    TORCH_CHECK_VALUE(float_code(code_of(q.scalar_type())) && k.scalar_type() == q.scalar_type() &&
                          v.scalar_type() == q.scalar_type(),
                      "fused attention expects bf16, fp16 or fp32 q/k/v of one dtype, got ", q.scalar_type(), "/",
                      k.scalar_type(), "/", v.scalar_type());
    TORCH_CHECK_VALUE(o.scalar_type() == q.scalar_type() && row_sums.scalar_type() == at::kFloat,
                      "the saved output must have q's dtype and the saved row sums fp32");
    TORCH_CHECK_VALUE(q.sizes() == grad.sizes() && o.sizes() == grad.sizes() && k.dim() == 4 && v.sizes() == k.sizes() &&
                          k.size(0) == q.size(0) && k.size(1) > 0 && q.size(1) % k.size(1) == 0 &&
                          k.size(2) == q.size(2) && k.size(3) == q.size(3) &&
                          row_sums.sizes() == q.sizes().slice(0, 3),
                      "the saved attention tensors must have the shapes that forward saved");
}

struct Flash : public torch::autograd::Function<Flash> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, double scale,
                          int64_t window, bool exact) {
        Tensor o, row_sums;
        flash_fwd(q, k, v, FlashCall{scale, static_cast<int>(window), exact}, o, row_sums);
        ctx->save_for_backward({q, k, v, o, row_sums});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["window"] = window;
        ctx->saved_data["exact"] = exact;
        return o;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list saved = ctx->get_saved_variables();
        check_saved(saved, grads[0]);
        // (unpack hooks may hand back tensors of another layout, or of a type that takes fewer head dims)
        const int64_t D0 = saved[0].size(3), step = saved[0].scalar_type() == at::kFloat ? 4 : 8;
        const int64_t pad = (step - D0 % step) % step;
        const auto fix = [pad](const Tensor& t) {
            if (pad != 0) return at::constant_pad_nd(t, {0, pad});
            return operand_ok(t) ? t : t.clone(at::MemoryFormat::Contiguous);
        };
        const Tensor q = fix(saved[0]), k = fix(saved[1]), v = fix(saved[2]), o = fix(saved[3]);
        const Tensor row_sums = saved[4].contiguous();
        const Tensor g = fix(grads[0].to(q.scalar_type()));
        const double scale = ctx->saved_data["scale"].toDouble();
        const int window = static_cast<int>(ctx->saved_data["window"].toInt());
        const bool exact = ctx->saved_data["exact"].toBool();
        const int B = dim(q, 0), Hq = dim(q, 1), Hkv = dim(k, 1), T = dim(q, 2), D = dim(q, 3);
        const int code = code_of(q.scalar_type());
        Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
        Tensor delta = at::empty({B, Hq, T}, q.options().dtype(at::kFloat));
        // fp32 partials of the dK/dV blocks split over their query tiles, when the library splits them
        const int64_t ws_bytes = std::max<int64_t>(abi.flash_bwd_workspace_size(B, Hq, Hkv, T, D, window, code), 0);
        Tensor ws;
        if (ws_bytes > 0) ws = at::empty({ws_bytes / 4}, delta.options());
        const c10::DeviceGuard guard(q.device());
        check(abi.flash_bwd_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), g.data_ptr(),
                               row_sums.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                               delta.data_ptr<float>(), B, Hq, Hkv, T, D, strides(q), strides(k), strides(v),
                               strides(o), strides(g), strides(dq), strides(dk), strides(dv),
                               static_cast<float>(scale), window, exact, code,
                               ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, stream_of(q)),
              "sa_flash_bwd_ws");
        for (Tensor* t : {&dq, &dk, &dv})
            if (pad != 0) *t = t->narrow(3, 0, D0).contiguous();
        return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
    }
};

// flash(q, k, v, scale or None, window, exact) -> o or None.
PyObject* py_flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const Tensor *q, *k, *v;
    FlashCall c;
    if (n != 6 || !plain_mode() || !(q = plain(a[0])) || !(k = plain(a[1])) || !(v = plain(a[2])) ||
        !flash_ok(*q, *k, *v) || !as_int(a[4], c.window) || !PyBool_Check(a[5]))
        Py_RETURN_NONE;
    if (a[3] == Py_None)
        c.scale = 1.0 / std::sqrt(static_cast<double>(q->size(3)));
    else if (!as_double(a[3], c.scale))
        Py_RETURN_NONE;
    c.exact = a[5] == Py_True;
    Tensor o;
    {
        const NoGil released;
        if (at::GradMode::is_enabled() && (q->requires_grad() || k->requires_grad() || v->requires_grad())) {
            o = Flash::apply(*q, *k, *v, c.scale, static_cast<int64_t>(c.window), c.exact);
        } else {
            Tensor row_sums;
            flash_fwd(*q, *k, *v, c, o, row_sums);
        }
    }
    return THPVariable_Wrap(o);
    END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------
// Paged decode and append.
// ---------------------------------------------------------------------------
// Caches [n_pages, Hkv, block_size, D], an int32 table and int32 lengths of
// at least B sequences, all on q's device and in the layout the kernels take.
bool paging_ok(const Tensor& like, int64_t B, int64_t Hkv, int64_t D, int block_size, const Tensor& k, const Tensor& v,
               const Tensor& table, const Tensor& lens) {
    for (const Tensor* t : {&k, &v, &table, &lens})
        if (t->device() != like.device()) return false;
    return k.dim() == 4 && v.sizes() == k.sizes() && v.scalar_type() == k.scalar_type() && k.numel() > 0 &&
           k.size(1) == Hkv && k.size(2) == block_size && k.size(3) == D && block_size > 0 &&
           (block_size & (block_size - 1)) == 0 && k.size(0) <= INT32_MAX && operand_ok(k) && operand_ok(v) &&
           table.scalar_type() == at::kInt && table.dim() == 2 && table.size(0) >= B && table.stride(1) == 1 &&
           table.size(1) <= INT32_MAX && lens.scalar_type() == at::kInt && lens.is_contiguous() && lens.numel() >= B;
}

// paged(q, k_cache, v_cache, block_table, context_lens, scale or None, block_size) -> out or None.
PyObject* py_paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const Tensor *q, *k, *v, *table, *lens;
    int block_size;
    if (n != 7 || !plain_mode() || !(q = plain(a[0])) || !(k = plain(a[1])) || !(v = plain(a[2])) ||
        !(table = plain(a[3])) || !(lens = plain(a[4])) || !as_int(a[6], block_size))
        Py_RETURN_NONE;
    if (q->dim() != 4 || q->size(2) != 1 || q->numel() == 0 || k->dim() != 4) Py_RETURN_NONE;
    const int64_t B = q->size(0), Hq = q->size(1), D = q->size(3), Hkv = k->size(1);
    const int qc = code_of(q->scalar_type()), kc = code_of(k->scalar_type());
    // one type for all, or bf16 q over e4m3fn caches (other pairs convert q first)
    const bool mixed = qc == SA_BF16 && kc == SA_FP8_E4M3FN;
    if (!(mixed || (qc == kc && float_code(qc))) || Hkv == 0 || Hq % Hkv != 0 || D % (mixed ? 16 : 8) != 0 || D > 512 ||
        B > INT32_MAX || Hq > INT32_MAX || !operand_ok(*q) ||
        !paging_ok(*q, B, Hkv, D, block_size, *k, *v, *table, *lens))
        Py_RETURN_NONE;
    double scale;
    if (a[5] == Py_None)
        scale = 1.0 / std::sqrt(static_cast<double>(D));
    else if (!as_double(a[5], scale))
        Py_RETURN_NONE;
    Tensor out;
    {
        const NoGil released;
        out = at::empty({B, Hq, D}, q->options().dtype(at::kBFloat16).requires_grad(false));
        const int b = static_cast<int>(B), hq = static_cast<int>(Hq), d = static_cast<int>(D);
        const int max_pages = static_cast<int>(table->size(1));
        const int64_t ws_bytes = abi.paged_decode_workspace_size(b, hq, d, max_pages, block_size);
        Tensor ws = at::empty({std::max<int64_t>(1, (ws_bytes + 3) / 4)}, out.options().dtype(at::kFloat));
        const c10::DeviceGuard guard(q->device());
        check(abi.paged_decode(q->data_ptr(), k->data_ptr(), v->data_ptr(), out.data_ptr(), table->data_ptr<int32_t>(),
                               lens->data_ptr<int32_t>(), b, hq, static_cast<int>(Hkv), d, block_size, max_pages,
                               static_cast<int>(k->size(0)), strides(*q), strides(*k), strides(*v), strides(out),
                               table->stride(0), static_cast<float>(scale), mixed ? SA_PAGED_DTYPES(qc, kc) : qc,
                               ws.data_ptr<float>(), ws.numel() * 4, stream_of(*q)),
              "sa_paged_decode");
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// paged_append(k_cache, v_cache, k_new, v_new, block_table, context_lens, block_size) -> new lengths or None.
PyObject* py_paged_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const Tensor *k, *v, *kn, *vn, *table, *lens;
    int block_size;
    if (n != 7 || !plain_mode() || !(k = plain(a[0])) || !(v = plain(a[1])) || !(kn = plain(a[2])) ||
        !(vn = plain(a[3])) || !(table = plain(a[4])) || !(lens = plain(a[5])) || !as_int(a[6], block_size))
        Py_RETURN_NONE;
    const int code = code_of(k->scalar_type());
    if (code < 0 || kn->dim() != 4 || kn->numel() == 0 || vn->sizes() != kn->sizes() ||
        kn->scalar_type() != k->scalar_type() || vn->scalar_type() != k->scalar_type() ||
        kn->device() != k->device() || vn->device() != k->device())
        Py_RETURN_NONE;
    const int64_t B = kn->size(0), Hkv = kn->size(1), n_new = kn->size(2), D = kn->size(3);
    if (!paging_ok(*k, B, Hkv, D, block_size, *k, *v, *table, *lens) || D % (16 / k->element_size()) != 0 ||
        !operand_ok(*kn) || !operand_ok(*vn) || kn->strides() != vn->strides() || B > INT32_MAX || n_new > INT32_MAX)
        Py_RETURN_NONE;
    Tensor out;
    {
        const NoGil released;
        const c10::DeviceGuard guard(k->device());
        out = at::empty(lens->sizes(), lens->options());
        check(abi.paged_kv_append_lens(kn->data_ptr(), vn->data_ptr(), k->data_ptr(), v->data_ptr(),
                                       table->data_ptr<int32_t>(), lens->data_ptr<int32_t>(), out.data_ptr<int32_t>(),
                                       lens->numel(), static_cast<int>(B), static_cast<int>(Hkv),
                                       static_cast<int>(n_new), static_cast<int>(D), block_size,
                                       static_cast<int>(table->size(1)), static_cast<int>(k->size(0)), strides(*kn),
                                       strides(*k), strides(*v), table->stride(0), code, stream_of(*k)),
              "sa_paged_kv_append_lens");
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

template <typename F>
PyCFunction fast(F f) {
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_O, "bind({name: address of a C ABI function})"},
    {"norm_out", fast(py_norm_out), METH_FASTCALL, "norm_out(out, x, causal, alpha, theta, power) -> bool"},
    {"causal_norm", fast(py_causal_norm), METH_FASTCALL, "causal_norm(x, alpha, theta, power) -> y or None"},
    {"flash", fast(py_flash), METH_FASTCALL, "flash(q, k, v, scale, window, exact) -> o or None"},
    {"paged", fast(py_paged), METH_FASTCALL,
     "paged(q, k_cache, v_cache, block_table, context_lens, scale, block_size) -> out or None"},
    {"paged_append", fast(py_paged_append), METH_FASTCALL,
     "paged_append(k_cache, v_cache, k_new, v_new, block_table, context_lens, block_size) -> lens or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native call path (see csrc/host/host.cpp).", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    // (the tensors' layout in memory is that torch's)
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
