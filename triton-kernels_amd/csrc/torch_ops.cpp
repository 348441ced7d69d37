// The operators' common calls without Python in between: a call whose tensors are what they nearly always are is checked,
// given its outputs and launched here, and every other call gets None back and takes the Python launcher of the same
// operator (triton_kernels/kernels), which accepts, converts or refuses it as before. The kernels and the library's
// entry points are the same on both ways.
//
// What bounds such calls is the host: the q/k norm module at 256 tokens is 3 us of the GPU and took 25 us of Python and
// ctypes a call. A training step of the norm was worse off than its parts: its forward takes Python 17 us and
// its backward 20, but the autograd engine runs the backward on a thread of its own, and an interpreter that two cores take
// turns with runs at half its speed (41 and 43 us, 129 for a step whose kernels take 30). A node of the
// engine's own kind leaves the interpreter on one core. us a call, before -> now: q/k norm module at 256 tokens 25.5 -> 10.3,
// training step of the norm at [4, 24, 1024, 128] 107 to 129 -> 57, rotation of short sequences 18.7 -> 6.9, linear at 512 x 3072
// x 3072 15.8 -> 15.1 (the GPU's own time).
#include <torch/csrc/python_headers.h>
#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <string>

#include "../../include/flux_hip.h"

namespace {

using at::Tensor;

constexpr int64_t kMaxRow = 65536;   // values of a normalised row

// Tracing, function transforms, dispatch and function modes and forward-mode derivatives see the operators of the
// Python launchers; a call under any of them is theirs.
bool quiet() {
    return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() &&
           !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing() &&
           torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr;
}

// A strided tensor with memory of its own on a GPU and nothing on top (no subclass, lazy bit or wrapper), at least one value.
bool plain(const Tensor& t) {
    constexpr c10::DispatchKeySet usual({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA, c10::DispatchKey::ADInplaceOrView});
    return t.defined() && (t.key_set().raw_repr() & ~usual.raw_repr()) == 0 && t.is_cuda() && t.has_storage() && t.numel() > 0;
}

// The tensor behind a Python object, or null for anything but a torch.Tensor or Parameter itself.
const Tensor* tensor_of(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    return plain(t) ? &t : nullptr;
}

int type_code(const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 ? FLUX_BF16 : t.scalar_type() == at::kFloat ? FLUX_F32 : -1;
}
bool same_kind(const Tensor& a, const Tensor& b) { return a.scalar_type() == b.scalar_type() && a.device() == b.device(); }

// The number that float() makes of a Python object; false where that is more than a number's own conversion (a text, or
// nothing that float() takes), which is left to the launchers.
bool number(PyObject* o, double& value) {
    value = PyFloat_AsDouble(o);
    if (value != -1.0 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Lets other Python threads run while outputs are allocated and kernels launched (a launch waits where the queue is full).
struct WithoutInterpreter {
    PyThreadState* const state = PyEval_SaveThread();
    WithoutInterpreter() = default;
    WithoutInterpreter(const WithoutInterpreter&) = delete;
    ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const Tensor& beside) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(beside.device()));
}

// Raises what the library answered, as the kind of error that the Python launchers make of it (_native.check).
void check(int rc, const char* what) {
    if (rc == FLUX_OK) return;
    const char* const last = flux_last_error();
    const std::string msg = last && *last ? last : what;
    TORCH_CHECK_TYPE(rc != FLUX_E_DTYPE, msg);
    TORCH_CHECK_VALUE(rc != FLUX_E_SHAPE && rc != FLUX_E_NULL && rc != FLUX_E_ALIGN, msg);
    TORCH_CHECK_NOT_IMPLEMENTED(rc != FLUX_E_UNSUPPORTED, msg);
    TORCH_CHECK(rc != FLUX_E_TOO_WIDE, msg);
    TORCH_CHECK(false, msg, " (hipError ", rc, ")");
}

// Rows of 16-byte vectors from the first one on.
bool vector_rows(const Tensor& t) {
    const int64_t per16 = 16 / t.element_size();
    if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0 || t.size(-1) % per16 != 0) return false;
    for (int64_t i = 0; i + 1 < t.dim(); ++i)
        if (t.stride(i) % per16 != 0) return false;
    return true;
}

// ---- RMS norm ----------------------------------------------------------------------------------

bool norm_args_ok(const Tensor& x, const Tensor& scale) {
    const int xc = type_code(x), sc = type_code(scale);
    return xc >= 0 && sc >= 0 && (sc == xc || xc == FLUX_BF16) && x.device() == scale.device() && x.dim() >= 1 && x.dim() <= 4 &&
           x.stride(-1) == 1 && x.size(-1) <= kMaxRow && x.numel() / x.size(-1) <= 0x7fffffff && scale.dim() == 1 && scale.numel() == x.size(-1) && scale.stride(0) == 1;
}

flux_rms_norm_args norm_args(const Tensor& x, const Tensor& scale, const Tensor& y, const Tensor* rstd) {
    flux_rms_norm_args a = {x.data_ptr(), scale.data_ptr(), y.data_ptr(), rstd ? static_cast<float*>(rstd->data_ptr()) : nullptr, 1, 1, 1, 0, 0, 0};
    int64_t* const size[3] = {&a.d0, &a.d1, &a.d2};
    int64_t* const stride[3] = {&a.s0, &a.s1, &a.s2};
    const int64_t lead = x.dim() - 1;
    for (int64_t i = 0; i < lead; ++i) {
        *size[3 - lead + i] = x.size(i);
        *stride[3 - lead + i] = x.stride(i);
    }
    return a;
}

void launch_norm(const Tensor& x, const Tensor& scale, const Tensor& y, const Tensor* rstd, double eps) {
    const c10::DeviceGuard guard(x.device());
    const flux_rms_norm_args a = norm_args(x, scale, y, rstd);
    check(flux_rms_norm(a.x, a.scale, a.y, a.rstd, a.d0, a.d1, a.d2, static_cast<int32_t>(x.size(-1)), a.s0, a.s1, a.s2, type_code(x), type_code(scale),
                        static_cast<float>(eps), stream_of(x)), "flux_rms_norm");
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x_in, const Tensor& scale, double eps) {
        const Tensor x = x_in.contiguous();
        const int64_t n = x.size(-1);
        const Tensor y = empty(x.sizes(), x.scalar_type(), x), rstd = empty({x.numel() / n}, at::kFloat, x);
        launch_norm(x, scale, y, &rstd, eps);
        ctx->save_for_backward({x.reshape({-1, n}), scale, rstd});
        return y;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();   // (what saved-tensor hooks gave back, of any type)
        const Tensor x = saved[0].contiguous(), r = saved[2].to(at::kFloat).contiguous();
        Tensor s = saved[1].contiguous();
        const Tensor& dy = grads[0];
        for (const Tensor* t : std::initializer_list<const Tensor*>{&dy, &s, &r})
            TORCH_CHECK(t->is_cuda() && t->device() == x.device(), "tensors on different devices: ", t->device(), " and ", x.device());
        TORCH_CHECK(x.dim() == 2 && s.numel() == x.size(1) && r.numel() == x.size(0), "rms_norm: saved tensors came back with other sizes");
        const int xc = type_code(x);
        TORCH_CHECK_TYPE(xc >= 0, "unsupported dtype ", x.scalar_type(), ": the HIP kernels take bfloat16 or float32");
        const at::ScalarType scale_type = s.scalar_type();
        if (scale_type != x.scalar_type() && !(xc == FLUX_BF16 && scale_type == at::kFloat)) s = s.to(x.scalar_type());
        const int64_t rows = x.size(0), n = x.size(1);
        Tensor dy2 = dy.contiguous().reshape({rows, n});
        if (dy2.scalar_type() != x.scalar_type()) dy2 = dy2.to(x.scalar_type());
        const void* const dy_at = dy2.data_ptr();   // (a wrapper without memory ends here)
        const c10::DeviceGuard guard(x.device());
        // the kernel's types; the gradient of a scale of another type is converted from fp32
        const Tensor dx = empty(x.sizes(), x.scalar_type(), x), dscale = empty(s.sizes(), scale_type == at::kBFloat16 ? at::kBFloat16 : at::kFloat, x);
        const int64_t ws_bytes = flux_rms_norm_bwd_workspace_bytes(rows, static_cast<int32_t>(n), xc);
        const Tensor ws = empty({ws_bytes}, at::kByte, x);
        check(flux_rms_norm_bwd_ws(dy_at, x.data_ptr(), s.data_ptr(), static_cast<const float*>(r.data_ptr()), dx.data_ptr(), dscale.data_ptr(), type_code(dscale),
                                   ws.data_ptr(), ws_bytes, rows, static_cast<int32_t>(n), xc, type_code(s), stream_of(x)), "flux_rms_norm_bwd");
        return {dx.reshape(dy.sizes()), dscale.scalar_type() == scale_type ? dscale : dscale.to(scale_type), Tensor()};
    }
};

// rms_norm(x, scale, eps)
PyObject* py_rms_norm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 3, "rms_norm takes 3 arguments");
    const Tensor *x = tensor_of(args[0]), *scale = tensor_of(args[1]);
    if (!x || !scale || !quiet() || !norm_args_ok(*x, *scale)) Py_RETURN_NONE;
    double eps;
    if (!number(args[2], eps)) Py_RETURN_NONE;
    const bool differentiable = x->requires_grad() || scale->requires_grad(), recorded = differentiable && at::GradMode::is_enabled();
    if (differentiable && !recorded && !vector_rows(*x)) Py_RETURN_NONE;   // (copied first)
    Tensor y;
    {
        const Tensor x_kept = *x, scale_kept = *scale;   // (the caller's objects are another thread's to drop from here on)
        const WithoutInterpreter free;
        if (recorded) {
            y = RmsNorm::apply(x_kept, scale_kept, eps);
        } else {
            y = empty(x_kept.sizes(), x_kept.scalar_type(), x_kept);
            launch_norm(x_kept, scale_kept, y, nullptr, eps);
        }
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

PyObject* two(const Tensor& a, const Tensor& b) {
    PyObject* const t = PyTuple_New(2);
    if (!t) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
    return t;
}

// rms_norm_pair(x0, scale0, x1, scale1, eps): both in one launch, where nothing is differentiated
PyObject* py_rms_norm_pair(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 5, "rms_norm_pair takes 5 arguments");
    const Tensor *x0 = tensor_of(args[0]), *s0 = tensor_of(args[1]), *x1 = tensor_of(args[2]), *s1 = tensor_of(args[3]);
    if (!x0 || !s0 || !x1 || !s1 || at::GradMode::is_enabled() || !quiet() || !norm_args_ok(*x0, *s0) || !norm_args_ok(*x1, *s1) ||
        !same_kind(*x0, *x1) || !same_kind(*s0, *s1) || x0->size(-1) != x1->size(-1) || !vector_rows(*x0) || !vector_rows(*x1))
        Py_RETURN_NONE;
    double eps;
    if (!number(args[4], eps)) Py_RETURN_NONE;
    Tensor y0, y1;
    {
        const Tensor xa = *x0, xb = *x1, sa = *s0, sb = *s1;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(xa.device());
        y0 = empty(xa.sizes(), xa.scalar_type(), xa);
        y1 = empty(xb.sizes(), xb.scalar_type(), xb);
        const flux_rms_norm_args a0 = norm_args(xa, sa, y0, nullptr), a1 = norm_args(xb, sb, y1, nullptr);
        check(flux_rms_norm_pair(&a0, &a1, static_cast<int32_t>(xa.size(-1)), type_code(xa), type_code(sa), static_cast<float>(eps), stream_of(xa)), "flux_rms_norm_pair");
    }
    return two(y0, y1);
    END_HANDLE_TH_ERRORS
}

// ---- layer norm + modulation -------------------------------------------------------------------

// layer_norm_modulation(x, scale, shift, eps)
PyObject* py_layer_norm_modulation(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4, "layer_norm_modulation takes 4 arguments");
    const Tensor *x = tensor_of(args[0]), *scale = tensor_of(args[1]), *shift = tensor_of(args[2]);
    if (!x || !scale || !shift || !quiet() || x->dim() < 2 || type_code(*x) < 0 || !same_kind(*x, *scale) || !same_kind(*x, *shift) || !x->is_contiguous()) Py_RETURN_NONE;
    const int64_t batch = x->size(0), n = x->size(-1), rows = x->numel() / n;
    auto modulates = [&](const Tensor& m) {
        return m.dim() >= 2 && m.size(0) == batch && m.size(-1) == n && m.numel() == batch * n && m.stride(-1) == 1 && (batch == 1 || (m.stride(0) == scale->stride(0) && m.stride(0) >= n));
    };
    if (n > kMaxRow || !modulates(*scale) || !modulates(*shift)) Py_RETURN_NONE;
    double eps;
    if (!number(args[3], eps)) Py_RETURN_NONE;
    Tensor y;
    int rc;
    {
        const Tensor xa = *x, sc = *scale, sh = *shift;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(xa.device());
        y = at::empty_like(xa);
        rc = flux_layer_norm_modulation(xa.data_ptr(), sc.data_ptr(), sh.data_ptr(), y.data_ptr(), batch, rows / batch, static_cast<int32_t>(n),
                                        batch > 1 ? sc.stride(0) : n, type_code(xa), static_cast<float>(eps), stream_of(xa));
    }
    if (rc < 0) Py_RETURN_NONE;   // (a refusal: its kind of error is the launcher's)
    check(rc, "flux_layer_norm_modulation");
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// ---- rotation ----------------------------------------------------------------------------------

flux_src4 source(const Tensor& t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// apply_rope(q, k, table)
PyObject* py_apply_rope(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 3, "apply_rope takes 3 arguments");
    const Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *pe = tensor_of(args[2]);
    if (!q || !k || !pe || !quiet() || q->dim() != 4 || q->sizes() != k->sizes() || type_code(*q) < 0 || !same_kind(*q, *k) || q->device() != pe->device() ||
        q->stride(3) != 1 || k->stride(3) != 1 || !vector_rows(*q) || !vector_rows(*k))
        Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), L = q->size(2), D = q->size(3), lead = pe->dim() - 4;
    if (D % 2 != 0 || pe->scalar_type() != at::kFloat || !pe->is_contiguous() || lead < 0 || pe->size(lead) != L || pe->size(lead + 1) != D / 2 || pe->size(lead + 2) != 2 ||
        pe->size(lead + 3) != 2)
        Py_RETURN_NONE;
    const int64_t tables = pe->numel() / (L * D * 2);
    if (tables != 1 && !(lead == 2 && pe->size(0) == B && pe->size(1) == 1)) Py_RETURN_NONE;
    Tensor yq, yk;
    int rc;
    {
        const Tensor qa = *q, ka = *k, table = *pe;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(qa.device());
        yq = empty(qa.sizes(), qa.scalar_type(), qa);
        yk = empty(qa.sizes(), qa.scalar_type(), qa);
        flux_qkv_prep_args a = {};
        a.q_img = source(qa);
        a.k_img = source(ka);
        a.q_out = yq.data_ptr();
        a.k_out = yk.data_ptr();
        a.pe = static_cast<const float*>(table.data_ptr());
        a.pe_batch_stride = tables == 1 ? 0 : L * D * 2;
        a.B = B; a.H = H; a.Li = L; a.D = static_cast<int32_t>(D);
        a.dtype = a.scale_dtype = type_code(qa);
        a.eps = 1e-6f;
        rc = flux_qkv_prep(&a, stream_of(qa));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_qkv_prep");
    return two(yq, yk);
    END_HANDLE_TH_ERRORS
}

// ---- linear ------------------------------------------------------------------------------------

// linear(x, w, b or None, activation): y = act(x w^T + b), activation 0 or 1 (tanh GELU)
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4, "linear takes 4 arguments");
    const Tensor *x = tensor_of(args[0]), *w = tensor_of(args[1]), *b = args[2] == Py_None ? nullptr : tensor_of(args[2]);
    if (!x || !w || (!b && args[2] != Py_None) || !quiet() || x->scalar_type() != at::kBFloat16 || !same_kind(*x, *w) || w->dim() != 2 || !w->is_contiguous() || x->dim() < 1 ||
        x->size(-1) != w->size(1) || !x->is_contiguous())
        Py_RETURN_NONE;
    const int64_t N = w->size(0), K = w->size(1), M = x->numel() / K;
    if (b && (!same_kind(*x, *b) || b->dim() != 1 || b->numel() != N || b->stride(0) != 1)) Py_RETURN_NONE;
    const long act = PyLong_AsLong(args[3]);
    if (PyErr_Occurred()) return nullptr;
    Tensor y;
    int rc;
    {
        const Tensor xa = *x, wa = *w, ba = b ? *b : Tensor();
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(xa.device());
        at::DimVector sizes(xa.sizes().begin(), xa.sizes().end());
        sizes.back() = N;
        y = empty(sizes, at::kBFloat16, xa);
        flux_linear_args a = {};
        a.A = xa.data_ptr(); a.W = wa.data_ptr(); a.bias = ba.defined() ? ba.data_ptr() : nullptr;
        a.Y = y.data_ptr();
        a.M = M; a.N = N; a.K = K;
        a.lda = a.ldw = K;
        a.ldy = a.split_n = N;
        a.act = static_cast<int32_t>(act);
        // (K is cut over workgroups beyond 3072 of it only, and up to 256 tiles of 192 x 192)
        const int64_t need = K > 3072 && M > 8 && M * N <= (int64_t{1} << 24) ? flux_linear_workspace_bytes(&a) : 0;
        const Tensor ws = need ? empty({need}, at::kByte, xa) : Tensor();
        rc = flux_linear_bf16_ws(&a, need ? ws.data_ptr() : nullptr, need, stream_of(xa));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_linear_bf16");
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// ---- attention ---------------------------------------------------------------------------------

// attention(q, k, v, scale or None): all of [B, H, L, D]
PyObject* py_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4, "attention takes 4 arguments");
    const Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]);
    if (!q || !k || !v || !quiet() || q->dim() != 4 || q->sizes() != k->sizes() || q->sizes() != v->sizes() || q->scalar_type() != at::kBFloat16 || !same_kind(*q, *k) ||
        !same_kind(*q, *v))
        Py_RETURN_NONE;
    for (const Tensor* t : {q, k, v})
        if (t->stride(3) != 1 || !vector_rows(*t)) Py_RETURN_NONE;
    double scale = 1.0 / std::sqrt(static_cast<double>(q->size(3)));
    if (args[3] != Py_None && !number(args[3], scale)) Py_RETURN_NONE;
    Tensor o;
    int rc;
    {
        const Tensor qa = *q, ka = *k, va = *v;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(qa.device());
        o = empty(qa.sizes(), at::kBFloat16, qa);
        flux_attn_args a = {};
        a.q = source(qa); a.k = source(ka); a.v = source(va);
        a.o = o.data_ptr();
        a.o_sb = o.stride(0); a.o_sh = o.stride(1); a.o_sl = o.stride(2);
        a.B = qa.size(0); a.H = qa.size(1); a.L = qa.size(2); a.D = static_cast<int32_t>(qa.size(3));
        a.sm_scale = static_cast<float>(scale);
        const int64_t need = flux_attention_workspace_bytes(a.B, a.H, a.L, a.D);   // keys cut over several workgroups
        const Tensor ws = need ? empty({need}, at::kByte, qa) : Tensor();
        rc = flux_attention_fwd_bf16_ws(&a, need ? ws.data_ptr() : nullptr, need, stream_of(qa));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_attention_fwd_bf16");
    return THPVariable_Wrap(o);
    END_HANDLE_TH_ERRORS
}

#define FLUX_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FLUX_METHOD(rms_norm), FLUX_METHOD(rms_norm_pair), FLUX_METHOD(layer_norm_modulation), FLUX_METHOD(apply_rope), FLUX_METHOD(linear),
                         FLUX_METHOD(attention), {nullptr, nullptr, 0, nullptr}};
#undef FLUX_METHOD

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

#define FLUX_TEXT_(x) #x
#define FLUX_TEXT(x) FLUX_TEXT_(x)

PyMODINIT_FUNC PyInit__torch_ops() {
    if (flux_abi_version() != FLUX_ABI_VERSION) {
        PyErr_Format(PyExc_ImportError, "libfluxhip.so has ABI version %d, the extension was built for %d", flux_abi_version(), FLUX_ABI_VERSION);
        return nullptr;
    }
    PyObject* const m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "built_for", "torch " TORCH_VERSION ", Python " FLUX_TEXT(PY_MAJOR_VERSION) "." FLUX_TEXT(PY_MINOR_VERSION)) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
