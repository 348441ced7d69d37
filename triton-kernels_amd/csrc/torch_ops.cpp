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
// x 3072 15.8 -> 15.1 (the GPU's own time). The calls that the fused blocks are made of are here as well. Host time of a pass: the six of a single-stream
// block at 320 tokens 135 -> 78 (the GPU 120 there), the nine of a double-stream block at 1024 + 256 tokens 327 -> 160, of two batch elements
// at 256 + 64 338 -> 155; first passes on new weights 304 -> 214, 586 -> 474 and 546 -> 396.
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

#include <algorithm>
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

bool layer_norm_args_ok(const Tensor& x, const Tensor& scale, const Tensor& shift) {
    if (x.dim() < 2 || type_code(x) < 0 || !same_kind(x, scale) || !same_kind(x, shift) || !x.is_contiguous()) return false;
    const int64_t batch = x.size(0), n = x.size(-1);
    auto modulates = [&](const Tensor& m) {
        return m.dim() >= 2 && m.size(0) == batch && m.size(-1) == n && m.numel() == batch * n && m.stride(-1) == 1 && (batch == 1 || (m.stride(0) == scale.stride(0) && m.stride(0) >= n));
    };
    return n <= kMaxRow && modulates(scale) && modulates(shift);
}

flux_layer_norm_args layer_norm_args(const Tensor& x, const Tensor& scale, const Tensor& shift, const Tensor& y) {
    const int64_t batch = x.size(0), n = x.size(-1);
    return {x.data_ptr(), scale.data_ptr(), shift.data_ptr(), y.data_ptr(), batch, x.numel() / n / batch, batch > 1 ? scale.stride(0) : n};
}

// layer_norm_modulation(x, scale, shift, eps)
PyObject* py_layer_norm_modulation(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4, "layer_norm_modulation takes 4 arguments");
    const Tensor *x = tensor_of(args[0]), *scale = tensor_of(args[1]), *shift = tensor_of(args[2]);
    if (!x || !scale || !shift || !quiet() || !layer_norm_args_ok(*x, *scale, *shift)) Py_RETURN_NONE;
    double eps;
    if (!number(args[3], eps)) Py_RETURN_NONE;
    Tensor y;
    int rc;
    {
        const Tensor xa = *x, sc = *scale, sh = *shift;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(xa.device());
        y = at::empty_like(xa);
        const flux_layer_norm_args a = layer_norm_args(xa, sc, sh, y);
        rc = flux_layer_norm_modulation(a.x, a.scale, a.shift, a.y, a.batch, a.seq, static_cast<int32_t>(xa.size(-1)), a.mod_batch_stride, type_code(xa), static_cast<float>(eps), stream_of(xa));
    }
    if (rc < 0) Py_RETURN_NONE;   // (a refusal: its kind of error is the launcher's)
    check(rc, "flux_layer_norm_modulation");
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// layer_norm_modulation_pair(x0, scale0, shift0, x1, scale1, shift1, eps)
PyObject* py_layer_norm_modulation_pair(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 7, "layer_norm_modulation_pair takes 7 arguments");
    const Tensor* t[6];
    for (int i = 0; i < 6; ++i) {
        t[i] = tensor_of(args[i]);
        if (!t[i]) Py_RETURN_NONE;
    }
    if (!quiet() || !layer_norm_args_ok(*t[0], *t[1], *t[2]) || !layer_norm_args_ok(*t[3], *t[4], *t[5]) || !same_kind(*t[0], *t[3]) || t[0]->size(-1) != t[3]->size(-1)) Py_RETURN_NONE;
    double eps;
    if (!number(args[6], eps)) Py_RETURN_NONE;
    Tensor y0, y1;
    int rc;
    {
        const Tensor x0 = *t[0], s0 = *t[1], h0 = *t[2], x1 = *t[3], s1 = *t[4], h1 = *t[5];
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(x0.device());
        y0 = at::empty_like(x0);
        y1 = at::empty_like(x1);
        const flux_layer_norm_args a0 = layer_norm_args(x0, s0, h0, y0), a1 = layer_norm_args(x1, s1, h1, y1);
        rc = flux_layer_norm_modulation_pair(&a0, &a1, static_cast<int32_t>(x0.size(-1)), type_code(x0), static_cast<float>(eps), stream_of(x0));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_layer_norm_modulation_pair");
    return two(y0, y1);
    END_HANDLE_TH_ERRORS
}

// ---- rotation ----------------------------------------------------------------------------------

flux_src4 source(const Tensor& t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// A table for all batch elements (stride 0) or one for each, as it lies in memory.
bool rotation_table(const Tensor& pe, int64_t B, int64_t L, int64_t D, int64_t& batch_stride) {
    const int64_t lead = pe.dim() - 4;
    if (D % 2 != 0 || pe.scalar_type() != at::kFloat || !pe.is_contiguous() || lead < 0 || pe.size(lead) != L || pe.size(lead + 1) != D / 2 || pe.size(lead + 2) != 2 ||
        pe.size(lead + 3) != 2)
        return false;
    const int64_t tables = pe.numel() / (L * D * 2);
    batch_stride = tables == 1 ? 0 : L * D * 2;
    return tables == 1 || (lead == 2 && pe.size(0) == B && pe.size(1) == 1);
}

// apply_rope(q, k, table)
PyObject* py_apply_rope(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 3, "apply_rope takes 3 arguments");
    const Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *pe = tensor_of(args[2]);
    if (!q || !k || !pe || !quiet() || q->dim() != 4 || q->sizes() != k->sizes() || type_code(*q) < 0 || !same_kind(*q, *k) || q->device() != pe->device() ||
        q->stride(3) != 1 || k->stride(3) != 1 || !vector_rows(*q) || !vector_rows(*k))
        Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), L = q->size(2), D = q->size(3);
    int64_t table_stride;
    if (!rotation_table(*pe, B, L, D, table_stride)) Py_RETURN_NONE;
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
        a.pe_batch_stride = table_stride;
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

// A tensor or None.
bool optional_tensor(PyObject* o, const Tensor*& t) {
    t = o == Py_None ? nullptr : tensor_of(o);
    return t != nullptr || o == Py_None;
}

PyObject* wrap_or_none(const Tensor& t) {
    if (t.defined()) return THPVariable_Wrap(t);
    Py_RETURN_NONE;
}

// qkv_prep(q_img, k_img, v_img, q_txt, k_txt, v_txt, table, q_scale_img, k_scale_img, q_scale_txt, k_scale_txt, eps): (q, k, v), where
// q and k are there, v and the three of the text may be None
PyObject* py_qkv_prep(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 12, "qkv_prep takes 12 arguments");
    const Tensor* t[11];
    for (int i = 0; i < 11; ++i)
        if (!optional_tensor(args[i], t[i])) Py_RETURN_NONE;
    const Tensor *q = t[0], *pe = t[6];
    if (!q || !t[1] || !quiet() || q->dim() != 4 || type_code(*q) < 0 || (t[3] && t[3]->dim() != 4)) Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), Li = q->size(2), D = q->size(3), Lt = t[3] ? t[3]->size(2) : 0;
    for (int i = 0; i < 6; ++i) {
        if (!t[i]) {
            if (i < 2 || (i >= 3 && Lt > 0 && t[i - 3])) Py_RETURN_NONE;   // (q and k are there; what the image has, the text has)
            continue;
        }
        if (i >= 3 && (Lt == 0 || !t[i - 3])) Py_RETURN_NONE;
        if (!same_kind(*q, *t[i]) || t[i]->sizes() != at::IntArrayRef({B, H, i < 3 ? Li : Lt, D}) || t[i]->stride(3) != 1 || !vector_rows(*t[i])) Py_RETURN_NONE;
    }
    int64_t table_stride = 0;
    if (pe && (pe->device() != q->device() || !rotation_table(*pe, B, Lt + Li, D, table_stride))) Py_RETURN_NONE;
    int scale_type = type_code(*q);
    bool first = true;
    for (int i = 7; i < 11; ++i) {
        if (!t[i]) continue;
        const int type = type_code(*t[i]);
        if (type < 0 || (!first && type != scale_type) || (type != type_code(*q) && type_code(*q) != FLUX_BF16) || t[i]->device() != q->device() || t[i]->dim() != 1 ||
            t[i]->numel() != D || t[i]->stride(0) != 1)
            Py_RETURN_NONE;
        scale_type = type;
        first = false;
    }
    double eps;
    if (!number(args[11], eps)) Py_RETURN_NONE;
    Tensor out[3];
    int rc;
    {
        Tensor kept[11];   // (the caller's objects are another thread's to drop from here on)
        for (int i = 0; i < 11; ++i)
            if (t[i]) kept[i] = *t[i];
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(kept[0].device());
        for (int i = 0; i < 3; ++i)
            if (kept[i].defined()) out[i] = empty({B, H, Lt + Li, D}, kept[0].scalar_type(), kept[0]);
        auto at = [&](int i) { return kept[i].defined() ? source(kept[i]) : flux_src4{}; };
        auto ptr = [](const Tensor& x) -> void* { return x.defined() ? x.data_ptr() : nullptr; };
        flux_qkv_prep_args a = {};
        a.q_img = at(0); a.k_img = at(1); a.v_img = at(2);
        a.q_txt = at(3); a.k_txt = at(4); a.v_txt = at(5);
        a.q_out = ptr(out[0]); a.k_out = ptr(out[1]); a.v_out = ptr(out[2]);
        a.pe = static_cast<const float*>(ptr(kept[6]));
        a.pe_batch_stride = table_stride;
        a.q_scale_img = ptr(kept[7]); a.k_scale_img = ptr(kept[8]); a.q_scale_txt = ptr(kept[9]); a.k_scale_txt = ptr(kept[10]);
        a.B = B; a.H = H; a.Lt = Lt; a.Li = Li; a.D = static_cast<int32_t>(D);
        a.dtype = type_code(kept[0]);
        a.scale_dtype = scale_type;
        a.eps = static_cast<float>(eps);
        rc = flux_qkv_prep(&a, stream_of(kept[0]));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_qkv_prep");
    PyObject* const r = PyTuple_New(3);
    if (!r) return nullptr;
    for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(r, i, wrap_or_none(out[i]));
    return r;
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

// One product in its general form, and what has to live until it is launched.
struct Product {
    flux_linear_args a = {};
    flux_linear_qk_fusion qk = {};
    int64_t a_rows = 0, a_batch_stride = 0;
    Tensor out;
    c10::SmallVector<Tensor, 12> keep;
    bool out_given = false;
};

bool whole_number(PyObject* o, int64_t& value) {
    value = PyLong_CheckExact(o) ? PyLong_AsLongLong(o) : -1;
    if (PyLong_CheckExact(o) && !(value == -1 && PyErr_Occurred())) return true;
    PyErr_Clear();
    return false;
}

// x as [rows, n] without copying it.
bool flat_rows(const Tensor& x, int64_t n, int64_t& rows, int64_t& ld) {
    if (x.dim() < 1 || x.size(-1) != n || (n > 1 && x.stride(-1) != 1)) return false;
    rows = 1;
    ld = n;
    for (int64_t d = x.dim() - 2; d >= 0; --d) {
        if (x.size(d) == 1) continue;
        if (rows == 1) ld = x.stride(d);
        else if (x.stride(d) != ld * rows) return false;
        rows *= x.size(d);
    }
    return ld >= n;
}

bool is_bf16(const Tensor& t, const Tensor& beside) { return t.scalar_type() == at::kBFloat16 && t.device() == beside.device(); }

// A matrix of at least `cols` columns to write to.
bool destination(const Tensor& t, const Tensor& x, int64_t rows, int64_t cols) {
    return is_bf16(t, x) && t.dim() == 2 && t.size(0) == rows && t.stride(1) == 1 && t.size(1) >= cols;
}

// call: (x, w, b, activation, act_begin, out, out2, split, resid, gate, qk, in_activation) as linear_into has them, absent ones None;
// qk: (q_out, k_out, q_scale, k_scale, table, heads, seq_len, pos0, eps) or None. slices: rows of x may lie in batches that are not evenly strided.
bool read_product(PyObject* call, Product& p, bool slices) {
    if (!PyTuple_CheckExact(call) || PyTuple_GET_SIZE(call) != 12) return false;
    auto item = [&](int i) { return PyTuple_GET_ITEM(call, i); };
    const Tensor *x = tensor_of(item(0)), *w = tensor_of(item(1)), *b, *out, *out2, *resid, *gate;
    int64_t act, act_begin, in_act, split = -1;
    if (!x || !w || !optional_tensor(item(2), b) || !optional_tensor(item(5), out) || !optional_tensor(item(6), out2) || !optional_tensor(item(8), resid) ||
        !optional_tensor(item(9), gate) || !whole_number(item(3), act) || !whole_number(item(4), act_begin) || !whole_number(item(11), in_act) ||
        (item(7) != Py_None && (!whole_number(item(7), split) || split < 0)))
        return false;
    if (act < 0 || in_act < 0 || x->scalar_type() != at::kBFloat16 || !is_bf16(*w, *x) || w->dim() != 2 || x->size(-1) != w->size(1) || (w->size(1) > 1 && w->stride(1) != 1)) return false;
    const int64_t N = w->size(0), K = w->size(1);
    if (N > 1 && w->stride(0) < K) return false;
    int64_t M, ld;
    if (slices && x->dim() == 3 && x->size(0) > 1 && x->stride(0) != x->size(1) * x->stride(1)) {
        const int64_t B = x->size(0), L = x->size(1);
        if (!(B * L > 8 && x->stride(2) == 1 && x->stride(1) >= K && x->stride(0) % 8 == 0 && x->stride(0) >= L * x->stride(1) && x->stride(1) % 8 == 0 && K % 8 == 0 &&
              reinterpret_cast<uintptr_t>(x->data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w->data_ptr()) % 16 == 0 && w->is_contiguous() && B * x->stride(0) * 2 < (int64_t{1} << 31)))
            return false;
        M = B * L;
        ld = x->stride(1);
        p.a_rows = L;
        p.a_batch_stride = x->stride(0);
    } else if (!flat_rows(*x, K, M, ld)) {
        return false;
    }
    if (in_act != FLUX_ACT_NONE && M > 8) return false;
    if (b && (!is_bf16(*b, *x) || b->dim() != 1 || b->numel() != N || b->stride(0) != 1)) return false;
    if (split > N) return false;   // (the launcher's output has `split` columns)
    const bool cut = split >= 0 && split < N;
    if (out && !destination(*out, *x, M, cut ? split : N)) return false;
    if (cut && (!out2 || !destination(*out2, *x, M, N - split))) return false;
    if ((gate == nullptr) != (resid == nullptr)) return false;
    flux_linear_args& a = p.a;
    if (gate) {
        int64_t rows, ldr;
        if (!is_bf16(*gate, *x) || !is_bf16(*resid, *x) || !flat_rows(*resid, N, rows, ldr) || rows != M) return false;
        const int64_t nb = gate->is_contiguous() ? gate->numel() / N : gate->size(0);
        if (gate->dim() < 1 || gate->size(-1) != N || gate->stride(-1) != 1 || gate->numel() != nb * N || nb == 0 || M % nb != 0) return false;
        a.resid = resid->data_ptr();
        a.ldresid = ldr;
        a.gate = gate->data_ptr();
        a.gate_batch_stride = nb > 1 && !gate->is_contiguous() ? gate->stride(0) : N;
        a.rows_per_batch = M / nb;
        p.keep.push_back(*gate);
        p.keep.push_back(*resid);
    }
    if (item(10) != Py_None) {
        PyObject* const q = item(10);
        if (!PyTuple_CheckExact(q) || PyTuple_GET_SIZE(q) != 9) return false;
        const Tensor* t[5];
        for (int i = 0; i < 5; ++i)
            if (!(t[i] = tensor_of(PyTuple_GET_ITEM(q, i))) || t[i]->device() != x->device() || !t[i]->is_contiguous()) return false;
        double eps;
        flux_linear_qk_fusion& f = p.qk;
        if (!whole_number(PyTuple_GET_ITEM(q, 5), f.heads) || !whole_number(PyTuple_GET_ITEM(q, 6), f.seq_len) || !whole_number(PyTuple_GET_ITEM(q, 7), f.pos0) ||
            !number(PyTuple_GET_ITEM(q, 8), eps))
            return false;
        if (t[0]->dim() != 4 || t[0]->sizes() != t[1]->sizes() || !is_bf16(*t[0], *x) || !is_bf16(*t[1], *x) || f.seq_len <= 0 || M % f.seq_len != 0 || t[0]->size(0) != M / f.seq_len ||
            t[0]->size(1) != f.heads || t[0]->size(3) != 128)
            return false;
        f.out_len = t[0]->size(2);
        const int64_t table = f.out_len * 256;
        if (t[4]->scalar_type() != at::kFloat || t[4]->numel() % table != 0) return false;
        for (int i = 2; i < 4; ++i)
            if (!is_bf16(*t[i], *x) || t[i]->numel() != 128) return false;
        f.q_out = t[0]->data_ptr(); f.k_out = t[1]->data_ptr();
        f.q_scale = t[2]->data_ptr(); f.k_scale = t[3]->data_ptr();
        f.pe = static_cast<const float*>(t[4]->data_ptr());
        f.pe_batch_stride = t[4]->numel() > table ? table : 0;
        f.eps = static_cast<float>(eps);
        for (const Tensor* k : t) p.keep.push_back(*k);
        a.qk = &f;
    }
    a.A = x->data_ptr(); a.W = w->data_ptr(); a.bias = b ? b->data_ptr() : nullptr;
    a.M = M; a.N = N; a.K = K;
    a.lda = M > 1 ? ld : K;
    a.ldw = N > 1 ? w->stride(0) : K;
    a.split_n = cut ? split : N;
    if (cut) { a.Y2 = out2->data_ptr(); a.ldy2 = out2->stride(0); p.keep.push_back(*out2); }
    a.act = static_cast<int32_t>(act);
    a.act_begin = act_begin;
    a.in_act = static_cast<int32_t>(in_act);
    p.keep.push_back(*x);
    p.keep.push_back(*w);
    if (b) p.keep.push_back(*b);
    if (out) { p.out = *out; p.out_given = true; }
    return true;
}

// The output, where the caller gave none, and its place in the call.
void place_output(Product& p, const Tensor& beside) {
    if (!p.out_given) p.out = empty({p.a.M, p.a.split_n}, at::kBFloat16, beside);
    p.a.Y = p.out.data_ptr();
    p.a.ldy = p.out.stride(0);
}

// (K is cut over workgroups beyond 3072 of it only, and up to 256 tiles of 192 x 192)
bool may_cut_k(int64_t rows, int64_t N, int64_t K) { return K > 3072 && rows > 8 && rows * N <= (int64_t{1} << 24); }

// linear_into(call)
PyObject* py_linear_into(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 1, "linear_into takes 1 argument");
    Product p;
    if (!quiet() || !read_product(args[0], p, false)) Py_RETURN_NONE;
    int rc;
    {
        const WithoutInterpreter free;
        const Tensor& beside = p.keep.back();
        const c10::DeviceGuard guard(beside.device());
        place_output(p, beside);
        const int64_t need = may_cut_k(p.a.M, p.a.N, p.a.K) ? flux_linear_workspace_bytes(&p.a) : 0;
        const Tensor ws = need ? empty({need}, at::kByte, beside) : Tensor();
        rc = flux_linear_bf16_ws(&p.a, need ? ws.data_ptr() : nullptr, need, stream_of(beside));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_linear_bf16");
    return THPVariable_Wrap(p.out);
    END_HANDLE_TH_ERRORS
}

// linear_pair_into(call, call)
PyObject* py_linear_pair_into(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 2, "linear_pair_into takes 2 arguments");
    Product p[2];
    if (!quiet() || !read_product(args[0], p[0], true) || !read_product(args[1], p[1], true) || p[0].keep.back().device() != p[1].keep.back().device()) Py_RETURN_NONE;
    int rc;
    {
        const WithoutInterpreter free;
        const Tensor& beside = p[0].keep.back();
        const c10::DeviceGuard guard(beside.device());
        flux_linear_pair_args a = {};
        for (int i = 0; i < 2; ++i) {
            place_output(p[i], beside);
            a.product[i] = p[i].a;
            a.a_rows[i] = p[i].a_rows;
            a.a_batch_stride[i] = p[i].a_batch_stride;
        }
        const int64_t need = may_cut_k(p[0].a.M + p[1].a.M, std::min(p[0].a.N, p[1].a.N), std::max(p[0].a.K, p[1].a.K)) ? flux_linear_pair_workspace_bytes(&a) : 0;
        const Tensor ws = need ? empty({need}, at::kByte, beside) : Tensor();
        rc = flux_linear_bf16_pair(&a, need ? ws.data_ptr() : nullptr, need, stream_of(beside));
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_linear_bf16_pair");
    return two(p[0].out, p[1].out);
    END_HANDLE_TH_ERRORS
}

// ---- attention ---------------------------------------------------------------------------------

// attention(q, k, v, scale or None): all of [B, H, L, D]; attention(q, k, v, scale or None, out, calls): to a tensor that is there, beside up to two
// products (as read_product has them)
PyObject* py_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4 || nargs == 6, "attention takes 4 or 6 arguments");
    const Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]), *out = nargs == 6 ? tensor_of(args[4]) : nullptr;
    if (!q || !k || !v || (nargs == 6 && !out) || !quiet() || q->dim() != 4 || q->sizes() != k->sizes() || q->sizes() != v->sizes() || q->scalar_type() != at::kBFloat16 ||
        !same_kind(*q, *k) || !same_kind(*q, *v) || (out && (out->sizes() != q->sizes() || !same_kind(*q, *out) || out->stride(3) != 1)))
        Py_RETURN_NONE;
    for (const Tensor* t : {q, k, v})
        if (t->stride(3) != 1 || !vector_rows(*t)) Py_RETURN_NONE;
    double scale = 1.0 / std::sqrt(static_cast<double>(q->size(3)));
    if (args[3] != Py_None && !number(args[3], scale)) Py_RETURN_NONE;
    Product p[2];
    const Py_ssize_t products = nargs == 6 && PyTuple_CheckExact(args[5]) ? PyTuple_GET_SIZE(args[5]) : 0;
    if (products > 2 || (nargs == 6 && !PyTuple_CheckExact(args[5]))) Py_RETURN_NONE;
    for (Py_ssize_t i = 0; i < products; ++i)
        if (!read_product(PyTuple_GET_ITEM(args[5], i), p[i], false) || !p[i].out_given || p[i].out.device() != q->device()) Py_RETURN_NONE;
    Tensor o;
    int rc;
    {
        const Tensor qa = *q, ka = *k, va = *v;
        if (out) o = *out;
        const WithoutInterpreter free;
        const c10::DeviceGuard guard(qa.device());
        if (!out) o = empty(qa.sizes(), at::kBFloat16, qa);
        flux_attn_args a = {};
        a.q = source(qa); a.k = source(ka); a.v = source(va);
        a.o = o.data_ptr();
        a.o_sb = o.stride(0); a.o_sh = o.stride(1); a.o_sl = o.stride(2);
        a.B = qa.size(0); a.H = qa.size(1); a.L = qa.size(2); a.D = static_cast<int32_t>(qa.size(3));
        a.sm_scale = static_cast<float>(scale);
        const int64_t need = flux_attention_workspace_bytes(a.B, a.H, a.L, a.D);   // keys cut over several workgroups
        const Tensor ws = need ? empty({need}, at::kByte, qa) : Tensor();
        void* const ws_at = need ? ws.data_ptr() : nullptr;
        if (products == 0) {
            rc = flux_attention_fwd_bf16_ws(&a, ws_at, need, stream_of(qa));
        } else {
            flux_linear_pair_args rows = {};
            for (int i = 0; i < 2; ++i) {
                Product& at = p[i < products ? i : 0];
                place_output(at, qa);
                rows.product[i] = at.a;
            }
            if (products == 1) rows.product[1].M = 0;
            rc = flux_attention_rows_bf16(&a, &rows, ws_at, need, stream_of(qa));
        }
    }
    if (rc < 0) Py_RETURN_NONE;
    check(rc, "flux_attention_fwd_bf16");
    return THPVariable_Wrap(o);
    END_HANDLE_TH_ERRORS
}

#define FLUX_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FLUX_METHOD(rms_norm), FLUX_METHOD(rms_norm_pair), FLUX_METHOD(layer_norm_modulation), FLUX_METHOD(layer_norm_modulation_pair), FLUX_METHOD(apply_rope),
                         FLUX_METHOD(qkv_prep), FLUX_METHOD(linear), FLUX_METHOD(linear_into), FLUX_METHOD(linear_pair_into), FLUX_METHOD(attention), {nullptr, nullptr, 0, nullptr}};
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
