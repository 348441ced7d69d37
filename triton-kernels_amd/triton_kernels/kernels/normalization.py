"""rms_norm and layer_norm_modulation: Python launchers over the HIP row-wise kernels.

Same call signatures, defaults and assertion behaviour as kernels/normalization.py:47-77 and
:142-193 of the reference; the device work is flux_rms_norm / flux_rms_norm_bwd /
flux_layer_norm_modulation in libfluxhip.so.
"""
from __future__ import annotations

import torch
from torch.compiler import is_compiling

from triton_kernels import _native as nv
from triton_kernels.kernels.utils import calculate_settings


def _as_4d_view(x: torch.Tensor):
    """Sizes (d0,d1,d2) and strides (s0,s1,s2) of x seen as [d0,d1,d2,n] rows, without copying when x
    has at most four dims and a contiguous last dim; otherwise a contiguous copy is described."""
    if x.dim() == 0:
        raise AssertionError("rms_norm needs at least one dimension")
    if x.dim() > 4 or x.stride(-1) != 1:
        x = x.contiguous()
        if x.dim() > 4:
            x = x.reshape(-1, x.shape[-1])
    lead, strides = tuple(x.shape)[:-1], x.stride()[:-1]
    short = 3 - len(lead)
    if short:
        lead, strides = (1,) * short + lead, (0,) * short + strides
    return x, lead, strides


def _rms_norm_args(x: torch.Tensor, scale: torch.Tensor, want_rstd: bool = False):
    """The call's arguments in the order of nv.RmsNormArgs, its outputs and the tensors that have to live until
    it is launched."""
    shape, dtype = x.shape, x.dtype
    assert shape[-1] == scale.shape[-1]
    dev = nv.require_gpu(x, scale)
    if shape[-1] > nv.MAX_ROW:
        calculate_settings(shape[-1])  # raises, like the reference
    scale = scale.contiguous()
    if scale.dtype != dtype and not (dtype == torch.bfloat16 and scale.dtype == torch.float32):
        scale = scale.to(dtype)
    xv, lead, strides = _as_4d_view(x)
    y = torch.empty(shape, dtype=dtype, device=dev)
    rstd = torch.empty((lead[0] * lead[1] * lead[2],), dtype=torch.float32, device=dev) if want_rstd else None
    return (xv.data_ptr(), scale.data_ptr(), y.data_ptr(), rstd.data_ptr() if want_rstd else None, *lead, *strides), y, rstd, (xv, scale)


def rms_norm_forward(x: torch.Tensor, scale: torch.Tensor, eps: float = 1e-6, want_rstd: bool = False):
    a, y, rstd, (xv, scale) = _rms_norm_args(x, scale, want_rstd)
    dev = y.device
    with nv.on_device(dev):
        rc = nv.lib().flux_rms_norm(
            *a[:7], y.shape[-1], *a[7:],
            nv.dtype_code(y), nv.dtype_code(scale), float(eps), nv.stream_ptr(dev))
    nv.check(rc, "flux_rms_norm")
    return y, rstd, xv


def _vector_rows(x: torch.Tensor) -> bool:
    """Whether every row of x starts on a 16-byte boundary, where the kernel holds a row in registers."""
    per16 = 16 // x.element_size()
    return x.data_ptr() % 16 == 0 and x.shape[-1] % per16 == 0 and all(s % per16 == 0 for s in x.stride()[:-1])


class _rms_norm(torch.autograd.Function):
    """y = x * rsqrt(mean(x^2, -1) + eps) * scale with a HIP forward and backward.

    grad_mode = False says that nothing will be differentiated (a parameter's requires_grad stays true under
    no_grad): a view with 16-byte rows is then read in place and no rstd is kept. Rows that are not 16-byte
    addressable are still copied first, since the kernel for such rows reads a row twice by elements."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, scale: torch.Tensor, eps: float = 1e-6, grad_mode: bool = True) -> torch.Tensor:
        need_grad = x.requires_grad or scale.requires_grad
        if need_grad and (grad_mode or not _vector_rows(x)):
            x = x.contiguous()
        need_grad = need_grad and grad_mode
        y, rstd, _ = rms_norm_forward(x, scale, eps, want_rstd=need_grad)
        if need_grad:
            ctx.save_for_backward(x.reshape(-1, x.shape[-1]), scale.contiguous(), rstd)
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        x2, scale, rstd = ctx.saved_tensors   # (what saved-tensor hooks gave back, of any type)
        dev = nv.require_gpu(dy, x2, scale, rstd)
        rows, n = x2.shape
        if scale.numel() != n or rstd.numel() != rows:
            raise RuntimeError("rms_norm: saved tensors came back with other sizes")
        x2, rstd = x2.contiguous(), rstd.float().contiguous()
        dy2 = dy.contiguous().reshape(rows, n)
        if dy2.dtype != x2.dtype:
            dy2 = dy2.to(x2.dtype)
        sc = scale.contiguous()
        if sc.dtype != x2.dtype and not (x2.dtype == torch.bfloat16 and sc.dtype == torch.float32):
            sc = sc.to(x2.dtype)
        dx = torch.empty_like(x2)
        # the kernel's types; the gradient of a scale of another type is converted from fp32 below
        dscale = torch.empty((n,), dtype=scale.dtype if scale.dtype == torch.bfloat16 else torch.float32, device=dev)
        xcode = nv.dtype_code(x2)
        ws = torch.empty((nv.lib().flux_rms_norm_bwd_workspace_bytes(rows, n, xcode),), dtype=torch.uint8, device=dev)
        with nv.on_device(dev):
            rc = nv.lib().flux_rms_norm_bwd_ws(
                dy2.data_ptr(), x2.data_ptr(), sc.data_ptr(), rstd.data_ptr(), dx.data_ptr(), dscale.data_ptr(), nv.dtype_code(dscale),
                ws.data_ptr(), ws.numel(), rows, n, xcode, nv.dtype_code(sc), nv.stream_ptr(dev))
        nv.check(rc, "flux_rms_norm_bwd")
        return dx.reshape(dy.shape), dscale.to(scale.dtype).reshape(scale.shape), None, None


def rms_norm(x: torch.Tensor, scale: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    y = None if is_compiling() else nv.ops().rms_norm(x, scale, eps)
    return _rms_norm.apply(x, scale, eps, torch.is_grad_enabled()) if y is None else y


class _rms_norm_pair(torch.autograd.Function):
    """rms_norm of two tensors in one launch, for calls that are not differentiated. A Function all the same, so
    that forward-mode derivatives and function transforms are refused as they are by rms_norm."""

    @staticmethod
    def forward(ctx, x0, scale0, x1, scale1, eps):
        a0, y0, _, (_x0, s0) = _rms_norm_args(x0, scale0)
        a1, y1, _, (_x1, s1) = _rms_norm_args(x1, scale1)
        dev = y0.device
        with nv.on_device(dev):
            rc = nv.lib().flux_rms_norm_pair(
                nv.byref(nv.RmsNormArgs(*a0)), nv.byref(nv.RmsNormArgs(*a1)), y0.shape[-1], nv.dtype_code(y0), nv.dtype_code(s0), float(eps), nv.stream_ptr(dev))
        nv.check(rc, "flux_rms_norm_pair")
        return y0, y1


def rms_norm_pair(x0, scale0, x1, scale1, eps: float = 1e-6) -> tuple[torch.Tensor, torch.Tensor]:
    """(rms_norm(x0, scale0), rms_norm(x1, scale1)): one launch where nothing is differentiated and the two have
    the same width, types and device and 16-byte rows, two calls otherwise. At [1, 24, 256, 128] (q and k of one projection) the
    two calls took 50 us of host time, the copies of the views included; this takes 23, and 8 in native code."""
    y = None if is_compiling() else nv.ops().rms_norm_pair(x0, scale0, x1, scale1, eps)
    if y is not None:
        return y
    if (torch.is_grad_enabled() or x0.dtype != x1.dtype or x0.device != x1.device or scale0.dtype != scale1.dtype
            or not x0.dim() or not x1.dim() or x0.shape[-1] != x1.shape[-1] or not (_vector_rows(x0) and _vector_rows(x1))):
        return rms_norm(x0, scale0, eps), rms_norm(x1, scale1, eps)
    return _rms_norm_pair.apply(x0, scale0, x1, scale1, eps)


def layer_norm_modulation(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, eps=1e-5) -> torch.Tensor:
    """(1 + weight) * layer_norm(x) + bias, where weight is the adaLN *scale* and bias the *shift*,
    each [B, 1, N] (or [B, N]); chunks of a wider modulation tensor are read in place."""
    y = None if is_compiling() else nv.ops().layer_norm_modulation(x, weight, bias, eps)
    if y is not None:
        return y
    a, y, _keep = _layer_norm_args(x, weight, bias)
    dev = y.device
    with nv.on_device(dev):
        rc = nv.lib().flux_layer_norm_modulation(
            *a[:6], y.shape[-1], a[6], nv.dtype_code(y), float(eps), nv.stream_ptr(dev))
    nv.check(rc, "flux_layer_norm_modulation")
    return y


def layer_norm_modulation_pair(first: tuple, second: tuple, eps=1e-5) -> tuple[torch.Tensor, torch.Tensor]:
    """layer_norm_modulation of two (x, weight, bias) triples of the same width and type in one launch."""
    y = nv.ops().layer_norm_modulation_pair(*first, *second, eps) if len(first) == len(second) == 3 and not is_compiling() else None
    if y is not None:
        return y
    a0, y0, _keep0 = _layer_norm_args(*first)
    a1, y1, _keep1 = _layer_norm_args(*second)
    assert y0.shape[-1] == y1.shape[-1] and y0.dtype == y1.dtype and y0.device == y1.device
    dev = y0.device
    with nv.on_device(dev):
        rc = nv.lib().flux_layer_norm_modulation_pair(
            nv.byref(nv.LayerNormArgs(*a0)), nv.byref(nv.LayerNormArgs(*a1)), y0.shape[-1], nv.dtype_code(y0), float(eps), nv.stream_ptr(dev))
    nv.check(rc, "flux_layer_norm_modulation_pair")
    return y0, y1


def _layer_norm_args(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor):
    """The call's arguments in the order of nv.LayerNormArgs, its output and the tensors that have to live until
    it is launched."""
    shape, weight_shape, bias_shape = x.shape, weight.shape, bias.shape
    batch, n = shape[0], shape[-1]
    assert batch == weight_shape[0] == bias_shape[0]
    assert n == weight_shape[-1] == bias_shape[-1]
    nv.require_gpu(x, weight, bias)
    if n > nv.MAX_ROW:
        calculate_settings(n)
    x = x.contiguous()
    if weight.dtype != x.dtype:
        weight = weight.to(x.dtype)
    if bias.dtype != x.dtype:
        bias = bias.to(x.dtype)
    assert weight.numel() == batch * n and bias.numel() == batch * n, "scale/shift must be [B, 1, N]"
    in_place = weight.stride(-1) == 1 and bias.stride(-1) == 1 and (batch == 1 or weight.stride(0) == bias.stride(0))
    if not in_place:
        weight, bias = weight.contiguous(), bias.contiguous()
    mod_stride = weight.stride(0) if batch > 1 else n
    if batch > 1 and mod_stride < n:
        weight, bias = weight.contiguous(), bias.contiguous()
        mod_stride = weight.stride(0)
    y = torch.empty_like(x)
    rows = x.numel() // n
    return (x.data_ptr(), weight.data_ptr(), bias.data_ptr(), y.data_ptr(), batch, rows // batch if batch else 0, mod_stride), y, (x, weight, bias)
