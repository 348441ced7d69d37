"""scaled_dot_product_attention: non-causal flash-attention forward (kernels/attention.py:173-221 of
the reference) on the HIP kernel flux_attention_fwd_bf16."""
from __future__ import annotations

import math

import torch
from torch import Tensor
from torch.compiler import is_compiling

from triton_kernels import _native as nv
from triton_kernels.kernels.linear import hooked, positional, rows_args


def _bhld_view(t: Tensor) -> Tensor:
    if t.stride(-1) != 1 or any(s % 8 for s in t.stride()[:-1]) or t.data_ptr() % 16:
        t = t.contiguous()
    return t


def _may_cut_keys(BH: int, L: int) -> bool:
    """False where flux_attention_workspace_bytes is known to be 0, so that the call is spared the question (0.4 of
    16 us of host time): keys are cut in two or more parts up to 256 workgroups of 128 rows in all, and sixteen
    tiles of 64 keys are too few to pay for the second launch."""
    return L > 1024 and BH * ((L + 127) // 128) <= 128


def takes_rows(BH: int, L: int, D: int, rows: int, K: int) -> bool:
    """Whether products of `rows` rows in all with K values each run beside an attention (attention_into's `beside`) and not in
    front of it (flux_attention_rows_bf16)."""
    return D == 128 and 64 < L and BH * ((L + 127) // 128) <= 256 and not _may_cut_keys(BH, L) and rows <= 4 and rows * K * 2 <= 48 * 1024


def attention_into(q: Tensor, k: Tensor, v: Tensor, out: Tensor, sm_scale: float | None = None,
                   lse: Tensor | None = None, beside: tuple[dict, ...] = ()) -> Tensor:
    """q,k,v,out are [B,H,L,D] views (bf16, last dim contiguous, any other strides).
    beside: one or two linear_into calls of a few rows (the keyword arguments of each) that have nothing to do with the
    attention; the library runs them beside it in one launch where it can."""
    if lse is None and not (beside and hooked()) and not is_compiling():
        o = nv.ops().attention(q, k, v, sm_scale, out, tuple(positional(**call) for call in beside))
        if o is not None:
            return o
    D = q.shape[-1]
    assert D == k.shape[-1] == v.shape[-1]
    assert D in {16, 32, 64, 128, 256}
    assert q.dim() == 4 and q.shape == k.shape == v.shape == out.shape
    if q.dtype != torch.bfloat16 or k.dtype != q.dtype or v.dtype != q.dtype or out.dtype != q.dtype:
        raise TypeError("scaled_dot_product_attention: the HIP kernel takes bfloat16 q, k, v")
    dev = nv.require_gpu(q, k, v, out, lse)
    if sm_scale is None:
        sm_scale = 1 / math.sqrt(D)
    q, k, v = _bhld_view(q), _bhld_view(k), _bhld_view(v)
    B, H, L, _ = q.shape
    a = nv.AttnArgs()
    a.q, a.k, a.v = nv.src4(q), nv.src4(k), nv.src4(v)
    a.o, a.o_sb, a.o_sh, a.o_sl = out.data_ptr(), out.stride(0), out.stride(1), out.stride(2)
    assert out.stride(3) == 1
    a.lse = nv.ptr(lse)
    a.B, a.H, a.L, a.D, a.sm_scale = B, H, L, D, float(sm_scale)
    with nv.on_device(dev):
        need = nv.lib().flux_attention_workspace_bytes(B, H, L, D) if _may_cut_keys(B * H, L) else 0
        if beside:
            rows, _keep = rows_args(beside, dev)
            ws = torch.empty((need,), dtype=torch.uint8, device=dev) if need else None
            rc = nv.lib().flux_attention_rows_bf16(nv.byref(a), nv.byref(rows), nv.ptr(ws), need, nv.stream_ptr(dev))
        elif need:   # keys cut over several workgroups: partial sums in memory of this launch's stream
            ws = torch.empty((need,), dtype=torch.uint8, device=dev)
            rc = nv.lib().flux_attention_fwd_bf16_ws(nv.byref(a), ws.data_ptr(), need, nv.stream_ptr(dev))
        else:
            rc = nv.lib().flux_attention_fwd_bf16(nv.byref(a), nv.stream_ptr(dev))
    nv.check(rc, "flux_attention_fwd_bf16")
    return out


def scaled_dot_product_attention(q: Tensor, k: Tensor, v: Tensor, sm_scale: float = None) -> Tensor:
    o = None if is_compiling() else nv.ops().attention(q, k, v, sm_scale)
    if o is not None:
        return o
    o = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    return attention_into(q, k, v, o, sm_scale)
