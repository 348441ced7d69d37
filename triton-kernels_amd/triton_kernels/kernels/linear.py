"""linear: y = act(x @ w.T + b) on the bf16 matrix cores (kernels/linear.py:104-151 of the reference),
with the extra epilogues the fused Flux blocks use."""
from __future__ import annotations

import ctypes

import torch
from torch import Tensor
from torch.compiler import is_compiling

from triton_kernels import _native as nv

_ACTIVATIONS = {"": nv.ACT_NONE, "GELU": nv.ACT_GELU_TANH}
# Tile plan per dtype; like the reference's table it has a single entry, so any other dtype is a KeyError.
_PLANS = {torch.bfloat16: {"tile": (256, 256, 64), "waves": 4, "mfma": "16x16x32"}}


# Optional callable(dict) invoked with the metadata of every launch of the linear kernel, on the launching
# thread, right before the launch. Profilers and benchmarks set it (e.g. to open a named range); None
# costs nothing. The dictionary is what the reference attaches to its launches for its profiler
# (kernels/linear.py:9-19): "name" with the problem size, "flops16" = 2 M N K and "bytes" = the three
# matrices once; a launch of two products names both row counts ("M=4096+512") and counts both.
launch_hook = None


def hooked() -> bool:
    return launch_hook is not None


def linear_launch_metadata(M: int, N: int, K: int, elem_bytes: int = 2, epilogue: str = "") -> dict:
    name = f"flux_linear_bf16 [M={M}, N={N}, K={K}]" + (f" {epilogue}" if epilogue else "")
    return {"name": name, f"flops{elem_bytes * 8}": 2.0 * M * N * K, "bytes": elem_bytes * (M * K + N * K + M * N)}


def _pair_launch_metadata(first: dict, second: dict, sizes: list) -> dict:
    both = {key: first[key] + second[key] for key in first if key != "name"}
    return {"name": first["name"].replace(f"[M={sizes[0][0]},", f"[M={sizes[0][0]}+{sizes[1][0]},"), **both}


def _rows_2d(x: Tensor, K: int) -> Tensor:
    x2 = x.reshape(-1, K)
    if x2.shape[0] > 1 and (x2.stride(1) != 1 or x2.stride(0) < K):
        x2 = x2.contiguous()
    elif x2.shape[0] <= 1 and x2.stride(1) != 1:
        x2 = x2.contiguous()
    return x2


def _may_cut_k(rows: int, N: int, K: int) -> bool:
    """False where flux_linear_workspace_bytes is known to be 0, so that the call is spared the question (0.5 us of
    14 us of host time, 1 to 3 us where the library has tiles to choose from): K is cut where that gains more than 6
    us, which takes more than 3072 of it, and only up to 256 tiles of 192 x 192."""
    return K > 3072 and rows > 8 and rows * N <= 1 << 24


_IN_ACTIVATIONS = {"": nv.ACT_NONE, "SiLU": nv.ACT_SILU}


def positional(x, w, b, *, activation="", act_begin=0, out=None, out2=None, split=None, resid=None, gate=None, qk=None, in_activation="", shared_gpu=False):
    """A linear_into call as the native calls take it."""
    if qk is not None:
        qk = (qk["q_out"], qk["k_out"], qk["q_scale"], qk["k_scale"], qk["pe"], qk["heads"], qk["seq_len"], qk.get("pos0", 0), qk.get("eps", 1e-6))
    return (x, w, b, -1 if shared_gpu else _ACTIVATIONS.get(activation, -1), act_begin, out, out2, split, resid, gate, qk, _IN_ACTIVATIONS.get(in_activation, -1))


def linear_into(x: Tensor, w: Tensor, b: Tensor | None, *, activation: str = "", act_begin: int = 0,
                out: Tensor | None = None, out2: Tensor | None = None, split: int | None = None,
                resid: Tensor | None = None, gate: Tensor | None = None, qk: dict | None = None,
                in_activation: str = "", shared_gpu: bool = False) -> Tensor:
    """General form of the fused linear.

    out   : [M, >=split] destination (row stride free) for columns [0, split)
    out2  : destination for columns [split, N), written starting at its column 0
    act_begin : GELU applies to columns >= act_begin only
    resid, gate : y = resid + gate * y with resid [..., N] and gate [B, 1, N] (or [B, N])
    in_activation : "SiLU" applies x * sigmoid(x) (rounded to bf16) to x on the way in; at most 8 rows
    qk    : QK RMSNorm + RoPE on the way out for the leading 2 * heads * 128 columns (q heads, then k
            heads), which then go to q_out / k_out [B, heads, out_len, 128] instead of `out`:
            dict(q_out, k_out, q_scale, k_scale, pe, heads, seq_len, pos0=0, eps=1e-6); see
            qk_fusable() for the shapes this form takes
    shared_gpu : the launch runs beside another stream's work; the library then keeps a tile shape
            that leaves CUs free in its last round instead of one that fills the GPU exactly (same
            result, only the schedule differs); for callers that run streams side by side
    """
    if launch_hook is None and not is_compiling():
        y = nv.ops().linear_into(positional(x, w, b, activation=activation, act_begin=act_begin, out=out, out2=out2, split=split, resid=resid, gate=gate, qk=qk,
                                             in_activation=in_activation, shared_gpu=shared_gpu))
        if y is not None:
            return y
    a = nv.LinearArgs()
    out, dev, M, N, K, _keep = _fill_args(a, x, w, b, activation, act_begin, out, out2, split, resid, gate, qk, in_activation, shared_gpu)
    with nv.on_device(dev):
        need = nv.lib().flux_linear_workspace_bytes(nv.byref(a)) if K > 3072 and _may_cut_k(M, N, K) else 0
        if need:   # K cut over several workgroups: partial sums in memory of this launch's stream
            ws = torch.empty((need,), dtype=torch.uint8, device=dev)
            rc = nv.lib().flux_linear_bf16_ws(nv.byref(a), ws.data_ptr(), need, nv.stream_ptr(dev))
        else:
            rc = nv.lib().flux_linear_bf16(nv.byref(a), nv.stream_ptr(dev))
    nv.check(rc, "flux_linear_bf16")
    return out


def linear_pair_into(first: dict, second: dict) -> tuple[Tensor, Tensor]:
    """Two linear_into calls (each the keyword arguments of one, `x`, `w` and `b` among them) in one library
    call: products of the same N, K and form of epilogue share a launch. An x of [B, L, K] may be a slice of
    a longer sequence, whose batch elements are not evenly strided rows."""
    if launch_hook is None and not is_compiling():
        both = nv.ops().linear_pair_into(positional(**first), positional(**second))
        if both is not None:
            return both
    args = nv.LinearPairArgs()
    outs, keep, sizes, notes = [], [], [], []
    for i, call in enumerate((first, second)):
        x = call["x"]
        if x.dim() == 3 and x.shape[0] > 1 and x.stride(0) != x.shape[1] * x.stride(1):
            B, L, K = x.shape
            if B * L > 8 and x.stride(2) == 1 and x.stride(1) >= K and x.stride(0) % 8 == 0 and x.stride(0) >= L * x.stride(1) \
                    and x.stride(1) % 8 == 0 and K % 8 == 0 and x.data_ptr() % 16 == 0 and call["w"].data_ptr() % 16 == 0 \
                    and call["w"].is_contiguous() and B * x.stride(0) * 2 < 2**31:
                args.a_rows[i], args.a_batch_stride[i] = L, x.stride(0)
        out, dev, M, N, K, kept = _fill_args(args.product[i], batches=bool(args.a_rows[i]), notes=notes, **call)
        outs.append(out)
        keep.append(kept)
        sizes.append((M, N, K))
    nv.require_gpu(*outs)
    with nv.on_device(dev):
        if launch_hook is None:
            _launch_pair(args, sizes, dev)
            return outs[0], outs[1]
        plan = nv.LinearPlan()
        nv.check(nv.lib().flux_linear_plan_of(nv.byref(args.product[0]), nv.byref(args.product[1]), 0, nv.byref(plan)), "flux_linear_plan_of")
        if plan.products == 2:
            launch_hook(_pair_launch_metadata(*notes, sizes))
            _launch_pair(args, sizes, dev)
            return outs[0], outs[1]
        for i in range(2):   # a launch each: each alone, beside a product without rows
            one = nv.LinearPairArgs()
            one.product[0], one.product[1] = args.product[i], args.product[i]
            one.product[1].M = 0
            one.a_rows[0], one.a_batch_stride[0] = args.a_rows[i], args.a_batch_stride[i]
            launch_hook(notes[i])
            _launch_pair(one, sizes[i:i + 1], dev)
    return outs[0], outs[1]


def rows_args(calls: tuple[dict, ...], dev: torch.device) -> tuple["nv.LinearPairArgs", list]:
    """One or two linear_into calls as the library takes them beside an attention, and what has to live until the launch."""
    args = nv.LinearPairArgs()
    keep, sizes, notes = [], [], []
    for i, call in enumerate(calls):
        out, at, M, N, _, kept = _fill_args(args.product[i], notes=notes, **call)
        assert at == dev, "tensors on different devices"
        keep += [out, kept]
        sizes.append((M, N))
    if len(calls) == 1:
        args.product[1] = args.product[0]
        args.product[1].M = 0
    if launch_hook is not None:
        if len(notes) == 2 and sizes[0] == sizes[1]:
            launch_hook(_pair_launch_metadata(*notes, sizes))
        else:
            for n in notes:
                launch_hook(n)
    return args, keep


def _launch_pair(args: "nv.LinearPairArgs", sizes: list, dev: torch.device) -> None:
    rows, N, K = sum(s[0] for s in sizes), min(s[1] for s in sizes), max(s[2] for s in sizes)
    need = nv.lib().flux_linear_pair_workspace_bytes(nv.byref(args)) if _may_cut_k(rows, N, K) else 0
    ws = torch.empty((need,), dtype=torch.uint8, device=dev) if need else None
    nv.check(nv.lib().flux_linear_bf16_pair(nv.byref(args), nv.ptr(ws), need, nv.stream_ptr(dev)), "flux_linear_bf16_pair")


def _fill_args(a: "nv.LinearArgs", x: Tensor, w: Tensor, b: Tensor | None, activation: str = "", act_begin: int = 0,
               out: Tensor | None = None, out2: Tensor | None = None, split: int | None = None, resid: Tensor | None = None,
               gate: Tensor | None = None, qk: dict | None = None, in_activation: str = "", shared_gpu: bool = False,
               batches: bool = False, notes: list | None = None):
    """Checks one call and writes it into `a`; returns the output, its device, M, N, K and what has to live until the launch.
    batches: x is [B, L, K] with evenly strided rows inside a batch element only. notes: receives the launch
    hook's metadata instead of the hook, for a caller that launches two products at once."""
    assert x.shape[-1] == w.shape[-1], "Incompatible dimensions"
    assert x.dtype == w.dtype, "Incompatible dtypes"
    _PLANS[x.dtype]  # KeyError for anything but bfloat16, as in the reference
    act = _ACTIVATIONS[activation]
    dev = nv.require_gpu(x, w, b, out, out2, resid, gate)
    N, K = w.shape
    x2 = x[0] if batches else _rows_2d(x, K)
    M = x.numel() // K if batches else x2.shape[0]
    if w.stride(1) != 1 or (N > 1 and w.stride(0) < K):
        w = w.contiguous()
    if b is not None:
        assert b.shape[-1] == N
        b = b.to(x.dtype).contiguous()
    a.A, a.W, a.bias = x2.data_ptr(), w.data_ptr(), nv.ptr(b)
    a.M, a.N, a.K = M, N, K
    a.lda = x2.stride(0) if M > 1 else K
    a.ldw = w.stride(0) if N > 1 else K
    if out is None:
        out = torch.empty((M, N if split is None else split), device=dev, dtype=x.dtype)
    else:
        assert out.dim() == 2 and out.shape[0] == M and out.stride(1) == 1 and out.dtype == x.dtype
    a.Y, a.ldy = out.data_ptr(), out.stride(0)
    if split is not None and split < N:
        assert out2 is not None and out2.dim() == 2 and out2.shape[0] == M and out2.stride(1) == 1
        assert out.shape[1] >= split and out2.shape[1] >= N - split and out2.dtype == x.dtype
        a.Y2, a.ldy2, a.split_n, a.y2_col0 = out2.data_ptr(), out2.stride(0), split, 0
    else:
        assert out.shape[1] >= N
        a.Y2, a.split_n = None, N
    keep = [x2, w, b]
    if gate is not None:
        assert resid is not None
        r2 = resid.reshape(-1, N)
        assert r2.shape[0] == M and r2.stride(1) == 1 and r2.dtype == x.dtype
        g2 = gate.reshape(-1, N) if gate.is_contiguous() else gate.reshape(gate.shape[0], N)
        if g2.dtype != x.dtype:
            g2 = g2.to(x.dtype)
        if g2.stride(1) != 1:
            g2 = g2.contiguous()
        nb = g2.shape[0]
        assert M % nb == 0
        keep += [r2, g2]
        a.resid, a.ldresid = r2.data_ptr(), r2.stride(0)
        a.gate, a.gate_batch_stride, a.rows_per_batch = g2.data_ptr(), (g2.stride(0) if nb > 1 else N), M // nb
    a.act, a.act_begin = act, act_begin
    a.flags = nv.LINEAR_SHARED_GPU if shared_gpu else 0
    a.in_act = _IN_ACTIVATIONS[in_activation]
    assert a.in_act == nv.ACT_NONE or M <= 8, "the input activation is fused for at most 8 rows"
    if qk is not None:
        f = nv.LinearQKFusion()
        q_out, k_out, pe = qk["q_out"], qk["k_out"], qk["pe"]
        heads, seq_len = int(qk["heads"]), int(qk["seq_len"])
        assert q_out.is_contiguous() and k_out.is_contiguous() and q_out.shape == k_out.shape and q_out.dtype == x.dtype
        assert q_out.dim() == 4 and q_out.shape[1] == heads and q_out.shape[3] == 128 and M % seq_len == 0 and q_out.shape[0] == M // seq_len
        out_len = q_out.shape[2]
        pe2 = pe.reshape(-1, out_len, 64, 2, 2)
        assert pe2.dtype == torch.float32 and pe2.is_contiguous()
        qs, ks = qk["q_scale"].to(x.dtype).contiguous(), qk["k_scale"].to(x.dtype).contiguous()
        f.q_out, f.k_out, f.q_scale, f.k_scale = q_out.data_ptr(), k_out.data_ptr(), qs.data_ptr(), ks.data_ptr()
        f.pe, f.pe_batch_stride = pe2.data_ptr(), (pe2.stride(0) if pe2.shape[0] > 1 else 0)
        f.heads, f.seq_len, f.out_len, f.pos0 = heads, seq_len, out_len, int(qk.get("pos0", 0))
        f.eps = float(qk.get("eps", 1e-6))
        a.qk = ctypes.pointer(f)
        keep += [f, qs, ks, pe2]
    if launch_hook is not None:
        parts = [activation and f"{activation}>={act_begin}", split is not None and f"split@{split}", gate is not None and "gated-residual",
                 qk is not None and "qk-norm-rope", in_activation and f"in:{in_activation}"]
        (launch_hook if notes is None else notes.append)(linear_launch_metadata(M, N, K, x.element_size(), "+".join(p for p in parts if p)))
    return out, dev, M, N, K, keep


def qk_fusable(x: Tensor, w: Tensor, seq_len: int, head_dim: int) -> bool:
    """Whether linear_into(..., qk=...) takes this projection and is worth it: bf16, heads of 128,
    columns in multiples of 256 (a wave's 128 columns are one head), sequences of at least 256 rows (a tile then holds
    rows of at most two batch elements; ragged row counts and sequence lengths are fine), and at least 160 outputs
    of 256 x 256, below which the preparation kernel behind a plain product is left alone."""
    M = x.numel() // x.shape[-1]
    N = w.shape[0]
    return (x.dtype == torch.bfloat16 and head_dim == 128 and seq_len >= 256 and M % seq_len == 0
            and N % 256 == 0 and w.shape[1] % 8 == 0 and -(-M // 256) * (N // 256) >= 160)


def qk_pays(rows: int, w: Tensor, heads: int) -> bool:
    """Whether a projection that qk_fusable() names is faster with the epilogue than with qkv_prep behind it: below two rounds of its tiles
    that depends on how the rows fall on the shapes that either way has."""
    return nv.lib().flux_linear_qk_pays(rows, w.shape[0], w.shape[1], heads) != 0


def linear(x: Tensor, w: Tensor, b: Tensor | None, activation: str = "", shared_gpu: bool = False) -> Tensor:
    act = _ACTIVATIONS.get(activation)
    if act is not None and launch_hook is None and not shared_gpu and not is_compiling():
        y = nv.ops().linear(x, w, b, act)
        if y is not None:
            return y
    N = w.shape[0]
    y = linear_into(x, w, b, activation=activation, shared_gpu=shared_gpu)
    return y.reshape(*x.shape[:-1], N)
