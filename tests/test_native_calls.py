"""The operators' calls in native code (csrc/torch_ops.cpp) against the Python launchers of the same operators, over the forms
they accept, and the calls that they leave to the launchers."""
import sys
import threading

import pytest
import torch
import torch.autograd.forward_ad as fwad

import triton_kernels as tk
from triton_kernels import _native as nv
from triton_kernels.kernels import normalization as norm_mod
from util import DEV, randn, seeded

gpu = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


class _Refuses:
    """Native calls that take nothing: every operator goes through its Python launcher."""

    def __getattr__(self, name):
        return lambda *args: None


def launcher(monkeypatch, fn, *args, **kw):
    with monkeypatch.context() as m:
        m.setattr(nv, "ops", lambda: _Refuses())
        return fn(*args, **kw)


def test_tensors_without_a_gpu_are_left_to_the_launchers():
    ops, x = nv.ops(), torch.ones(2, 2, 4, 8)
    assert ops.rms_norm(x, torch.ones(8), 1e-6) is None
    assert ops.rms_norm_pair(x, torch.ones(8), x, torch.ones(8), 1e-6) is None
    assert ops.layer_norm_modulation(x, x, x, 1e-5) is None
    assert ops.apply_rope(x, x, x) is None
    assert ops.linear(x.bfloat16(), torch.ones(8, 8, dtype=BF), None, 0) is None
    assert ops.attention(x.bfloat16(), x.bfloat16(), x.bfloat16(), None) is None
    for bad in (None, 3, "x", [x]):
        assert ops.rms_norm(bad, torch.ones(8), 1e-6) is None
    with pytest.raises(RuntimeError, match="GPU"):
        tk.rms_norm(x, torch.ones(8))


def _views(g, dtype):
    """Rows of one to 300 values in every order and stride that a norm reads in place, and those it copies or refuses."""
    base = randn(g, 3, 4, 5, 128, dtype=dtype).to(DEV)
    wide = randn(g, 2, 6, 3 * 256, dtype=dtype).to(DEV)
    return [base, base[0, 0, 0], base[1], base.permute(2, 0, 1, 3), base.transpose(1, 2)[::2], wide[..., 256:512], wide.view(2, 6, 3, 2, 128).permute(2, 0, 3, 1, 4)[1],
            base[..., :100], base[..., 1:129:1][..., :50], base[:, :, :1].expand(3, 4, 7, 128), base.flatten()[:7 * 300].view(7, 300), base.flatten()[3:3 + 5 * 33].view(5, 33),
            base[..., ::2], base.view(3, 2, 2, 5, 128), base[:0], base.flatten()[:9].view(9, 1)]


def test_the_extension_says_why_it_does_not_load(monkeypatch, tmp_path):
    """Not there, not loadable, built for another torch: three messages, and the library's own comes before them."""
    import triton_kernels
    monkeypatch.setattr(nv, "_ops", None)

    class _Broken:
        def find_spec(self, name, *args):
            if name == "triton_kernels._torch_ops":
                raise ImportError("undefined symbol: _ZN2at5emptyE")

    with monkeypatch.context() as m:
        m.setattr(nv, "_OPS_PATH", str(tmp_path / "_torch_ops.so"))
        with pytest.raises(RuntimeError, match="_torch_ops.so is not built"):
            nv.ops()
    with monkeypatch.context() as m:
        m.delitem(sys.modules, "triton_kernels._torch_ops", raising=False)
        m.delattr(triton_kernels, "_torch_ops", raising=False)
        m.setattr(sys, "meta_path", [_Broken(), *sys.meta_path])
        with pytest.raises(RuntimeError, match="undefined symbol.*make -B"):
            nv.ops()
    with monkeypatch.context() as m:
        m.setattr(nv, "_lib", None)
        m.setattr(nv, "ABI_VERSION", nv.ABI_VERSION + 1)
        with pytest.raises(RuntimeError, match="ABI version"):
            nv.ops()
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "1.0.0+other")
        with pytest.raises(RuntimeError, match=r"built for torch 2.*this is torch 1\.0\.0"):
            nv.ops()
    assert nv.ops().rms_norm(3, 3, 3) is None


@gpu
@pytest.mark.parametrize("dtype,scale_dtype", [(BF, BF), (BF, F32), (F32, F32), (F32, BF)])
def test_rms_norm_forms(monkeypatch, dtype, scale_dtype):
    g = seeded(1)
    for x in _views(g, dtype):
        for scale in (randn(g, x.shape[-1], dtype=scale_dtype).to(DEV), randn(g, 1, x.shape[-1], dtype=scale_dtype).to(DEV)):
            if x.numel():
                got = tk.rms_norm(x, scale)
                want = launcher(monkeypatch, tk.rms_norm, x, scale)
                assert torch.equal(got, want) and got.stride() == want.stride() and got.dtype == want.dtype
            xs = [x.detach().clone(memory_format=torch.preserve_format).requires_grad_(True) for _ in range(2)]
            ss = [scale.detach().clone().requires_grad_(True) for _ in range(2)]
            dy = randn(g, *x.shape, dtype=dtype).to(DEV)
            if not x.numel():
                continue
            ys = tk.rms_norm(xs[0], ss[0]), launcher(monkeypatch, tk.rms_norm, xs[1], ss[1])
            for y in ys:
                y.backward(dy)
            assert torch.equal(ys[0], ys[1]) and torch.equal(xs[0].grad, xs[1].grad) and xs[0].grad.stride() == xs[1].grad.stride()
            # (rows that are no 16-byte vectors add the scale's gradient with atomics, in any order)
            torch.testing.assert_close(ss[0].grad, ss[1].grad, atol=1e-5 if scale_dtype == F32 else 2e-2, rtol=1e-5 if scale_dtype == F32 else 2.0 ** -7)
            assert ss[0].grad.dtype == scale_dtype and ss[0].grad.shape == scale.shape


@gpu
def test_rms_norm_pair_and_layer_norm_forms(monkeypatch):
    g = seeded(2)
    for dtype in (BF, F32):
        views = [v for v in _views(g, dtype) if v.numel()]
        with torch.no_grad():
            for x0 in views:
                for x1 in views:
                    if x0.shape[-1] == x1.shape[-1]:
                        s = [randn(g, x0.shape[-1], dtype=dtype).to(DEV) for _ in range(2)]
                        got, want = norm_mod.rms_norm_pair(x0, s[0], x1, s[1]), launcher(monkeypatch, norm_mod.rms_norm_pair, x0, s[0], x1, s[1])
                        assert all(torch.equal(a, b) for a, b in zip(got, want))
        for x in views:
            if x.dim() < 2:
                continue
            B, N = x.shape[0], x.shape[-1]
            mod = randn(g, B, 1, 3 * N, dtype=dtype).to(DEV)
            for w, b in (mod.chunk(3, -1)[:2], (mod[..., :N].contiguous(), mod[..., N:2 * N]), (mod[:, 0, :N], mod[:, 0, N:2 * N]), (mod[..., ::3], mod[..., 1::3]),
                         (mod[:1, :, :N].expand(B, 1, N), mod[:1, :, N:2 * N].expand(B, 1, N)), (mod[..., :N].float(), mod[..., N:2 * N].float())):
                assert torch.equal(tk.layer_norm_modulation(x, w, b), launcher(monkeypatch, tk.layer_norm_modulation, x, w, b))


@gpu
def test_rope_linear_attention_forms(monkeypatch):
    g = seeded(3)
    for dtype in (BF, F32):
        for D in (128, 64, 16):
            qkv = randn(g, 2, 9, 3 * 4 * D, dtype=dtype).to(DEV).view(2, 9, 3, 4, D).permute(2, 0, 3, 1, 4)
            pes = [randn(g, *lead, 9, D // 2, 2, 2).to(DEV) for lead in ((1, 1), (), (2, 1), (1, 4), (1,))]
            for q, k in ((qkv[0], qkv[1]), (qkv[0].contiguous(), qkv[1].contiguous()), (qkv[0].transpose(2, 3).contiguous().transpose(2, 3), qkv[1])):
                for pe in pes + [pes[0].double(), pes[0].transpose(-1, -2)]:
                    got, want = tk.apply_rope(q, k, pe), launcher(monkeypatch, tk.apply_rope, q, k, pe)
                    assert all(torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(got, want))
    for M, N, K in ((1, 64, 64), (8, 40, 72), (9, 40, 72), (300, 136, 3080), (64, 33, 50), (256, 256, 3136)):
        x, w, b = randn(g, M, K, dtype=BF).to(DEV), randn(g, N, K, dtype=BF, std=K ** -0.5).to(DEV), randn(g, N, dtype=BF).to(DEV)
        half = randn(g, M, 2 * K, dtype=BF).to(DEV)[:, :K]
        for xx in (x, x.view(1, M, K), x.t().contiguous().t(), half, x[0]):
            for ww in (w, randn(g, K, N, dtype=BF).to(DEV).t()):
                for bb in (b, None, b.float(), b.view(1, N)):
                    for act in ("", "GELU"):
                        got, want = tk.linear(xx, ww, bb, activation=act), launcher(monkeypatch, tk.linear, xx, ww, bb, activation=act)
                        assert torch.equal(got, want) and got.shape == want.shape and got.stride() == want.stride()
    for B, H, L, D in ((1, 2, 1, 64), (2, 3, 77, 128), (1, 2, 1500, 64), (1, 2, 40, 32), (4, 24, 300, 128)):
        qkv = randn(g, B, L, 3, H, D, dtype=BF).to(DEV).permute(2, 0, 3, 1, 4)
        for q, k, v in (qkv.unbind(0), [t.contiguous() for t in qkv], (qkv[0], qkv[1].transpose(2, 3).contiguous().transpose(2, 3), qkv[2])):
            for scale in (None, 0.3, 0.0, torch.tensor(0.2)):
                got, want = tk.scaled_dot_product_attention(q, k, v, scale), launcher(monkeypatch, tk.scaled_dot_product_attention, q, k, v, scale)
                assert torch.equal(got, want) and got.stride() == want.stride()


class _Records:
    """The native calls, and for each one made whether it served the call."""

    def __init__(self):
        self.ops, self.served = nv.ops(), []

    def __getattr__(self, name):
        def call(*args):
            y = getattr(self.ops, name)(*args)
            self.served.append((name, y is not None))
            return y
        return call


@gpu
def test_which_calls_are_served_in_native_code(monkeypatch):
    """The forms that programs use are served by the native call itself, with the launcher's bits; the listed others are not."""
    g = seeded(11)

    def check(op, expected, fn, *args, **kw):
        records = _Records()
        with monkeypatch.context() as m:
            m.setattr(nv, "ops", lambda: records)
            got = fn(*args, **kw)
        assert (op, True) in records.served if expected else (op, True) not in records.served, (op, records.served, [getattr(a, "shape", a) for a in args])
        want = launcher(monkeypatch, fn, *args, **kw)
        for a, b in zip(got, want) if isinstance(got, tuple) else [(got, want)]:
            assert torch.equal(a, b) and a.stride() == b.stride() and a.dtype == b.dtype

    def t(*shape, dtype=BF, std=1.0):
        return randn(g, *shape, dtype=dtype, std=std).to(DEV)

    for dtype, scale_dtype in ((BF, BF), (BF, F32), (F32, F32), (F32, BF)):
        for x in _views(g, dtype):
            if x.numel():
                scale, taken = t(x.shape[-1], dtype=scale_dtype), (dtype, scale_dtype) != (F32, BF) and x.stride(-1) == 1 and x.dim() <= 4
                check("rms_norm", taken, tk.rms_norm, x, scale)
                check("rms_norm", taken, tk.rms_norm, x.detach().requires_grad_(True), scale)
                check("rms_norm", False, tk.rms_norm, x, scale[None])
    for dtype in (BF, F32):
        qkv = t(2, 9, 3 * 4 * 128, dtype=dtype).view(2, 9, 3, 4, 128).permute(2, 0, 3, 1, 4)
        s = t(128, dtype=dtype)
        with torch.no_grad():
            check("rms_norm_pair", True, norm_mod.rms_norm_pair, qkv[0], s, qkv[1], s)
            check("rms_norm_pair", False, norm_mod.rms_norm_pair, qkv[0][..., 1:], s[1:], qkv[1][..., 1:], s[1:])
        check("rms_norm_pair", False, norm_mod.rms_norm_pair, qkv[0], s, qkv[1], s)
        pe = t(1, 1, 9, 64, 2, 2, dtype=F32)
        check("apply_rope", True, tk.apply_rope, qkv[0], qkv[1], pe)
        check("apply_rope", True, tk.apply_rope, qkv[0].contiguous(), qkv[1].contiguous(), pe.expand(2, 1, 9, 64, 2, 2).contiguous())
        check("apply_rope", False, tk.apply_rope, qkv[0], qkv[1], pe.double())
        x, mod = t(2, 7, 256, dtype=dtype), t(2, 1, 3 * 256, dtype=dtype)
        check("layer_norm_modulation", True, tk.layer_norm_modulation, x, *mod.chunk(3, -1)[:2])
        check("layer_norm_modulation", True, tk.layer_norm_modulation, x, mod[:, 0, :256].contiguous(), mod[:, 0, 256:512].contiguous())
        check("layer_norm_modulation", True, tk.layer_norm_modulation, x[:1], mod[:1, :, :256], mod[:1, :, 256:512])
        check("layer_norm_modulation", False, tk.layer_norm_modulation, x, mod[..., ::3], mod[..., 1::3])
        check("layer_norm_modulation", False, tk.layer_norm_modulation, x.transpose(0, 1).contiguous().transpose(0, 1), *mod.chunk(3, -1)[:2])
    for M, N, K in ((1, 64, 64), (8, 40, 72), (300, 136, 3080), (320, 3072, 15360)):
        x, w, b = t(M, K), t(N, K, std=K ** -0.5), t(N)
        for act in ("", "GELU"):
            check("linear", True, tk.linear, x, w, b, activation=act)
            check("linear", True, tk.linear, x.view(1, M, K), w, None, activation=act)
        check("linear", False, tk.linear, x, w, b.float())
        check("linear", False, tk.linear, x, t(K, N, std=K ** -0.5).t(), b)
        check("linear", False, tk.linear, x, w, b, shared_gpu=True)
        with monkeypatch.context() as m:
            m.setattr(sys.modules["triton_kernels.kernels.linear"], "launch_hook", lambda meta: None)
            check("linear", False, tk.linear, x, w, b)
    for B, H, L, D in ((1, 2, 1, 64), (2, 3, 77, 128), (1, 2, 2048, 128), (1, 2, 40, 32)):
        qkv = t(B, L, 3, H, D).permute(2, 0, 3, 1, 4)
        check("attention", True, tk.scaled_dot_product_attention, *qkv.unbind(0))
        check("attention", True, tk.scaled_dot_product_attention, *(v.contiguous() for v in qkv), 0.3)
        check("attention", L == 1, tk.scaled_dot_product_attention, qkv[0], qkv[1].transpose(2, 3).contiguous().transpose(2, 3), qkv[2])
    assert nv.lib().flux_attention_workspace_bytes(1, 2, 2048, 128) > 0   # (of the calls above: keys in parts, K in parts)
    a = nv.LinearArgs()
    a.A = a.W = a.Y = 1 << 20
    a.M, a.N, a.K, a.lda, a.ldw, a.ldy, a.split_n = 320, 3072, 15360, 15360, 15360, 3072, 3072
    assert nv.lib().flux_linear_workspace_bytes(nv.byref(a)) > 0


def _served(monkeypatch, name, served, fn):
    """fn() by the native call `name` (or, where served is False, by the launcher behind it) and by the launcher, whose bits it has to have."""
    answers, real = [], getattr(nv.ops(), name)

    class Spy:
        def __getattr__(self, other):
            return getattr(nv_ops, other) if other != name else lambda *a: answers.append(real(*a)) or answers[-1]

    nv_ops = nv.ops()
    with monkeypatch.context() as m:
        m.setattr(nv, "ops", lambda: Spy())
        got = fn()
    assert answers and (answers[0] is not None) == served
    want = launcher(monkeypatch, fn)
    for a, b in zip(got, want):
        assert (a is None and b is None) or (torch.equal(a, b) and a.stride() == b.stride())


@gpu
def test_calls_of_the_blocks_forms(monkeypatch):
    """The general linear, two of them, the norm pair, the q/k/v preparation and attention to a given tensor: rows and batches in
    every order that is read in place, the ones that are copied or refused, each against its launcher bit for bit."""
    from triton_kernels.kernels.attention import attention_into
    from triton_kernels.kernels.linear import linear_into, linear_pair_into
    from triton_kernels.kernels.positional_embedding import qkv_prep
    g = seeded(11)
    t = lambda *s, std=1.0, dtype=BF: (randn(g, *s) * std).to(dtype).to(DEV)
    K, N = 72, 136
    w, b, wide = t(N, K, std=K ** -0.5), t(N), t(2, 40, 2 * K)
    into = lambda **kw: lambda: (linear_into(**kw),)
    for x, served in ((wide[..., :K].contiguous(), True), (wide[..., :K], True), (wide[0, :, :K], True), (wide[:, 3, :K], True), (wide[:, 4:20, :K], False), (wide[..., ::2], False),
                      (wide[:1, :1, :K], True), (wide[..., :K].transpose(0, 1), False)):
        M = x.numel() // K
        _served(monkeypatch, "linear_into", served, into(x=x, w=w, b=b, activation="GELU", act_begin=64))
        gate, resid = t(1, 1, 3 * N)[..., N:2 * N], t(M, N)
        _served(monkeypatch, "linear_into", served, into(x=x, w=w, b=None, resid=resid, gate=gate))
        _served(monkeypatch, "linear_into", served, into(x=x, w=t(N, 2 * K)[:, :K], b=b, resid=resid.view(1, M, N), gate=gate.contiguous()))

        def split():
            a, c = torch.zeros(M, 64, device=DEV, dtype=BF), torch.zeros(M, N, device=DEV, dtype=BF)
            return linear_into(x, w, b, out=a, out2=c[:, 8:], split=64), c

        _served(monkeypatch, "linear_into", served, split)
    x, few = wide[0, :, :K], t(2, K)
    for kw, served in ((dict(x=few, in_activation="SiLU"), True), (dict(x=x, shared_gpu=True), False), (dict(x=x, b=b.float()), False), (dict(x=x, w=w.t().contiguous().t()), False), (dict(x=x, split=N), True)):
        _served(monkeypatch, "linear_into", served, into(**{"w": w, "b": b, **kw}))
    _served(monkeypatch, "linear_into", False, lambda: (linear_into(x, w, b, split=N + 8)[:, :N],))   # (its last eight columns are nobody's)
    gates = t(2, 1, 3 * N)[..., :N]
    for first, second, served in ((wide[:, :30, :K], wide[:, 30:, :K], True), (wide[:1, :30, :K], wide[:1, 30:, :K], True), (few[:1], few[1:], True), (wide[..., ::2], x, False)):
        calls = [dict(x=v, w=w, b=b) for v in (first, second)]
        _served(monkeypatch, "linear_pair_into", served, lambda: linear_pair_into(*calls))
        rows = [v.numel() // K for v in (first, second)]
        if first.dim() == 3 and served:
            gated = [dict(c, resid=t(n, N), gate=gates[:v.shape[0]]) for c, n, v in zip(calls, rows, (first, second))]
            _served(monkeypatch, "linear_pair_into", True, lambda: linear_pair_into(*gated))
    heads, L = 2, 300
    hid = heads * 128
    x, w1, b1, pe = t(2 * L, hid), t(40 * 256, hid, std=hid ** -0.5), t(40 * 256), t(1, 1, L, 64, 2, 2, dtype=F32)
    scales = t(128).abs() + 0.5, t(128).abs() + 0.5
    for table, served in ((pe, True), (t(2, 1, L, 64, 2, 2, dtype=F32), True)):
        def fused():
            q, k = (torch.zeros(2, heads, L, 128, device=DEV, dtype=BF) for _ in range(2))
            qk = dict(q_out=q, k_out=k, q_scale=scales[0], k_scale=scales[1], pe=table, heads=heads, seq_len=L)
            return linear_into(x, w1, b1, activation="GELU", act_begin=2 * hid, out=torch.zeros(2 * L, 40 * 256, device=DEV, dtype=BF), qk=qk), q, k
        _served(monkeypatch, "linear_into", served, fused)
    for dtype in (BF, F32):
        img, txt = (t(2, n, 3 * hid, dtype=dtype).view(2, n, 3, heads, 128).permute(2, 0, 3, 1, 4) for n in (9, 4))
        s, pe = t(128, dtype=dtype), t(1, 1, 13, 64, 2, 2, dtype=F32)
        for args, kw, served in (((*img, *txt), dict(pe=pe, q_scale_img=s, k_scale_img=s, q_scale_txt=s, k_scale_txt=s), True), ((*img, *txt), {}, True), ((img[0], img[1], None), dict(pe=pe[:, :, :9].double()), False),
                                 ((img[0], img[1], None), dict(pe=pe[:, :, :9].contiguous(), q_scale_img=s, k_scale_img=s), True), ((None, img[1], img[2]), {}, False), ((*img, txt[0], txt[1], txt[2].transpose(0, 1).contiguous().transpose(0, 1)), {}, True),
                                 ((img[0], img[1], None, txt[0], txt[1], None), dict(pe=pe, q_scale_img=s, k_scale_img=s, q_scale_txt=s, k_scale_txt=s), True), ((img[0], img[1], None, txt[0], txt[1], None), {}, True),
                                 ((*(v[..., ::2] for v in img),), {}, False)):
            _served(monkeypatch, "qkv_prep", served, lambda: qkv_prep(*args, **kw))
        mod = t(2, 1, 6 * 256, dtype=dtype).chunk(6, -1)
        a, c = t(2, 7, 256, dtype=dtype), t(2, 3, 256, dtype=dtype)
        for first, second, served in (((a, mod[0], mod[1]), (c, mod[3], mod[4]), True), ((a[:, :5], mod[0], mod[1]), (c, mod[3], mod[4]), False), ((a, mod[0].float(), mod[1]), (c, mod[3], mod[4]), dtype == F32)):
            _served(monkeypatch, "layer_norm_modulation_pair", served, lambda: norm_mod.layer_norm_modulation_pair(first, second))
    qkv = t(2, 150, 3, heads, 128).permute(2, 0, 3, 1, 4)
    for kw, q, served in (({}, qkv[0], True), (dict(sm_scale=0.3), qkv[0].contiguous(), True), ({}, qkv[0].transpose(2, 3).contiguous().transpose(2, 3), False)):
        _served(monkeypatch, "attention", served, lambda: (attention_into(q, qkv[1], qkv[2], torch.zeros(2, 150, heads, 136, device=DEV, dtype=BF).permute(0, 2, 1, 3)[..., :128], **kw),))


@gpu
@pytest.mark.parametrize("kind,batch,tokens", [("single", 1, 96), ("single", 2, 300), ("double", 1, 96), ("double", 2, 96), ("double", 1, 1100), ("double", 5, 40)])
def test_a_pass_of_a_fused_block_stays_in_native_code(monkeypatch, kind, batch, tokens):
    """Every call that a fused block makes is served, with a modulation beside the attention or in front, one batch element or several."""
    g, heads, hid, calls, native = seeded(batch + tokens), 4, 512, [], nv.ops()
    blk = (tk.SingleStreamBlock(hid, heads) if kind == "single" else tk.DoubleStreamBlock(hid, heads, mlp_ratio=4.0, qkv_bias=True)).to(BF).to(DEV)
    xs = [randn(g, batch, n, hid, dtype=BF).to(DEV) for n in ((tokens,) if kind == "single" else (tokens, 7))]
    vec, pe = randn(g, batch, hid, dtype=BF).to(DEV), randn(g, 1, 1, sum(x.shape[1] for x in xs), 64, 2, 2).to(DEV)

    class Spy:
        def __getattr__(self, name):
            return lambda *a: calls.append((name, getattr(native, name)(*a))) or calls[-1][1]

    with torch.no_grad():
        want = launcher(monkeypatch, blk, *xs, vec, pe)
        with monkeypatch.context() as m:
            m.setattr(nv, "ops", lambda: Spy())
            got = blk(*xs, vec, pe)
    assert [name for name, out in calls if out is None] == []
    assert len(calls) == (6 if kind == "single" else 9)
    for a, b in zip((got,) if kind == "single" else got, (want,) if kind == "single" else want):
        assert torch.equal(a, b)


@gpu
def test_refusals_stay_what_they_were(monkeypatch):
    x, w = torch.ones(4, 64, device=DEV, dtype=BF), torch.ones(32, 64, device=DEV, dtype=BF)
    h = x.view(1, 1, 4, 64)
    calls = [(tk.rms_norm, x, torch.ones(32, device=DEV, dtype=BF)), (tk.rms_norm, torch.ones(1, 70000, device=DEV), torch.ones(70000, device=DEV)),
             (tk.rms_norm, x.half(), w[0].half()), (tk.rms_norm, x, w[0].cpu()), (tk.linear, x, w[:, :32], None), (tk.linear, x.float(), w, None), (tk.linear, x.float(), w.float(), None),
             (tk.linear, x, w, None, "RELU"), (tk.linear, x, w, torch.ones(7, device=DEV, dtype=BF)), (tk.scaled_dot_product_attention, h, h, h.float()),
             (tk.scaled_dot_product_attention, h, h, h, float("nan")), (tk.scaled_dot_product_attention, h[..., :24], h[..., :24], h[..., :24]),
             (tk.scaled_dot_product_attention, h, h, h[:, :, :2]), (tk.apply_rope, h, h, torch.ones(1, 1, 5, 32, 2, 2, device=DEV)), (tk.apply_rope, h, h.float(), h), (tk.apply_rope, h[..., :24], h[..., :24], torch.ones(1, 1, 4, 12, 2, 2, device=DEV)),
             (tk.layer_norm_modulation, h, h[:, :, 0], h[:, :, :1, :32]), (tk.layer_norm_modulation, x, x[:2], x),
             (norm_mod.layer_norm_modulation_pair, (h, h[:, :, 0]), (h, h[:, :, 0], h[:, :, 0])), (norm_mod.layer_norm_modulation_pair, (h, h[:, :, 0]), (h[:, :, 0], h, h[:, :, 0], h[:, :, 0]))]
    for fn, *args in calls:
        errors = []
        for call in (lambda: fn(*args), lambda: launcher(monkeypatch, fn, *args)):
            with pytest.raises(Exception) as e:
                call()
            errors.append(e)
        assert errors[0].type is errors[1].type and str(errors[0].value) == str(errors[1].value)


@gpu
def test_transforms_tracing_and_forward_mode_see_the_launchers():
    ops, g = nv.ops(), seeded(4)
    x, s = randn(g, 3, 64).to(DEV), randn(g, 64).to(DEV)
    assert ops.rms_norm(x, s, 1e-6) is not None
    for transform in (torch.func.vmap, lambda f: torch.func.grad(lambda t: f(t).sum())):
        with pytest.raises(RuntimeError):
            transform(lambda t: tk.rms_norm(t, s))(x)
    with fwad.dual_level():
        assert ops.rms_norm(x, s, 1e-6) is None
        with pytest.raises((RuntimeError, NotImplementedError)):
            tk.rms_norm(fwad.make_dual(x, torch.ones_like(x)), s)
        with torch.no_grad(), pytest.raises((RuntimeError, NotImplementedError)):
            norm_mod.rms_norm_pair(fwad.make_dual(x, torch.ones_like(x)), s, x, s)
    seen = []

    def traced(t):
        seen.append(ops.rms_norm(t, s, 1e-6))
        return t + 1

    torch.jit.trace(traced, x, check_trace=False)
    assert seen == [None]

    class Sub(torch.Tensor):
        pass

    assert ops.rms_norm(x.as_subclass(Sub), s, 1e-6) is None
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert ops.rms_norm(x, s, 1e-6) is None
    with torch.inference_mode():
        assert torch.equal(tk.rms_norm(x, s), norm_mod.rms_norm_forward(x, s)[0])


@gpu
def test_rms_norm_graph_behaves_like_the_function():
    g = seeded(5)
    x, s = randn(g, 8, 128, dtype=BF).to(DEV).requires_grad_(True), randn(g, 128, dtype=BF).to(DEV).requires_grad_(True)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(DEV)):
        y = tk.rms_norm(x, s)
    assert packed == [(8, 128), (128,), (8,)]
    plain = tk.rms_norm(x, s)
    dy = torch.ones_like(y)
    for a, b in zip(torch.autograd.grad(y, (x, s), dy), torch.autograd.grad(plain, (x, s), dy, retain_graph=True)):
        assert torch.equal(a, b)
    assert torch.autograd.grad(plain, x, dy, retain_graph=True)[0].shape == x.shape
    assert torch.equal(torch.autograd.grad(plain, s, torch.ones(1, 1, device=DEV, dtype=BF).expand(8, 128), retain_graph=True)[0], torch.autograd.grad(plain, s, dy, retain_graph=True)[0])
    dx = torch.autograd.grad(plain, x, dy, create_graph=True)[0]
    assert not dx.requires_grad
    torch.autograd.grad(plain, x, dy)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(plain, x, dy)
    y = tk.rms_norm(x, s)
    with torch.no_grad():
        s.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(y, x, dy)


@gpu
def test_streams_and_threads():
    """Every thread trains on a stream of its own: launches, allocations and the backward follow the stream."""
    g = seeded(6)
    x0, s0 = randn(g, 4096, 128).to(DEV), randn(g, 128).to(DEV)
    want_y = norm_mod.rms_norm_forward(x0, s0)[0]
    torch.cuda.synchronize()
    bad = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                x = torch.zeros_like(x0)
                torch.cuda._sleep(200000)
                x.add_(x0).requires_grad_(True)            # late on this stream: a launch on another one would read zeros
                y = tk.rms_norm(x, s0)
                (dx,) = torch.autograd.grad(y, x, y.detach())
                ok = torch.equal(y, want_y) & torch.isfinite(dx).all()
                if not bool(ok):
                    bad.append(1)
        stream.synchronize()

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@gpu
@pytest.mark.parametrize("grad", [False, True])
def test_refusals_of_the_library_keep_their_kind(monkeypatch, grad):
    """Tensors whose memory has been given back are refused by the library (null pointers): the norm's native calls raise
    what the launchers raise."""
    x, s = torch.ones(4, 64, device=DEV), torch.ones(64, device=DEV)
    gone, s_gone = torch.ones(4, 64, device=DEV), torch.ones(64, device=DEV)
    for t in (gone, s_gone):
        t.untyped_storage().resize_(0)
        t.requires_grad_(grad)
    for fn, *args in ((tk.rms_norm, gone, s), (tk.rms_norm, x, s_gone), (norm_mod.rms_norm_pair, gone, s, x, s), (norm_mod.rms_norm_pair, x, s, x, s_gone)):
        with torch.set_grad_enabled(grad):
            errors = []
            for call in (lambda: fn(*args), lambda: launcher(monkeypatch, fn, *args)):
                with pytest.raises(Exception) as e:
                    call()
                errors.append(e)
        assert errors[0].type is errors[1].type is ValueError and str(errors[0].value) == str(errors[1].value)


@gpu
def test_numbers_that_float_takes(monkeypatch):
    """eps and the attention's scale may be anything that float() makes a number of, texts among them."""
    g = seeded(7)
    x, s = randn(g, 2, 4, 6, 64, dtype=BF).to(DEV), randn(g, 64, dtype=BF).to(DEV)
    mod = randn(g, 2, 1, 64, dtype=BF).to(DEV)
    with torch.no_grad():
        for fn, args in ((tk.rms_norm, (x, s)), (norm_mod.rms_norm_pair, (x, s, x, s)), (tk.layer_norm_modulation, (x, mod, mod)), (tk.scaled_dot_product_attention, (x, x, x))):
            for number in ("1e-3", b"0.25", torch.tensor(0.5), 1, True):
                got, want = fn(*args, number), launcher(monkeypatch, fn, *args, number)
                pairs = zip(got, want) if isinstance(got, tuple) else [(got, want)]
                assert all(torch.equal(a, b) for a, b in pairs)
            for bad in ("x", [], object()):
                errors = []
                for call in (lambda: fn(*args, bad), lambda: launcher(monkeypatch, fn, *args, bad)):
                    with pytest.raises((TypeError, ValueError)) as e:
                        call()
                    errors.append(e)
                assert errors[0].type is errors[1].type and str(errors[0].value) == str(errors[1].value)


@gpu
@pytest.mark.parametrize("dtype,scale_dtype", [(BF, BF), (BF, F32), (F32, F32)])
@pytest.mark.parametrize("kept", [torch.float32, torch.float64])
@pytest.mark.parametrize("scale_too", [False, True])
def test_saved_tensors_of_another_type(monkeypatch, dtype, scale_dtype, kept, scale_too):
    """What a saved-tensor hook hands back may have another type than what was saved: the launcher's backward converts the
    scale to what the kernels take beside x, and refuses an x they do not take; so does the native one."""
    g = seeded(8)
    x0, s0, dy = randn(g, 40, 96, dtype=dtype).to(DEV), randn(g, 96, dtype=scale_dtype).to(DEV), randn(g, 40, 96, dtype=dtype).to(DEV)
    got = []
    for call in (tk.rms_norm, lambda *a: launcher(monkeypatch, tk.rms_norm, *a)):
        x, s = x0.clone().requires_grad_(True), s0.clone().requires_grad_(True)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.to(kept) if t.dim() == 2 or scale_too and t.numel() == 96 else t):
            y = call(x, s)
        if kept == torch.float64:
            with pytest.raises(TypeError):
                y.backward(dy)
            continue
        y.backward(dy)
        got.append((x.grad, s.grad))
    if got:
        assert torch.equal(got[0][0], got[1][0]) and got[0][0].dtype == dtype and got[0][1].dtype == scale_dtype
        torch.testing.assert_close(got[0][1], got[1][1], atol=2e-2, rtol=2.0 ** -7)


@gpu
@pytest.mark.parametrize("native", [True, False])
def test_saved_row_norms_of_another_type(monkeypatch, native):
    """The kernel reads one fp32 value a row of what the forward kept; a hook that halves everything it keeps gets the
    gradients of the halved input, and values that came back too few or on the CPU are refused."""
    g = seeded(10)
    x0, s0, dy = randn(g, 40, 96).to(DEV), randn(g, 96).to(DEV), randn(g, 40, 96).to(DEV)

    def step(unpack):
        x, s = x0.clone().requires_grad_(True), s0.clone().requires_grad_(True)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            y = tk.rms_norm(x, s) if native else launcher(monkeypatch, tk.rms_norm, x, s)
        y.backward(dy)
        return x.grad, s.grad

    dx, ds = step(lambda t: t.bfloat16())
    rx, rs = step(lambda t: t)
    # (three roundings to bf16 of half an ulp, 2^-9 of the value, and the gradient's own)
    assert (dx - rx).norm() <= 2.0 ** -6 * rx.norm() and (ds - rs).norm() <= 2.0 ** -6 * rs.norm() and dx.dtype == ds.dtype == F32
    for bad in (lambda t: t[:20] if t.numel() == 40 else t, lambda t: t[:50] if t.numel() == 96 else t, lambda t: t.cpu() if t.dim() == 1 else t):
        with pytest.raises(RuntimeError):
            step(bad)


@gpu
def test_layer_norm_output_is_laid_out_like_its_input(monkeypatch):
    """A dimension of one element may have any stride in a contiguous input; the output has the same."""
    g = seeded(9)
    x, mod = randn(g, 1, 5, 64).to(DEV)[:, :1], randn(g, 1, 1, 64).to(DEV)
    assert x.is_contiguous() and x.stride(0) == 320
    got, want = tk.layer_norm_modulation(x, mod, mod), launcher(monkeypatch, tk.layer_norm_modulation, x, mod, mod)
    assert torch.equal(got, want) and got.stride() == want.stride()


@gpu
def test_the_norms_node_under_hooks_and_a_compiled_backward():
    """The native backward is a C++ node of the graph: hooks, edges and the engine's compiled mode treat it like any other,
    with the same gradients."""
    from torch._dynamo import compiled_autograd
    g = seeded(12)
    x0, s0, dy = randn(g, 40, 96, dtype=BF).to(DEV), randn(g, 96, dtype=BF).to(DEV), randn(g, 40, 96, dtype=BF).to(DEV)
    got = []
    for compiled in (False, True):
        x, s = x0.clone().requires_grad_(True), s0.clone().requires_grad_(True)
        y = tk.rms_norm(x * 2, s)
        assert [e[0].name() for e in y.grad_fn.next_functions[:2]] == ["MulBackward0", "torch::autograd::AccumulateGrad"]
        seen = []
        y.grad_fn.register_hook(lambda grads_in, grads_out: seen.append((grads_in[0].shape, grads_in[1].shape, grads_out[0].shape)))
        if compiled:
            with compiled_autograd._enable(torch.compile(backend="eager")):
                y.backward(dy)
        else:
            y.backward(dy)
        assert seen == [((40, 96), (96,), (40, 96))]
        got.append((x.grad, s.grad))
    assert all(torch.equal(a, b) for a, b in zip(*got))
