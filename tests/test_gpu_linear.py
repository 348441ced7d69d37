"""HIP linear (bf16 MFMA GEMM with fused epilogues) vs the oracle.

Grid and tolerances of the reference's tests/test_linear.py (bf16; atol 1e-5 without activation is
not attainable against a *different* bf16 GEMM on inputs ~N(0,1) with K up to 1024, where one bf16
ulp of the output is 0.25, so the no-activation cases compare against the fp32 result with the
half-ulp bound instead), plus the Flux shapes at atol 2e-2 vs fp32, ragged shapes, and every
epilogue the fused blocks use.
"""
import math

import pytest
import torch

import triton_kernels as tk
from oracle import flux_oracle as oracle
from triton_kernels import testing as cfg
from test_linear_plan import EIGHT_WAVES, PTR, RECT, SQUARE, linear_args, plan_of, qk_args
from triton_kernels import _native as nv
from triton_kernels.kernels import qk_fusable
from triton_kernels.kernels.linear import linear_pair_into
from util import DEV, randn, seeded

pytestmark = pytest.mark.gpu


def half_ulp_bound(ref_fp32: torch.Tensor) -> torch.Tensor:
    """One correct rounding to bf16 is off by at most half an ulp <= 2^-8 |x|. On top of that the
    fp32 sum itself depends on the order of accumulation: an absolute term for results that cancel
    to nearly zero and 1% slack for results that sit on a rounding boundary."""
    return ref_fp32.abs() * (2.0 ** -8 * 1.01) + 2e-3


@pytest.mark.parametrize("batch_size", [1, 4])
@pytest.mark.parametrize("seq_len", [256, 1024])
@pytest.mark.parametrize("in_channel", [256, 1024])
@pytest.mark.parametrize("out_channel", [1024, 3072])
@pytest.mark.parametrize("activation", ["", "GELU"])
def test_linear_reference_grid(batch_size, seq_len, in_channel, out_channel, activation):
    g = seeded(batch_size + seq_len + in_channel + out_channel)
    x = randn(g, batch_size, seq_len, in_channel, dtype=torch.bfloat16).to(DEV)
    w = randn(g, out_channel, in_channel, dtype=torch.bfloat16).to(DEV)
    b = randn(g, out_channel, dtype=torch.bfloat16).to(DEV)
    y = tk.linear(x, w, b, activation=activation)
    assert y.shape == (batch_size, seq_len, out_channel) and y.dtype == torch.bfloat16
    ref32 = oracle.linear_ref_fp32(x, w, b, activation)
    assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()
    if activation == "GELU":
        # the reference's own comparison (tests/test_linear.py:21-27: bf16 F.linear then F.gelu, atol 0.02);
        # that oracle rounds twice, so where |y| is large it may sit one bf16 ulp away
        ref = oracle.linear_ref(x, w, b, activation).float()
        assert ((y.float() - ref).abs() <= 0.02 + ref.abs() * 2.0 ** -7).all()


@pytest.mark.parametrize("which,act", [("mlp_in", "GELU"), ("proj_out", ""), ("linear1", "")])
def test_linear_flux_shapes_vs_fp32(which, act):
    """All three Flux GEMMs through the public operator at the full 4608 rows, plain epilogue (bias,
    optional GELU), against the fp32 product at the stated 2e-2 and at the half-ulp bound."""
    a, w, b = cfg.config4(DEV, which, m=4608)
    y = tk.linear(a, w, b, activation=act)
    ref32 = oracle.linear_ref_fp32(a, w, b, act)
    torch.testing.assert_close(y.float(), ref32, atol=2e-2, rtol=0)
    assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()


@pytest.mark.parametrize("M,N,K", [(1, 9216, 3072), (2, 1000, 512), (7, 33, 64), (8, 18432, 3072), (9, 40, 72),
                                   (130, 70, 200), (257, 513, 136), (300, 256, 8), (64, 64, 1000), (513, 1025, 264)])
@pytest.mark.parametrize("bias", [True, False])
def test_linear_ragged_shapes(M, N, K, bias):
    g = seeded(M * 3 + N * 5 + K)
    x = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16).to(DEV) if bias else None
    y = tk.linear(x, w, b)
    ref32 = oracle.linear_ref_fp32(x, w, b)
    assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()


@pytest.mark.parametrize("B,L,N,K,act,bias,gated", [
    (1, 4608, 3072, 512, "", True, True),       # linear2's output shape: 256 tiles of 288 x 192, gated residual
    (2, 1152, 6144, 200, "", False, True),      # K tail, two batch elements of four tile rows each, no bias
    (1, 2304, 6144, 136, "GELU", True, False),  # GELU on every column
    (1, 2304, 6144, 64, "", True, False),       # a single slab
    (1, 4608, 3072, 8, "", True, False),        # less than a slab
    (1, 4096, 3072, 512, "", True, True),       # the double block's img tails: 256 tiles of 256 x 192, gated residual
    (2, 2048, 3072, 200, "", False, True),      # K tail, two batch elements of eight tile rows each, no bias
    (1, 2048, 6144, 136, "GELU", True, False),  # GELU on every column, 256 x 192
    (1, 4096, 9216, 64, "", True, False),       # the double block's img qkv shape: three exact rounds, a single slab
    (1, 4096, 3072, 8, "", True, False),        # less than a slab
    (1, 2816, 3072, 320, "GELU", True, False),  # too few square tiles, two rounds of 128-wide ones: 176 tiles of 256 x 192
])
def test_linear_rectangular_tiles(B, L, N, K, act, bias, gated):
    """Shapes that 288 x 192 or 256 x 192 tiles divide and that fill the 256 CUs better on them than on
    square ones take the rectangular-tile kernel: every epilogue it has, with and without a K tail."""
    g = seeded(B * L + N + K)
    M = B * L
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV) if bias else None
    ref32 = oracle.linear_ref_fp32(a, w, b, act)
    if not gated:
        y = tk.linear(a, w, b, activation=act)
        assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()
        return
    x = randn(g, B, L, N, dtype=torch.bfloat16).to(DEV)
    gate = randn(g, B, 1, N, dtype=torch.bfloat16).to(DEV)
    out = torch.empty_like(x)
    tk.linear_into(a, w, b, out=out.view(M, N), resid=x.view(M, N), gate=gate)
    gy = gate.float() * ref32.view(B, L, N)
    want32 = x.float() + gy
    bound = 2.0 ** -8 * 1.01 * (2 * gy.abs() + want32.abs()) + 2e-3
    assert ((out.float() - want32).abs() <= bound).all()
    # and exactly the two PyTorch ops on the kernel's own (once rounded) product
    y = tk.linear(a, w, b)
    assert torch.equal(out, oracle.gated_residual_ref(x, gate, y.view(B, L, N)))


@pytest.mark.parametrize("M,N,K", [(4096, 3072, 192), (4608, 3072, 200), (1124, 8792, 64)])
def test_linear_shared_gpu_flag_changes_the_schedule_only(M, N, K):
    """FLUX_LINEAR_SHARED_GPU keeps the square tiles where the library would otherwise fill the CUs
    exactly with rectangular ones; both orders of accumulation are the same, so are the bits."""
    assert plan_of(linear_args(M, N, K)).family == RECT and plan_of(linear_args(M, N, K, flags=1)).family == SQUARE
    g = seeded(M + K)
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
    y0 = tk.linear_into(a, w, b, activation="GELU")
    y1 = tk.linear_into(a, w, b, activation="GELU", shared_gpu=True)
    assert torch.equal(y0, y1)
    assert ((y1.float() - oracle.linear_ref_fp32(a, w, b, "GELU")).abs() <= half_ulp_bound(oracle.linear_ref_fp32(a, w, b, "GELU"))).all()


def test_linear_unaligned_k_and_strided_input():
    g = seeded(3)
    x = randn(g, 50, 77, dtype=torch.bfloat16).to(DEV)       # K = 77: no 16-byte rows
    w = randn(g, 30, 77, dtype=torch.bfloat16, std=0.1).to(DEV)
    y = tk.linear(x, w, None)
    torch.testing.assert_close(y.float(), oracle.linear_ref_fp32(x, w, None), atol=2e-2, rtol=1e-2)
    big = randn(g, 300, 1024, dtype=torch.bfloat16).to(DEV)
    xs = big[:, 256:768]                                      # row stride 1024, K = 512
    w = randn(g, 384, 512, dtype=torch.bfloat16, std=512 ** -0.5).to(DEV)
    torch.testing.assert_close(tk.linear(xs, w, None).float(), oracle.linear_ref_fp32(xs, w, None), atol=2e-2, rtol=0)


def test_linear_rejects_fp32_like_the_reference():
    x = torch.zeros(4, 8, device=DEV)
    with pytest.raises(KeyError):
        tk.linear(x, torch.zeros(16, 8, device=DEV), None)


@pytest.mark.parametrize("M,hid,mlp", [(512, 256, 1024), (300, 128, 512), (4608, 3072, 12288)])
def test_linear_split_gelu_epilogue(M, hid, mlp):
    """linear1 of the single block: columns [0, 3*hid) plain -> out, columns [3*hid, ..) GELU -> out2."""
    g = seeded(M + hid)
    x = randn(g, M, hid, dtype=torch.bfloat16).to(DEV)
    w = randn(g, 3 * hid + mlp, hid, dtype=torch.bfloat16, std=hid ** -0.5).to(DEV)
    b = randn(g, 3 * hid + mlp, dtype=torch.bfloat16, std=0.02).to(DEV)
    qkv = torch.empty(M, 3 * hid, dtype=torch.bfloat16, device=DEV)
    both = torch.zeros(M, hid + mlp, dtype=torch.bfloat16, device=DEV)
    tk.linear_into(x, w, b, activation="GELU", act_begin=3 * hid, out=qkv, out2=both[:, hid:], split=3 * hid)
    ref32 = oracle.linear_ref_fp32(x, w, b)
    torch.testing.assert_close(qkv.float(), ref32[:, :3 * hid], atol=2e-2, rtol=0)
    want_mlp = oracle.gelu_tanh_ref(ref32[:, 3 * hid:])
    torch.testing.assert_close(both[:, hid:].float(), want_mlp, atol=2e-2, rtol=0)
    assert (both[:, :hid] == 0).all()                        # the attention half is left alone


@pytest.mark.parametrize("B,L,hid,K", [(1, 512, 256, 1280), (2, 300, 128, 640), (1, 4608, 3072, 15360)])
def test_linear_gated_residual_epilogue(B, L, hid, K):
    g = seeded(B + L + hid)
    a = randn(g, B * L, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, hid, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, hid, dtype=torch.bfloat16, std=0.02).to(DEV)
    x = randn(g, B, L, hid, dtype=torch.bfloat16).to(DEV)
    mod = randn(g, B, 3 * hid, dtype=torch.bfloat16).to(DEV)
    gate = mod[:, None, :].chunk(3, dim=-1)[2]
    out = torch.empty_like(x)
    tk.linear_into(a, w, b, out=out.view(B * L, hid), resid=x.view(B * L, hid), gate=gate)
    y32 = oracle.linear_ref_fp32(a, w, b).view(B, L, hid)
    # the two-op oracle (x + gate * y, modules/blocks.py:123) on the rounded product: y may sit on the
    # other side of a bf16 rounding boundary than the kernel's, which |gate| then magnifies
    want = oracle.gated_residual_ref(x, gate, y32.to(torch.bfloat16))
    torch.testing.assert_close(out, want, atol=4e-2, rtol=1e-2)
    # element-wise bound against the unrounded fp32 value: the kernel rounds y, gate * y and the sum,
    # each by at most half an ulp (2^-8 relative) of its own magnitude
    gy = gate.float() * y32
    want32 = x.float() + gy
    bound = 2.0 ** -8 * 1.01 * (2 * gy.abs() + want32.abs()) + 2e-3
    err = (out.float() - want32).abs()
    assert (err <= bound).all(), f"max excess {(err - bound).max().item()}"
    assert err.mean().item() < 6e-3


@pytest.mark.parametrize("B,L,H,mlp,bias,per_batch_pe", [(2, 256, 3, 1152, True, False), (1, 512, 2, 256, False, False),
                                                         (2, 256, 2, 256, True, True), (1, 4608, 24, 12288, True, False),
                                                         # ragged: rows and sequence length no multiple of the tile, tiles that
                                                         # hold the end of one batch element and the start of the next
                                                         (3, 300, 2, 256, True, True), (2, 421, 3, 1152, False, False),
                                                         (1, 333, 2, 256, True, False), (3, 4336, 24, 12288, True, False),
                                                         # 224 x 256 tiles, whole and with two batch elements in a tile
                                                         (1, 672, 24, 12288, True, False), (2, 300, 24, 12288, True, True), (1, 513, 24, 12288, False, False)])
def test_linear_qk_norm_rope_epilogue(B, L, H, mlp, bias, per_batch_pe):
    """linear1 with QKNorm + RoPE in the epilogue: q and k leave as [B,H,L,128], v and the GELU'd mlp
    columns as in the split epilogue. Checked against the oracle chain on the un-fused projection
    and against the preparation kernel the block otherwise runs."""
    D, hid = 128, H * 128
    M, N = B * L, 3 * hid + mlp
    g = seeded(L + H)
    x = randn(g, M, hid, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, hid, dtype=torch.bfloat16, std=hid ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.02).to(DEV) if bias else None
    qs = (torch.rand(D, generator=g) + 0.5).to(torch.bfloat16).to(DEV)
    ks = (torch.rand(D, generator=g) + 0.5).to(torch.bfloat16).to(DEV)
    pe = randn(g, B if per_batch_pe else 1, 1, L, D // 2, 2, 2).to(DEV)

    qkv = torch.zeros(M, 3 * hid, dtype=torch.bfloat16, device=DEV)
    both = torch.zeros(M, hid + mlp, dtype=torch.bfloat16, device=DEV)
    q = torch.empty(B, H, L, D, dtype=torch.bfloat16, device=DEV)
    k = torch.empty_like(q)
    assert qk_fusable(x, w, L, D) == (-(-M // 256) * (N // 256) >= 160)   # small ones are taken, just not preferred
    tk.linear_into(x, w, b, activation="GELU", act_begin=3 * hid, out=qkv, out2=both[:, hid:], split=3 * hid,
                   qk=dict(q_out=q, k_out=k, q_scale=qs, k_scale=ks, pe=pe, heads=H, seq_len=L, eps=1e-6))

    # un-fused: the same projection, then the preparation kernel
    qkv_u = torch.empty_like(qkv)
    both_u = torch.zeros_like(both)
    tk.linear_into(x, w, b, activation="GELU", act_begin=3 * hid, out=qkv_u, out2=both_u[:, hid:], split=3 * hid)
    fused = plan_of(qk_args(B, L, H, mlp))
    plain = plan_of(linear_args(M, N, hid, Y2=PTR, ldy=3 * hid, ldy2=hid + mlp, split_n=3 * hid, act=nv.ACT_GELU_TANH, act_begin=3 * hid))
    if (fused.family == EIGHT_WAVES) == (plain.family == EIGHT_WAVES):   # v and mlp columns: K summed in the same order, same bits
        assert torch.equal(qkv[:, 2 * hid:], qkv_u[:, 2 * hid:])
        assert torch.equal(both, both_u)
    else:                                                                # in another order: a value at a rounding boundary may go either way
        for got, want in ((qkv[:, 2 * hid:], qkv_u[:, 2 * hid:]), (both, both_u)):
            assert ((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 1e-4).all() and (got != want).float().mean() < 5e-3
    assert (qkv[:, :2 * hid] == 0).all()                               # q and k columns are not written
    heads = qkv_u.view(B, L, 3, H, D).permute(2, 0, 3, 1, 4)
    q_u, k_u, _ = tk.qkv_prep(heads[0], heads[1], None, pe=pe, q_scale_img=qs, k_scale_img=ks)
    # oracle chain on the bf16 projection
    qn = oracle.rms_norm_ref(heads[0].cpu(), qs.cpu())
    kn = oracle.rms_norm_ref(heads[1].cpu(), ks.cpu())
    rq, rk = oracle.apply_rope_ref(qn, kn, pe.cpu())

    def close(got, want, normed, atol, rtol):
        """atol + rtol |want|, plus what one bf16 ulp of a normalised value is worth behind the 2 x 2 matrix:
        where x * rstd falls on a rounding boundary two correct evaluations may round it either way, and
        the table here is random (entries of several units, rows that cancel), which magnifies that ulp."""
        xn = normed.float().reshape(*normed.shape[:-1], -1, 1, 2).abs()
        amp = (pe.cpu().float().abs() * xn).sum(-1).reshape(normed.shape)
        err = (got.cpu().float() - want.cpu().float()).abs()
        assert (err <= atol + rtol * want.cpu().float().abs() + 2.0 ** -7 * amp).all(), err.max().item()
        assert err.mean().item() < 2e-3

    close(q, q_u, qn, 1e-2, 1e-2)
    close(k, k_u, kn, 1e-2, 1e-2)
    close(q, rq, qn, 2e-2, 2e-2)
    close(k, rk, kn, 2e-2, 2e-2)


@pytest.mark.parametrize("M", [1, 2, 5, 8])
@pytest.mark.parametrize("N,K", [(9216, 3072), (18432, 3072), (40, 72), (33, 50)])
def test_linear_input_silu_is_modulation(M, N, K):
    """lin(silu(vec)) of Modulation (modules/blocks.py:62-67) as one launch: SiLU in fp32 rounded to bf16
    on the way in, bit-identical to the two-launch form and within tolerance of the oracle."""
    from triton_kernels.modules.blocks import _silu
    g = seeded(M + N + K)
    vec = randn(g, M, K, dtype=torch.bfloat16, std=2.0).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.02).to(DEV)
    fused = tk.linear_into(vec, w, b, in_activation="SiLU")
    two = tk.linear(_silu(vec), w, b)
    assert torch.equal(fused, two)
    ref32 = oracle.linear_ref_fp32(oracle.silu_ref(vec), w, b)
    torch.testing.assert_close(fused.float(), ref32, atol=2e-2, rtol=1e-2)


def test_linear_input_silu_needs_few_rows_and_modulation_uses_it():
    g = seeded(3)
    vec = randn(g, 9, 64, dtype=torch.bfloat16).to(DEV)
    w = randn(g, 32, 64, dtype=torch.bfloat16).to(DEV)
    with pytest.raises(AssertionError):
        tk.linear_into(vec, w, None, in_activation="SiLU")
    from triton_kernels.modules.blocks import Modulation
    torch.manual_seed(0)
    mod = Modulation(256, double=True).to(torch.bfloat16).to(DEV)
    for rows in (1, 3, 9):                                    # 9 rows: the two-launch form
        v = randn(g, rows, 256, dtype=torch.bfloat16).to(DEV)
        m1, m2 = mod(v)
        want = oracle.linear_ref_fp32(oracle.silu_ref(v), mod.lin.weight, mod.lin.bias)[:, None, :].chunk(6, dim=-1)
        for got, ref in zip((m1.shift, m1.scale, m1.gate, m2.shift, m2.scale, m2.gate), want):
            assert got.shape == (rows, 1, 256)
            torch.testing.assert_close(got.float(), ref, atol=2e-2, rtol=1e-2)
        mod.fused_silu = False
        u1, _ = mod(v)
        mod.fused_silu = True
        assert torch.equal(u1.scale, m1.scale)


@pytest.mark.parametrize("gated", [False, True])
def test_linear_mlp_in_shape(gated):
    """4608 x 12288 outputs, 3.375 rounds of 256 x 256 tiles: compared with the fp32 product."""
    g = seeded(77 + gated)
    M, N, K = 4608, 12288, 192
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.02).to(DEV)
    if not gated:
        y = tk.linear(a, w, b, activation="GELU")
        ref32 = oracle.linear_ref_fp32(a, w, b, "GELU")
        assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()
        return
    B, L = 9, 512
    x = randn(g, B, L, N, dtype=torch.bfloat16).to(DEV)
    gate = randn(g, B, 1, N, dtype=torch.bfloat16).to(DEV)
    out = torch.empty_like(x)
    tk.linear_into(a, w, b, out=out.view(M, N), resid=x.view(M, N), gate=gate)
    gy = gate.float() * oracle.linear_ref_fp32(a, w, b).view(B, L, N)
    want32 = x.float() + gy
    bound = 2.0 ** -8 * 1.01 * (2 * gy.abs() + want32.abs()) + 2e-3
    assert ((out.float() - want32).abs() <= bound).all()


@pytest.mark.parametrize("B,L,N,K,splits", [
    (1, 9, 64, 64, 1), (1, 65, 96, 128, 1),          # one slab, two slabs; a row past the smallest tile
    (3, 43, 200, 8192, 2), (1, 320, 384, 6144, 2),   # few tiles, long K: K over several workgroups (batch elements inside a tile)
    (7, 19, 1000, 520, 1),                           # K tail, columns past the last tile, seven batch elements in two tiles
    (1, 333, 9216, 192, 1), (2, 640, 3072, 640, 1), (1, 2700, 3072, 192, 1), (3, 1445, 3072, 128, 1), (1, 2049, 9224, 72, 1),
])
def test_linear_tile_edges(B, L, N, K, splits):
    """Tiles where they can go wrong: row, column and K remainders, several batch elements in a tile, K split
    over workgroups (test_linear_every_tile has each tile by name). Plain, GELU and gated-residual epilogues against the fp32 product, at
    half a bf16 ulp per rounding plus the spread of an fp32 sum in another order."""
    g = seeded(B + L + N + K)
    M = B * L
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
    args = nv.LinearArgs()
    y0 = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    args.A, args.W, args.Y, args.M, args.N, args.K = a.data_ptr(), w.data_ptr(), y0.data_ptr(), M, N, K
    args.lda, args.ldw, args.ldy, args.split_n = K, K, N, N
    assert (nv.lib().flux_linear_workspace_bytes(nv.byref(args)) > 0) == (splits > 1)
    for act in ("", "GELU"):
        ref32 = oracle.linear_ref_fp32(a, w, b, act)
        y = tk.linear(a, w, b, activation=act)
        assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all(), act
    x = randn(g, B, L, N, dtype=torch.bfloat16).to(DEV)
    gate = randn(g, B, 1, N, dtype=torch.bfloat16).to(DEV)
    out = torch.full((B, L, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    tk.linear_into(a, w, b, out=out.view(M, N), resid=x.view(M, N), gate=gate)
    assert torch.equal(out, oracle.gated_residual_ref(x, gate, tk.linear(a, w, b).view(B, L, N)))
    # without a workspace the same product runs unsplit
    args.bias = b.data_ptr()
    nv.check(nv.lib().flux_linear_bf16(nv.byref(args), nv.stream_ptr(a.device)), "flux_linear_bf16")
    ref32 = oracle.linear_ref_fp32(a, w, b)
    assert ((y0.float() - ref32).abs() <= half_ulp_bound(ref32)).all()


# Every tile that a product can get, by a product of few operations that gets it: with rows and columns to spare, with
# and without a K tail, and with K in parts.
EVERY_TILE = [
    (EIGHT_WAVES, 64, 64, (9, 72, 64), (11, 72, 72), (9, 72, 8192)),
    (EIGHT_WAVES, 64, 96, (132, 5968, 64), (131, 6256, 72), (1397, 72, 6144)),
    (EIGHT_WAVES, 96, 96, (65, 8624, 64), (93, 8472, 80), (74, 1488, 6144)),
    (EIGHT_WAVES, 128, 96, (108, 12648, 64), (229, 8904, 72), (201, 1376, 12288)),
    (EIGHT_WAVES, 128, 192, (406, 11984, 64), (999, 5128, 80), (3703, 136, 12288)),
    (EIGHT_WAVES, 160, 96, (302, 7368, 64), (138, 12496, 104), (135, 2032, 12288)),
    (EIGHT_WAVES, 160, 128, (341, 8312, 64), (250, 12560, 72), (3011, 104, 12288)),
    (EIGHT_WAVES, 160, 192, (4844, 1184, 64), (407, 12728, 72), (278, 3384, 12288)),
    (EIGHT_WAVES, 192, 128, (180, 12624, 64), (183, 12560, 96), (2105, 208, 12288)),
    (EIGHT_WAVES, 192, 192, (535, 12624, 64), (829, 8384, 72), (1607, 920, 12288)),
    (EIGHT_WAVES, 224, 128, (650, 8432, 64), (666, 8736, 88), (200, 2344, 12288)),
    (EIGHT_WAVES, 256, 128, (692, 10200, 64), (490, 12688, 72), (988, 1248, 12288)),
    (RECT, 224, 192, (774, 9936, 64), (1034, 8288, 72), None),
    (RECT, 256, 192, (711, 12584, 64), (936, 10536, 72), None),
    (RECT, 288, 192, (1124, 8792, 64), (1557, 7600, 72), None),
    (SQUARE, 256, 256, (1174, 9880, 64), (4128, 3320, 72), None),
]


@pytest.mark.parametrize("family,tile_m,tile_n,whole,tail,parts", EVERY_TILE)
def test_linear_every_tile(family, tile_m, tile_n, whole, tail, parts):
    """Each tile against the fp32 product (half a bf16 ulp plus the spread of an fp32 sum in another order): plain, and
    the gated residual as the two operators on the kernel's own product. The plan is asserted, so that a change of
    the costs cannot leave a tile untested."""
    for M, N, K in filter(None, (whole, tail, parts)):
        plan = plan_of(linear_args(M, N, K))
        assert (plan.family, plan.tile_m, plan.tile_n, plan.splits > 1) == (family, tile_m, tile_n, (M, N, K) == parts), (M, N, K)
        g = seeded(M + N + K)
        a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
        w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
        b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
        y = tk.linear(a, w, b)
        ref32 = oracle.linear_ref_fp32(a, w, b)
        assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all(), (M, N, K)
        x, gate = randn(g, 1, M, N, dtype=torch.bfloat16).to(DEV), randn(g, 1, 1, N, dtype=torch.bfloat16).to(DEV)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        tk.linear_into(a, w, b, out=out, resid=x.view(M, N), gate=gate)
        assert torch.equal(out.view(1, M, N), oracle.gated_residual_ref(x, gate, y.view(1, M, N))), (M, N, K)


@pytest.mark.parametrize("M,N,K", [
    (320, 10920, 4096), (320, 10928, 4096),    # the last W walked in turn and the first one that is not
    (330, 3072, 15360), (1100, 3072, 15360),   # K in parts, two tile rows; groups of four and of three
    (940, 3072, 15360), (900, 3072, 15360),    # a group of four and a tile row of its own, full enough and not
    (470, 3072, 15360), (500, 8200, 6152),     # three tile rows: K in parts, and a K tail in a last group of one slab
    (400, 15000, 3080), (1000, 2920, 15416),   # K tail in a last group of slabs that is shorter and in a whole one
])
def test_linear_slabs_out_of_turn(M, N, K):
    """Eight-wave tiles that walk K in orders of their own, against the fp32 product: half a bf16 ulp plus the spread of an fp32 sum in another order."""
    assert plan_of(linear_args(M, N, K)).family == EIGHT_WAVES
    g = seeded(M + N + K)
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
    ref32 = oracle.linear_ref_fp32(a, w, b)
    assert ((tk.linear(a, w, b).float() - ref32).abs() <= half_ulp_bound(ref32)).all()


@pytest.mark.parametrize("L", [320, 257])
def test_linear_qk_slabs_out_of_turn(L):
    """The same with QKNorm + RoPE in the epilogue: v and mlp columns against the fp32 product, q and k against the preparation kernel on the plain
    one. A product on a rounding boundary may go either way: one bf16 ulp, and one for each rounding of norm, scale and rotation."""
    H, D, mlp = 24, 128, 12288
    hid = H * D
    N = 3 * hid + mlp
    assert plan_of(qk_args(1, L, H, mlp)).family == EIGHT_WAVES
    g = seeded(L)
    x = randn(g, L, hid, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, hid, dtype=torch.bfloat16, std=hid ** -0.5).to(DEV)
    qs, ks = [(torch.rand(D, generator=g) + 0.5).to(torch.bfloat16).to(DEV) for _ in range(2)]
    angle = randn(g, 1, 1, L, D // 2).to(DEV)
    pe = torch.stack([angle.cos(), -angle.sin(), angle.sin(), angle.cos()], dim=-1).reshape(1, 1, L, D // 2, 2, 2)
    qkv = torch.zeros(L, 3 * hid, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(L, mlp, dtype=torch.bfloat16, device=DEV)
    q = torch.empty(1, H, L, D, dtype=torch.bfloat16, device=DEV)
    k = torch.empty_like(q)
    tk.linear_into(x, w, None, activation="GELU", act_begin=3 * hid, out=qkv, out2=out, split=3 * hid, qk=dict(q_out=q, k_out=k, q_scale=qs, k_scale=ks, pe=pe, heads=H, seq_len=L, eps=1e-6))
    ref32, gelu32 = oracle.linear_ref_fp32(x, w, None), oracle.linear_ref_fp32(x, w, None, "GELU")
    for got, want in ((qkv[:, 2 * hid:], ref32[:, 2 * hid:3 * hid]), (out, gelu32[:, 3 * hid:])):
        assert ((got.float() - want).abs() <= half_ulp_bound(want)).all()
    heads = ref32[:, :3 * hid].to(torch.bfloat16).view(1, L, 3, H, D).permute(2, 0, 3, 1, 4)
    wants = tk.qkv_prep(heads[0], heads[1], None, pe=pe, q_scale_img=qs, k_scale_img=ks)
    for got, want, raw, scale in ((q, wants[0], heads[0], qs), (k, wants[1], heads[1], ks)):
        xn = oracle.rms_norm_ref(raw.cpu(), scale.cpu()).to(DEV).float().abs().unflatten(-1, (-1, 2)).sum(-1, keepdim=True).expand(-1, -1, -1, -1, 2).flatten(-2)
        assert ((got.float() - want.float()).abs() <= 4 * 2.0 ** -7 * xn + 1e-5).all()


@pytest.mark.parametrize("B,L,N,K,split,act_begin", [
    (1, 9, 3, 64, None, 0), (1, 65, 97, 128, 50, 33),        # less than a tile; a segment of 8 columns on both sides of the split
    (2, 100, 1001, 72, 1000, 1000), (3, 43, 201, 8192, None, 7),   # K tail; K over several workgroups, batch elements inside a tile
    (1, 320, 3073, 640, 8, 3000), (1, 700, 6001, 64, 3080, 3080),  # several sizes of eight-wave tiles
    (3, 1000, 1001, 192, 500, 0), (1, 2300, 6001, 192, None, 0), (4, 1000, 3073, 3072, 500, 0),
    (6, 250, 12289, 3072, 12000, 12288), (6, 256, 12289, 3072, None, 0),   # 256-wide tiles, the last rows on 128-wide ones
])
def test_linear_outside_the_branch_free_form(B, L, N, K, split, act_begin):
    """Columns of any number, outputs that are not 16-byte addressable, a split and the first GELU column
    anywhere, GELU in front of the gate: against the fp32 product, half a bf16 ulp per rounding plus the spread of an
    fp32 sum in another order."""
    g = seeded(B + L + N + K)
    M, S = B * L, N if split is None else split
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
    plain32, gelu32 = oracle.linear_ref_fp32(a, w, b), oracle.linear_ref_fp32(a, w, b, "GELU")
    ref32 = torch.cat([plain32[:, :act_begin], gelu32[:, act_begin:]], dim=1)
    for pad in (0, 1):     # outputs with rows at any element
        y = torch.full((M, S + pad), float("nan"), dtype=torch.bfloat16, device=DEV)
        y2 = torch.full((M, N - S + 3), float("nan"), dtype=torch.bfloat16, device=DEV)
        tk.linear_into(a, w, b, activation="GELU", act_begin=act_begin, out=y[:, pad:], **({} if split is None else dict(out2=y2[:, 3:], split=split)))
        got = torch.cat([y[:, pad:], y2[:, 3:]], dim=1).float()
        assert ((got - ref32).abs() <= half_ulp_bound(ref32)).all()
        assert y[:, :pad].isnan().all() and y2[:, :3].isnan().all()    # nothing beside the outputs is written
    if split is None:
        x = randn(g, B, L, N, dtype=torch.bfloat16).to(DEV)
        gate = randn(g, B, 1, N, dtype=torch.bfloat16).to(DEV)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        tk.linear_into(a, w, b, activation="GELU", act_begin=act_begin, out=out, resid=x.view(M, N), gate=gate)
        gy = (gate.float() * ref32.view(B, L, N)).view(M, N)
        want32 = x.view(M, N).float() + gy
        bound = half_ulp_bound(ref32) * gate.float().abs().expand(B, L, N).reshape(M, N) + 2.0 ** -8 * 1.01 * (gy.abs() + want32.abs()) + 1e-6
        assert ((out.float() - want32).abs() <= bound).all()


@pytest.mark.parametrize("B,L0,L1,N,K", [
    (1, 65, 9, 96, 128),          # one tile row each, the smallest tiles
    (2, 100, 33, 1000, 8192),     # K over several workgroups, batch elements inside a tile
    (2, 300, 77, 200, 520),       # K tail, columns past the last tile
    (1, 320, 64, 3072, 12288), (2, 150, 40, 3072, 12288),   # the same on larger tiles, as in a double block of a small image
    (2, 1445, 256, 3072, 192), (1, 4096, 512, 1024, 64), (1, 4096, 512, 12288, 64),   # ragged rows in both products; large tiles
])
def test_linear_pair(B, L0, L1, N, K):
    """Two products in one launch against each product in fp32 (half a bf16 ulp plus the spread of another
    order of summation): plain, GELU, and the gated residual with x as slices of one longer sequence, whose
    batch elements are not evenly strided."""
    g = seeded(B + L0 + L1 + N + K)
    whole = randn(g, B, L0 + L1, K, dtype=torch.bfloat16).to(DEV)
    xs = [whole[:, :L0], whole[:, L0:]]
    ws = [randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV) for _ in xs]
    bs = [randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV) for _ in xs]
    refs = [oracle.linear_ref_fp32(x.reshape(-1, K), w, b) for x, w, b in zip(xs, ws, bs)]
    for act in ("", "GELU"):
        ys = linear_pair_into(*(dict(x=x, w=w, b=b, activation=act) for x, w, b in zip(xs, ws, bs)))
        for y, x, w, b in zip(ys, xs, ws, bs):
            ref32 = oracle.linear_ref_fp32(x.reshape(-1, K), w, b, act)
            assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all(), act
    rs = [randn(g, B, n, N, dtype=torch.bfloat16).to(DEV) for n in (L0, L1)]
    gates = [randn(g, B, 1, N, dtype=torch.bfloat16).to(DEV) for _ in xs]
    outs = linear_pair_into(*(dict(x=x, w=w, b=b, resid=r, gate=gt) for x, w, b, r, gt in zip(xs, ws, bs, rs, gates)))
    plain = linear_pair_into(*(dict(x=x, w=w, b=b) for x, w, b in zip(xs, ws, bs)))
    for out, y, r, gt, ref in zip(outs, plain, rs, gates, refs):
        assert torch.equal(out.view(r.shape), oracle.gated_residual_ref(r, gt, y.view(r.shape)))
    # products that cannot share a launch run one after the other
    ys = linear_pair_into(dict(x=xs[0], w=ws[0], b=bs[0]), dict(x=xs[1], w=ws[1][:8], b=None))
    assert ((ys[0].float() - refs[0]).abs() <= half_ulp_bound(refs[0])).all()
    ref32 = oracle.linear_ref_fp32(xs[1].reshape(-1, K), ws[1][:8], None)
    assert ((ys[1].float() - ref32).abs() <= half_ulp_bound(ref32)).all()


@pytest.mark.parametrize("rows", [1, 3])
def test_linear_pair_of_row_vectors(rows):
    """The two modulation projections of a double-stream block in one launch: the bits of two launches."""
    g = seeded(rows)
    x = randn(g, rows, 3072, dtype=torch.bfloat16).to(DEV)
    calls = [dict(x=x, w=randn(g, 1026, 3072, dtype=torch.bfloat16, std=0.02).to(DEV), b=randn(g, 1026, dtype=torch.bfloat16).to(DEV), in_activation="SiLU")
             for _ in range(2)]
    for y, call in zip(linear_pair_into(*calls), calls):
        assert torch.equal(y, tk.linear_into(**call))


@pytest.mark.parametrize("M,K", [(1, 8), (1, 2048), (1, 4096), (1, 4104), (1, 24576), (2, 3080), (3, 3072), (3, 3416), (4, 3072),
                                 (4, 3080), (5, 3072), (6, 4096), (7, 3072), (8, 3072), (8, 3080)])
@pytest.mark.parametrize("N", [1, 129])
def test_linear_row_vector_activation_shares(M, K, N):
    """The activation rows of a row-vector product reach the workgroup in shares of 2048 values, some of them requested in
    front of the weights: K at the edges of the shares, one past them, and past the memory they are staged in. Against
    the float64 product of the separate operator's activations: half a bf16 ulp, and the fp32 sum's own error of at
    most K 2^-24 of the sum of its terms' sizes."""
    from triton_kernels.modules.blocks import _silu
    g = seeded(M * K + N)
    x = randn(g, M, K, dtype=torch.bfloat16, std=2.0).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16).to(DEV)
    got = tk.linear_into(x, w, b, in_activation="SiLU")
    torch.testing.assert_close(_silu(x), oracle.silu_ref(x), atol=1e-6, rtol=2.0 ** -7)
    a = _silu(x).double()
    ref = a @ w.double().T + b.double()
    sizes = a.abs() @ w.double().abs().T + b.double().abs()
    assert ((got.double() - ref).abs() <= ref.abs() * (2.0 ** -8 * 1.01) + sizes * (K * 2.0 ** -24)).all()
    assert torch.equal(tk.linear_into(x, w, None, in_activation="SiLU"), tk.linear_into(x, w, torch.zeros_like(b), in_activation="SiLU"))


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("K", [1528, 1536, 1544, 3064, 3072, 3080, 6152])
def test_linear_row_vector_weight_depths(M, K):
    """K where a lane has three or six vectors of a weight row in flight, and one vector to either side: the same bound as
    above, and the columns of a wider call have the same bits."""
    g = seeded(M * K)
    x = randn(g, M, K, dtype=torch.bfloat16, std=2.0).to(DEV)
    w = randn(g, 75, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, 75, dtype=torch.bfloat16).to(DEV)
    got = tk.linear(x, w, b)
    ref = x.double() @ w.double().T + b.double()
    sizes = x.double().abs() @ w.double().abs().T + b.double().abs()
    assert ((got.double() - ref).abs() <= ref.abs() * (2.0 ** -8 * 1.01) + sizes * (K * 2.0 ** -24)).all()
    assert torch.equal(got[:, :9], tk.linear(x, w[:9], b[:9]))


@pytest.mark.parametrize("M,K", [(1, 3080), (2, 3080), (4, 3080), (4, 6144), (1, 24576), (8, 15360)])
def test_line_of_weights_read_past_the_cache(M, K):
    """Weights of half the cache, and of a column more: the columns of both have the bits of a call with the few of them."""
    N = (128 << 20) // (2 * K)
    x = randn(seeded(K), M, K, dtype=torch.bfloat16).to(DEV)
    w = torch.randn(N + 1, K, generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).bfloat16()
    few = tk.linear(x, w[N - 100:], None)
    ref = x.double() @ w[N - 100:].double().T
    assert ((few.double() - ref).abs() <= ref.abs() * (2.0 ** -8 * 1.01) + (x.double().abs() @ w[N - 100:].double().abs().T) * (K * 2.0 ** -24)).all()
    assert torch.equal(tk.linear(x, w, None)[:, N - 100:], few) and torch.equal(tk.linear(x, w[:N], None)[:, N - 100:], few[:, :100])


@pytest.mark.parametrize("M", [2, 3, 4, 5])
def test_line_of_whole_weight_rows_in_flight(M):
    """Weights of 80 MiB, up to which three and four activation rows have whole rows of 3072 in flight, and of a column more:
    every column has the bits of a call with few of them."""
    K, N = 3072, (80 << 20) // (2 * 3072)
    x = randn(seeded(M), M, K, dtype=torch.bfloat16).to(DEV)
    w = torch.randn(N + 1, K, generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).bfloat16()
    few = tk.linear(x, w[N - 100:], None)
    ref = x.double() @ w[N - 100:].double().T
    assert ((few.double() - ref).abs() <= ref.abs() * (2.0 ** -8 * 1.01) + (x.double().abs() @ w[N - 100:].double().abs().T) * (K * 2.0 ** -24)).all()
    assert torch.equal(tk.linear(x, w, None)[:, N - 100:], few) and torch.equal(tk.linear(x, w[:N], None)[:, N - 100:], few[:, :100])
    assert torch.equal(tk.linear(x, w, None, activation="GELU")[:, N - 100:], tk.linear(x, w[N - 100:], None, activation="GELU"))


@pytest.mark.parametrize("tile_m,tile_n,M,N,K", [(256, 224, 916, 12384, 1024), (256, 224, 1178, 9944, 1032), (224, 256, 880, 12320, 1024), (224, 256, 872, 12376, 1032),
                                                 (224, 288, 1586, 8200, 1024), (224, 288, 1580, 8312, 1032)])
def test_linear_wide_rectangles(tile_m, tile_n, M, N, K):
    """Rectangles of 50000 and more outputs with rows and columns to spare, with and without a K tail, against the fp32
    product (half a bf16 ulp plus the spread of an fp32 sum in another order): plain, two outputs with GELU in the second
    from a wave's edge on, a gated residual whose batch elements end inside a tile, and two products in one launch."""
    assert (lambda p: (p.family, p.tile_m, p.tile_n))(plan_of(linear_args(M, N, K))) == (RECT, tile_m, tile_n)
    g = seeded(M + N + K)
    a = randn(g, M, K, dtype=torch.bfloat16).to(DEV)
    w = randn(g, N, K, dtype=torch.bfloat16, std=K ** -0.5).to(DEV)
    b = randn(g, N, dtype=torch.bfloat16, std=0.5).to(DEV)
    y = tk.linear(a, w, b)
    ref32 = oracle.linear_ref_fp32(a, w, b)
    assert ((y.float() - ref32).abs() <= half_ulp_bound(ref32)).all()
    cut = tile_n // 2 * 3
    out = [torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=DEV) for n in (cut, N - cut)]
    tk.linear_into(a, w, b, activation="GELU", act_begin=cut, out=out[0], out2=out[1], split=cut)
    assert torch.equal(out[0], y[:, :cut])
    gelu32 = torch.nn.functional.gelu(ref32[:, cut:], approximate="tanh")
    assert ((out[1].float() - gelu32).abs() <= half_ulp_bound(gelu32) + 2.0 ** -10).all()   # (tanh by exp2 and rcp: 1e-3 at most)
    x, gate = randn(g, 2, M // 2, N, dtype=torch.bfloat16).to(DEV), randn(g, 2, 1, N, dtype=torch.bfloat16).to(DEV)
    both = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    tk.linear_into(a, w, b, out=both, resid=x.view(M, N), gate=gate)
    assert torch.equal(both.view(2, M // 2, N), oracle.gated_residual_ref(x, gate, y.view(2, M // 2, N)))
    rows = M // 3
    pair = linear_pair_into(dict(x=a[:rows], w=w, b=b), dict(x=a[rows:], w=w, b=b))
    # (its rows of tiles are others, and with them the tile: the same product at half an ulp)
    assert ((torch.cat(pair).float() - ref32).abs() <= half_ulp_bound(ref32)).all()
