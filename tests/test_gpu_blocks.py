"""Flux blocks on the HIP kernels vs the plain-PyTorch blocks, the way the reference's
tests/test_blocks.py does it (state dict shared, bf16, atol 0.1), plus the full 4608-token single
block against the CPU oracle and fused-vs-unfused agreement."""
import pytest
import torch

import triton_kernels as tk
from oracle import flux_oracle as oracle
from triton_kernels import flux
from triton_kernels import testing as cfg
from util import DEV, randn, seeded

pytestmark = pytest.mark.gpu

HEADS, HEAD_DIM = 24, 128
HID = HEADS * HEAD_DIM


def _close(got, want, atol=0.1, mean=6e-3):
    """The reference's own bound (tests/test_blocks.py: atol 0.1 on outputs of size ~1) catches gross
    errors only; a wrong rounding site or epilogue shows in the mean error, which for two correct bf16
    evaluations of a block stays at a few 1e-3."""
    torch.testing.assert_close(got, want, atol=atol, rtol=0)
    err = (got.float() - want.float()).abs()
    assert err.mean().item() < mean, f"mean error {err.mean().item()}"
    rel = err.pow(2).sum().sqrt() / want.float().pow(2).sum().sqrt()
    assert rel.item() < 1e-2, f"relative error {rel.item()}"


def _pair(kind, seed):
    torch.manual_seed(seed)
    if kind == "single":
        ref = flux.SingleStreamBlock(HID, HEADS, mlp_ratio=4.0).to(torch.bfloat16)
        hip = tk.SingleStreamBlock(HID, HEADS, mlp_ratio=4.0).to(torch.bfloat16)
    else:
        ref = flux.DoubleStreamBlock(HID, HEADS, mlp_ratio=4.0).to(torch.bfloat16)
        hip = tk.DoubleStreamBlock(HID, HEADS, mlp_ratio=4.0).to(torch.bfloat16)
    hip.load_state_dict(ref.state_dict())
    return ref.to(DEV), hip.to(DEV)


@pytest.mark.parametrize("batch_size", [1, 2])
@pytest.mark.parametrize("seq_len", [256, 1024])
def test_single_stream_block(batch_size, seq_len, monkeypatch):
    from triton_kernels.modules import blocks
    ref, hip = _pair("single", seq_len + batch_size)
    g = seeded(seq_len)
    x = randn(g, batch_size, seq_len, HID, dtype=torch.bfloat16).to(DEV)
    vec = randn(g, batch_size, HID, dtype=torch.bfloat16).to(DEV)
    pe = randn(g, 1, 1, seq_len, HEAD_DIM // 2, 2, 2).to(DEV)
    with torch.no_grad():
        y_ref = ref(x=x, vec=vec, pe=pe)
        y_hip = hip(x=x, vec=vec, pe=pe)              # fused, QKNorm + RoPE wherever that is the faster way at this size
        with monkeypatch.context() as m:              # fused, QKNorm + RoPE in linear1's epilogue wherever that is possible
            calls = []
            m.setattr(blocks, "qk_pays", lambda *a: True)
            m.setattr(blocks, "linear_into", lambda *a, **kw: calls.append(kw.get("qk") is not None) or tk.linear_into(*a, **kw))
            y_epilogue = hip(x=x, vec=vec, pe=pe)
        assert any(calls) == blocks.qk_fusable(x, hip.linear1.weight, seq_len, HEAD_DIM) == (batch_size * seq_len > 256)
        hip.fuse_qk_epilogue = False
        y_prep = hip(x=x, vec=vec, pe=pe)             # fused, QKNorm + RoPE as one kernel behind linear1
        hip.fused = False
        y_unfused = hip(x=x, vec=vec, pe=pe)
    _close(y_hip, y_ref)
    _close(y_prep, y_ref)
    _close(y_unfused, y_ref)
    _close(y_hip, y_unfused, atol=0.05)
    _close(y_hip, y_prep, atol=0.05)
    _close(y_epilogue, y_ref)
    _close(y_epilogue, y_unfused, atol=0.05)
    _close(y_epilogue, y_prep, atol=0.05)


@pytest.mark.parametrize("batch_size", [1, 2])
@pytest.mark.parametrize("img_seq_len", [256, 1024])
def test_double_stream_block(batch_size, img_seq_len):
    ref, hip = _pair("double", img_seq_len + batch_size)
    g = seeded(img_seq_len)
    txt_len = 256
    img = randn(g, batch_size, img_seq_len, HID, dtype=torch.bfloat16).to(DEV)
    txt = randn(g, batch_size, txt_len, HID, dtype=torch.bfloat16).to(DEV)
    vec = randn(g, batch_size, HID, dtype=torch.bfloat16).to(DEV)
    pe = randn(g, 1, 1, txt_len + img_seq_len, HEAD_DIM // 2, 2, 2).to(DEV)
    with torch.no_grad():
        r_img, r_txt = ref(img=img, txt=txt, vec=vec, pe=pe)
        h_img, h_txt = hip(img=img, txt=txt, vec=vec, pe=pe)         # fused, text and image rows in shared launches
        for _ in range(3):                                           # the same bits every time
            a_img, a_txt = hip(img=img, txt=txt, vec=vec, pe=pe)
            assert torch.equal(a_img, h_img) and torch.equal(a_txt, h_txt)
        hip.fused = False
        u_img, u_txt = hip(img=img, txt=txt, vec=vec, pe=pe)
    _close(h_img, r_img)
    _close(h_txt, r_txt)
    _close(u_img, r_img)
    _close(u_txt, r_txt)
    _close(h_img, u_img, atol=0.05)
    _close(h_txt, u_txt, atol=0.05)


@pytest.mark.parametrize("batch_size,img_len,txt_len", [(1, 1024, 256), (2, 256, 77), (3, 300, 5), (1, 256, 4)])
def test_double_block_shared_launches_against_separate_ones(batch_size, img_len, txt_len, monkeypatch):
    """The fused double block with two products and two norms per launch against the same steps launched one by
    one. Both round every intermediate to bf16 (an ulp is up to 2^-7 of a value) and sum K in fp32, in another order
    where another tile is chosen, which moves the few values at a rounding boundary: 1e-3 of the output's 2-norm is a
    quarter of what the block's own roundings amount to (4e-3 against float64)."""
    from triton_kernels.modules import blocks
    torch.manual_seed(7)
    blk = tk.DoubleStreamBlock(HID, HEADS, mlp_ratio=4.0, qkv_bias=True).to(torch.bfloat16).to(DEV)
    g = seeded(img_len + txt_len)
    img = randn(g, batch_size, img_len, HID, dtype=torch.bfloat16).to(DEV)
    txt = randn(g, batch_size, txt_len, HID, dtype=torch.bfloat16).to(DEV)
    vec = randn(g, batch_size, HID, dtype=torch.bfloat16).to(DEV)
    pe = randn(g, 1, 1, txt_len + img_len, HEAD_DIM // 2, 2, 2).to(DEV)
    with torch.no_grad():
        together = blk(img=img, txt=txt, vec=vec, pe=pe)
        calls = []
        monkeypatch.setattr(blocks, "linear_pair_into", lambda *c: calls.append("linear") or tuple(tk.linear_into(**x) for x in c))
        monkeypatch.setattr(blocks, "layer_norm_modulation_pair", lambda *c: calls.append("norm") or tuple(tk.layer_norm_modulation(*x) for x in c))
        apart = blk(img=img, txt=txt, vec=vec, pe=pe)
    assert calls.count("linear") == 5 and calls.count("norm") == 2
    for a, b in zip(together, apart):
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 1e-3


def test_single_block_4608_tokens_vs_oracle():
    """The headline workload: 512 txt + 64x64 img tokens, hidden 3072, against the state-dict driven
    oracle evaluated by PyTorch on the same device (the CPU evaluation of a quarter-size sequence is
    in test_single_block_small_vs_cpu_oracle)."""
    x, vec, pe, sd = cfg.config5_block(DEV)
    blk = tk.SingleStreamBlock(HID, HEADS).to(torch.bfloat16).to(DEV)
    blk.load_state_dict(sd)
    with torch.no_grad():
        y = blk(x, vec, pe)
        want = oracle.single_stream_block_ref(sd, x, vec, pe, HEADS)
    torch.testing.assert_close(y, want, atol=0.1, rtol=0)
    err = (y.float() - want.float()).abs()
    assert err.mean().item() < 5e-3, f"mean error {err.mean().item()}"


def test_single_block_small_vs_cpu_oracle():
    x, vec, pe, sd = cfg.config5_block("cpu", n_txt=64, grid=16)
    want = oracle.single_stream_block_ref(sd, x, vec, pe, HEADS)     # CPU, same bits
    blk = tk.SingleStreamBlock(HID, HEADS).to(torch.bfloat16).to(DEV)
    blk.load_state_dict(sd)
    with torch.no_grad():
        y = blk(x.to(DEV), vec.to(DEV), pe.to(DEV))
    torch.testing.assert_close(y.cpu(), want, atol=0.1, rtol=0)
