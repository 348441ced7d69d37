"""The work that users of this package have it do, as measurable cases: whole Flux blocks from the
smallest image to a batch of large ones, and the operators under the block at the shapes and element
types of the operator sweeps.

A case is a dict of plain values. `prepare` makes what a program holds before the call (inputs,
weights, the rotation table), `run` is one pass through the public entry points, `work` the bytes and
operations a pass cannot do without, `tolerance` how far two correct evaluations may differ.
Imported with the repository's root as the working folder.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "triton-kernels_amd"))

import triton_kernels as tk  # noqa: E402
from triton_kernels.flux.layers import EmbedND  # noqa: E402

# The model width of every block: 24 heads of 128, an mlp of four times the hidden size.
HEADS, HEAD_DIM, HIDDEN, MLP = 24, 128, 3072, 12288
# The largest block pass, in tokens: batch 3 of 4336. Drawn cases stay at or below it.
MOST_TOKENS = 3 * 4336
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # One 1024 x 1024 image in a single-stream block, the shape the package is quoted on.
        {"name": "single_4608", "kind": "single", "batch": 1, "txt": 512, "img": 4096},
        # A batch of three with a ragged token count: the block script's shape and the largest pass.
        {"name": "single_b3_4336", "kind": "single", "batch": 3, "txt": 256, "img": 4080},
        # A 256 x 256 preview with a short prompt: weights and launches weigh more than tokens.
        {"name": "single_320", "kind": "single", "batch": 1, "txt": 64, "img": 256},
        # One 1024 x 1024 image in a double-stream block: separate text and image weights, joint attention.
        {"name": "double_4096_512", "kind": "double", "batch": 1, "txt": 512, "img": 4096},
        # A 512 x 512 image with a short prompt in a double-stream block.
        {"name": "double_1024_256", "kind": "double", "batch": 1, "txt": 256, "img": 1024},
        # Attention by itself, head dim 128, in the middle of the sweep (batch 4, 24 heads).
        {"name": "attention_b4_1024", "kind": "attention", "batch": 4, "heads": 24, "tokens": 1024, "head_dim": 128},
        # Attention at head dim 64 and a length no tile divides.
        {"name": "attention_d64_1084", "kind": "attention", "batch": 2, "heads": 24, "tokens": 1084, "head_dim": 64},
        # A projection of a few hundred rows (batch 4 of 128), as the linear sweep has it.
        {"name": "linear_512", "kind": "linear", "rows": 512, "in": 3072, "out": 3072, "act": ""},
        # Training step of the q/k norm: forward, then the gradients of input and scale.
        {"name": "rms_norm_train_1024", "kind": "rms_norm_train", "dtype": "bf16", "batch": 4, "heads": 24, "tokens": 1024, "head_dim": 128},
        # Layer norm with adaLN modulation in float32, the element type the sweep scripts feed it.
        {"name": "layer_norm_fp32_2048", "kind": "layer_norm", "dtype": "fp32", "batch": 4, "tokens": 2048, "width": 3072},
        # Rotation of q and k over a batch with an odd length.
        {"name": "rope_b4_1001", "kind": "rope", "dtype": "bf16", "batch": 4, "heads": 24, "tokens": 1001, "head_dim": 128},
        # The smallest call: the q/k norm module on the views of a 256-token projection.
        {"name": "qk_norm_256", "kind": "qk_norm", "dtype": "bf16", "batch": 1, "heads": 24, "tokens": 256, "head_dim": 128},
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the same ranges, every kind as often as it is listed."""
    kind = rng.choice([c["kind"] for c in listed()])
    if kind in ("single", "double"):
        batch = rng.randint(1, 3)
        img = _log_int(rng, 256, min(4096, MOST_TOKENS // batch - 512))
        return {"kind": kind, "batch": batch, "txt": _log_int(rng, 64, 512), "img": img}
    if kind == "attention":
        head_dim, heads = rng.choice([64, 128]), rng.choice([2, 24])
        return {"kind": kind, "batch": rng.choice([1, 2, 4]), "heads": heads, "tokens": _log_int(rng, 256, 4096), "head_dim": head_dim}
    if kind == "linear":
        shape = rng.choice([(HIDDEN, HIDDEN, ""), (HIDDEN, MLP, "GELU"), (MLP, HIDDEN, "")])
        return {"kind": kind, "rows": _log_int(rng, 256, 8192), "in": shape[0], "out": shape[1], "act": shape[2]}
    dtype, batch, tokens = rng.choice(["bf16", "fp32"]), rng.randint(1, 4), _log_int(rng, 256, 4096)
    if kind == "layer_norm":
        return {"kind": kind, "dtype": dtype, "batch": batch, "tokens": tokens, "width": rng.choice([1024, 2048, 3072])}
    head_dim = rng.choice([128, 128, 256]) if kind != "qk_norm" else 128
    return {"kind": kind, "dtype": dtype, "batch": batch, "heads": 24, "tokens": tokens, "head_dim": head_dim}


def _rotation_table(txt, img, head_dim, device):
    """[1, 1, txt + img, head_dim / 2, 2, 2]: text at position 0, image tokens on a raster as wide as the
    square image of at least that many tokens."""
    side = math.isqrt(img - 1) + 1
    ids = torch.zeros(1, txt + img, 3, device=device)
    at = torch.arange(img, device=device)
    ids[0, txt:, 1] = torch.div(at, side, rounding_mode="floor").float()
    ids[0, txt:, 2] = (at % side).float()
    axes = [head_dim // 8, head_dim * 7 // 16, head_dim * 7 // 16]
    return EmbedND(dim=head_dim, theta=10000, axes_dim=axes)(ids).contiguous()


class _Inputs:
    """Seeded normal values, drawn on the GPU in float32."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std).to(dtype)

    def scale(self, n, dtype=torch.bfloat16):
        return (torch.rand(n, generator=self.g, device="cuda") + 0.5).to(dtype)


def _block(kind, inputs):
    """A block with weights N(0, 1 / fan_in), biases N(0, 0.02) and norm scales U(0.5, 1.5)."""
    with torch.device("meta"):
        blk = tk.SingleStreamBlock(HIDDEN, HEADS) if kind == "single" else tk.DoubleStreamBlock(HIDDEN, HEADS, mlp_ratio=4.0, qkv_bias=True)
    blk = blk.to(torch.bfloat16).to_empty(device="cuda")
    with torch.no_grad():
        for name, p in blk.named_parameters():
            if name.endswith("scale"):
                p.copy_(inputs.scale(p.shape[0]))
            else:
                p.copy_(inputs.normal(*p.shape, std=p.shape[1] ** -0.5 if p.dim() == 2 else 0.02))
    return blk.eval()


def prepare(case, seed):
    kind, inputs = case["kind"], _Inputs(seed)
    state = {"kind": kind}
    if kind in ("single", "double"):
        batch, txt, img = case["batch"], case["txt"], case["img"]
        state["block"] = _block(kind, inputs)
        state["vec"] = inputs.normal(batch, HIDDEN)
        state["pe"] = _rotation_table(txt, img, HEAD_DIM, "cuda")
        if kind == "single":
            state["x"] = inputs.normal(batch, txt + img, HIDDEN)
        else:
            state["img"], state["txt"] = inputs.normal(batch, img, HIDDEN), inputs.normal(batch, txt, HIDDEN)
        return state
    if kind == "linear":
        state["x"] = inputs.normal(case["rows"], case["in"])
        state["w"] = inputs.normal(case["out"], case["in"], std=case["in"] ** -0.5)
        state["b"] = inputs.normal(case["out"], std=0.02)
        state["act"] = case["act"]
        return state
    dtype = DTYPES[case.get("dtype", "bf16")]
    if kind == "layer_norm":
        state["x"] = inputs.normal(case["batch"], case["tokens"], case["width"], dtype=dtype)
        state["scale"] = inputs.normal(case["batch"], 1, case["width"], std=0.1, dtype=dtype)
        state["shift"] = inputs.normal(case["batch"], 1, case["width"], std=0.1, dtype=dtype)
        return state
    shape = (case["batch"], case["heads"], case["tokens"], case["head_dim"])
    if kind == "attention":
        state["q"], state["k"], state["v"] = (inputs.normal(*shape) for _ in range(3))
    elif kind == "rope":
        state["q"], state["k"] = inputs.normal(*shape, dtype=dtype), inputs.normal(*shape, dtype=dtype)
        state["pe"] = _rotation_table(0, case["tokens"], case["head_dim"], "cuda")
    elif kind == "rms_norm_train":
        state["x"] = inputs.normal(*shape, dtype=dtype).requires_grad_(True)
        state["scale"] = inputs.scale(shape[-1], dtype).requires_grad_(True)
        state["dy"] = inputs.normal(*shape, dtype=dtype)
    else:
        # q and k as the views of a [batch, tokens, 3 * heads * head_dim] projection, as the blocks split it
        qkv = inputs.normal(shape[0], shape[2], 3 * shape[1] * shape[3], dtype=dtype)
        state["q"], state["k"], state["v"] = qkv.view(shape[0], shape[2], 3, shape[1], shape[3]).permute(2, 0, 3, 1, 4).unbind(0)
        norm = tk.QKNorm(shape[3]).to(device="cuda", dtype=dtype).eval()
        with torch.no_grad():
            norm.query_norm.scale.copy_(inputs.scale(shape[3], dtype))
            norm.key_norm.scale.copy_(inputs.scale(shape[3], dtype))
        state["norm"] = norm
    return state


def run(state):
    kind = state["kind"]
    if kind == "rms_norm_train":
        y = tk.rms_norm(state["x"], state["scale"])
        dx, dscale = torch.autograd.grad(y, (state["x"], state["scale"]), state["dy"])
        return y, dx, dscale
    with torch.no_grad():
        if kind == "single":
            return state["block"](state["x"], state["vec"], state["pe"])
        if kind == "double":
            return state["block"](state["img"], state["txt"], state["vec"], state["pe"])
        if kind == "attention":
            return tk.scaled_dot_product_attention(state["q"], state["k"], state["v"])
        if kind == "linear":
            return tk.linear(state["x"], state["w"], state["b"], activation=state["act"])
        if kind == "layer_norm":
            return tk.layer_norm_modulation(state["x"], state["scale"], state["shift"])
        if kind == "rope":
            return tk.apply_rope(state["q"], state["k"], state["pe"])
        return state["norm"](state["q"], state["k"], state["v"])


def work(case):
    kind = case["kind"]
    if kind in ("single", "double"):
        batch, tokens = case["batch"], case["txt"] + case["img"]
        rows = batch * tokens
        per_row = HIDDEN * (3 * HIDDEN + MLP) + (HIDDEN + MLP) * HIDDEN      # weights that a token meets
        vec = (3 if kind == "single" else 12) * HIDDEN * HIDDEN              # weights of the modulation projections
        weights = per_row * (1 if kind == "single" else 2) + vec
        flops = 2.0 * rows * per_row + 4.0 * batch * HEADS * tokens * tokens * HEAD_DIM + 2.0 * batch * vec
        return {"bytes": 2.0 * (2 * rows * HIDDEN + weights) + 8.0 * tokens * HEAD_DIM, "flops": flops}
    if kind == "linear":
        m, k, n = case["rows"], case["in"], case["out"]
        return {"bytes": 2.0 * (m * k + n * k + n + m * n), "flops": 2.0 * m * n * k}
    size = 4.0 if case.get("dtype") == "fp32" else 2.0
    if kind == "layer_norm":
        values = case["batch"] * case["tokens"] * case["width"]
        return {"bytes": size * (2 * values + 2 * case["batch"] * case["width"]), "flops": 9.0 * values}
    b, h, n, d = case["batch"], case["heads"], case["tokens"], case["head_dim"]
    values = b * h * n * d
    if kind == "attention":
        return {"bytes": size * 4 * values, "flops": 4.0 * b * h * n * n * d}
    if kind == "rope":
        return {"bytes": size * 4 * values + 8.0 * n * d, "flops": 6.0 * values}
    if kind == "rms_norm_train":
        # forward reads x and writes y; backward reads x and dy and writes dx
        return {"bytes": size * 5 * values, "flops": 13.0 * values}
    return {"bytes": size * 4 * values, "flops": 8.0 * values}


# About four times the error against the same path evaluated in float64 (relative, largest), per kind and
# element type. bf16 outputs carry one to four roundings of 2^-9 (a block: q, k, P and every intermediate);
# the float32 operators sum rows in float32, the gradient of the norm's scale over all rows of a tensor.
_TOLERANCE = {
    ("single", "bf16"): (1.2e-2, 0.14), ("double", "bf16"): (1.5e-2, 0.15), ("attention", "bf16"): (1.2e-2, 0.11),
    ("linear", "bf16"): (7e-3, 1.6e-2), ("rope", "bf16"): (6e-3, 1.6e-2), ("layer_norm", "bf16"): (1.4e-2, 6e-2),
    ("qk_norm", "bf16"): (1e-2, 3e-2), ("rms_norm_train", "bf16"): (1e-2, 3e-2),
    ("rope", "fp32"): (2e-7, 1e-6), ("layer_norm", "fp32"): (3e-7, 1.6e-6),
    ("qk_norm", "fp32"): (3e-7, 1.2e-6), ("rms_norm_train", "fp32"): (2e-6, 1e-5),
}


def tolerance(case):
    rel, largest = _TOLERANCE[case["kind"], case.get("dtype", "bf16")]
    return {"rel": rel, "max": largest}
