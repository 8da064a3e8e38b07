"""Performance cases of the QLoRA path: what a program that trains, serves or publishes a QLoRA model calls.

`listed()` names the cases that are followed from version to version, `draw(rng)` gives further ones of the same ranges.
`prepare(case, seed)` builds what such a program holds before the call (modules with packed weights and LoRA factors,
activations, upstream gradients), `run(state)` is one pass through the public entry points.  Everything is synthetic and
made from the seed.

  op                what it stands for                                                     public entry point
  linear_decode     one projection for a few tokens (generation, one sequence or a small batch)   module(x)
  qkv_decode        the three attention projections on one hidden state, same regime       qlora_linears_forward
  mlp_infer         the SwiGLU MLP without gradients: decode, batched rollout, prefill     qlora_mlp_forward
  linear_train      forward + backward of one projection                                   module(x), autograd
  attention_train   forward + backward of q, k, v on one input and of o                    qlora_linears_forward, module(x)
  mlp_train         forward + backward of the SwiGLU MLP                                   qlora_mlp_forward
  moe_infer         routed experts without gradients                                       expert module(x, weights, ids)
  moe_train         routed experts, forward + backward, routing weights included           expert module(x, weights, ids)
  merge             base + LoRA update, published as bf16 or re-encoded in its own format  merged_weight, merge_requant_*
  quantize          bf16 checkpoint weight -> packed bytes and scales (model load)         xorl_amd.quantize
  dequantize        packed bytes and scales -> bf16                                        xorl_amd.quantize
"""

from __future__ import annotations

import math

import torch

from xorl_amd import functional as F
from xorl_amd import quantize as Q
from xorl_amd.qlora import (BlockFP8QLoRAMoeExperts, NF4QLoRAMoeExperts, NvFP4QLoRAMoeExperts, QLoRALinear,
                            qlora_linears_forward, qlora_mlp_forward)

DEVICE = "cuda"
DENSE_FORMATS = ("int4", "nvfp4", "block_fp8", "nf4")
EXPERT_MODULES = {"nvfp4": NvFP4QLoRAMoeExperts, "block_fp8": BlockFP8QLoRAMoeExperts, "nf4": NF4QLoRAMoeExperts}
# bytes of scales per weight element: int4 bf16 per 128, nvfp4 e4m3 per 16, block_fp8 fp32 per 128 x 128, nf4 fp32 per 64
SCALE_BYTES = {"int4": 2 / 128, "nvfp4": 1 / 16, "block_fp8": 4 / 16384, "nf4": 4 / 64}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one token through the smallest projection of an 8B model: launch and host latency
        {"name": "linear_decode_int4_m1", "op": "linear_decode", "fmt": "int4", "tokens": 1, "n": 1024, "k": 4096, "r": 16},
        # eight sequences, separate q / k / v modules of an 8B model
        {"name": "qkv_decode_nvfp4_m8", "op": "qkv_decode", "fmt": "nvfp4", "tokens": 8, "q": 4096, "kv": 1024, "k": 4096, "r": 16},
        # one token through the MLP of an 8B model: a read of 144 MiB of weights
        {"name": "mlp_decode_fp8_m1", "op": "mlp_infer", "fmt": "block_fp8", "tokens": 1, "hidden": 4096, "inter": 12288, "r": 16},
        # a rollout batch of 64 sequences
        {"name": "mlp_rollout_int4_m64", "op": "mlp_infer", "fmt": "int4", "tokens": 64, "hidden": 4096, "inter": 12288, "r": 16},
        # the prefill of one prompt of an uneven length
        {"name": "mlp_prefill_nf4_m1357", "op": "mlp_infer", "fmt": "nf4", "tokens": 1357, "hidden": 4096, "inter": 12288, "r": 16},
        # a small training micro-batch on one projection
        {"name": "linear_train_int4_m512", "op": "linear_train", "fmt": "int4", "tokens": 512, "n": 4096, "k": 4096, "r": 16},
        # attention projections of a 32B model, an ordinary micro-batch
        {"name": "attention_train_nvfp4_m4096", "op": "attention_train", "fmt": "nvfp4", "tokens": 4096, "q": 8192, "kv": 1024,
         "k": 5120, "r": 16},
        # the MLP of an 8B model at a full micro-batch: the headline workload
        {"name": "mlp_train_fp8_m8192", "op": "mlp_train", "fmt": "block_fp8", "tokens": 8192, "hidden": 4096, "inter": 12288, "r": 32},
        # 16 sequences through 128 routed experts
        {"name": "moe_decode_nvfp4_t16", "op": "moe_infer", "fmt": "nvfp4", "tokens": 16, "experts": 128, "topk": 8, "hidden": 2048,
         "inter": 768, "r": 16, "shared": False},
        # a full micro-batch through 128 routed experts with uneven loads
        {"name": "moe_train_fp8_t16384", "op": "moe_train", "fmt": "block_fp8", "tokens": 16384, "experts": 128, "topk": 8,
         "hidden": 2048, "inter": 768, "r": 16, "shared": False},
        # folding the trained update into the base weight
        {"name": "merge_requant_fp8", "op": "merge", "fmt": "block_fp8", "n": 12288, "k": 4096, "r": 32, "publish": False},
        # encoding a checkpoint's weight at load
        {"name": "quantize_nvfp4", "op": "quantize", "fmt": "nvfp4", "n": 12288, "k": 4096, "experts": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    op = rng.choice(("linear_decode", "qkv_decode", "mlp_infer", "mlp_infer", "mlp_infer", "linear_train", "attention_train",
                     "mlp_train", "moe_infer", "moe_train", "merge", "codec"))
    hidden = 128 * rng.randint(8, 40)                                   # 1024 .. 5120
    inter = 128 * round(hidden * rng.uniform(2.4, 3.4) / 128)
    q, kv = 128 * rng.randint(8, 64), 128 * rng.choice((2, 4, 8))
    r = rng.choice((8, 16, 32, 64))
    fmt = rng.choice(DENSE_FORMATS)
    few = _log_int(rng, 1, 16)
    if op == "linear_decode":
        n, k = rng.choice(((q, hidden), (kv, hidden), (hidden, q), (inter, hidden), (hidden, inter)))
        return {"op": op, "fmt": fmt, "tokens": _log_int(rng, 1, 64), "n": n, "k": k, "r": r}
    if op == "qkv_decode":
        return {"op": op, "fmt": fmt, "tokens": few, "q": q, "kv": kv, "k": hidden, "r": r}
    if op == "mlp_infer":
        lo, hi = rng.choice(((1, 16), (17, 64), (65, 8192)))            # decode, rollout, prefill
        tokens = min(_log_int(rng, lo, hi), int(3e12 / (6.0 * hidden * inter)))
        return {"op": op, "fmt": fmt, "tokens": tokens, "hidden": hidden, "inter": inter, "r": r}
    if op in ("linear_train", "attention_train", "mlp_train"):
        tokens = _log_int(rng, 64, 8192)
        if op == "linear_train":
            n, k = rng.choice(((q, hidden), (kv, hidden), (hidden, q), (inter, hidden), (hidden, inter)))
            return {"op": op, "fmt": fmt, "tokens": tokens, "n": n, "k": k, "r": r}
        if op == "attention_train":
            return {"op": op, "fmt": fmt, "tokens": tokens, "q": q, "kv": kv, "k": hidden, "r": r}
        tokens = min(tokens, int(3e12 / (12.0 * hidden * inter)))
        return {"op": op, "fmt": fmt, "tokens": tokens, "hidden": hidden, "inter": inter, "r": r}
    if op in ("moe_infer", "moe_train"):
        experts = rng.choice((8, 16, 32, 64, 128))
        topk = rng.choice((2, 4) if experts < 32 else (4, 6, 8))
        hidden, inter = 256 * rng.randint(4, 16), 128 * rng.randint(4, 12)
        experts = min(experts, max(8, (1 << 28) // (hidden * inter)))
        tokens = _log_int(rng, *rng.choice(((1, 64), (65, 4096)))) if op == "moe_infer" else _log_int(rng, 64, 16384)
        tokens = min(tokens, int(1.5e12 / (topk * (4.0 if op == "moe_infer" else 12.0) * hidden * inter)))
        return {"op": op, "fmt": rng.choice(tuple(EXPERT_MODULES)), "tokens": tokens, "experts": experts, "topk": topk,
                "hidden": hidden, "inter": inter, "r": min(r, 32), "shared": rng.random() < 0.5}
    n, k = rng.choice(((q, hidden), (kv, hidden), (hidden, q), (inter, hidden), (hidden, inter)))
    if op == "merge":
        return {"op": op, "fmt": fmt, "n": n, "k": k, "r": r, "publish": rng.random() < 0.5}
    experts = fmt in ("nvfp4", "nf4") and rng.random() < 0.5            # one expert's [in, out] slice: packed down the rows
    if experts:
        n, k = 256 * rng.randint(4, 16), 128 * rng.randint(4, 12)
    return {"op": rng.choice(("quantize", "dequantize")), "fmt": fmt, "n": n, "k": k, "experts": experts}


# ---------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------
class _Maker:
    """Seeded tensors on the GPU: weights ~ N(0, 0.02), activations and upstream gradients ~ N(0, 1)."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device=DEVICE).mul_(std).to(dtype)

    def acts(self, *shape):
        return self.randn(*shape, dtype=torch.bfloat16)

    def linear(self, fmt, n, k, r):
        lin = torch.nn.Linear(k, n, bias=False, device="meta")
        lin.weight = torch.nn.Parameter(self.randn(n, k, std=0.02, dtype=torch.bfloat16), requires_grad=False)
        m = QLoRALinear.from_module(lin, r=r, lora_alpha=2 * r, quant_format=fmt)
        with torch.no_grad():
            m.lora_A.copy_(self.randn(r, k, std=0.02))
            m.lora_B.copy_(self.randn(n, r, std=0.02))
        return m

    def experts(self, c):
        E, H, I, r = c["experts"], c["hidden"], c["inter"], c["r"]
        m = EXPERT_MODULES[c["fmt"]](E, E, I, H, r=r, lora_alpha=2 * r, hybrid_shared=c["shared"], device=DEVICE)
        w = lambda *shape: self.randn(*shape, std=0.02)
        m.load_weights(w(E, H, I), w(E, H, I), w(E, I, H))
        with torch.no_grad():
            for p in m.get_lora_parameters():
                p.copy_(w(*p.shape))
        return m

    def routing(self, tokens, experts, topk):
        """A router's output with uneven loads: token counts per expert follow Zipf(1.1), a few experts stay empty."""
        popularity = -1.1 * torch.log(torch.arange(1, experts + 1, device=DEVICE, dtype=torch.float32))
        popularity = popularity[torch.randperm(experts, generator=self.g, device=DEVICE)]
        noise = torch.rand(tokens, experts, generator=self.g, device=DEVICE).clamp_(1e-9, 1 - 1e-7)
        logits = popularity - torch.log(-torch.log(noise))
        weights, ids = torch.topk(torch.softmax(logits, -1), topk, dim=-1)
        return (weights / weights.sum(-1, keepdim=True)).to(torch.bfloat16), ids


def _quantize(fmt, w, experts):
    """The codec call a loader makes for one weight; -> (packed, scales[, global scale])."""
    if fmt == "int4":
        return Q.int4_quantize_sym(w, 128)
    if fmt == "block_fp8":
        return Q.block_fp8_quantize_gkn(w)
    if fmt == "nvfp4":
        return (Q.nvfp4_quantize_gkn if experts else Q.nvfp4_quantize)(w)
    return (Q.nf4_quantize_gkn if experts else Q.nf4_quantize)(w)


def _dequantize(fmt, codes, n, k, experts):
    if fmt == "int4":
        return Q.int4_dequantize(*codes, n, k, 128)
    if fmt == "block_fp8":
        return Q.block_fp8_dequantize_gkn(*codes, out_dtype=torch.bfloat16)
    if fmt == "nvfp4":
        return Q.nvfp4_dequantize_gkn(*codes, n, k) if experts else Q.nvfp4_dequantize(*codes, n * k)
    return Q.nf4_dequantize_gkn(*codes, n, k) if experts else Q.nf4_dequantize(*codes, n * k)


def prepare(case, seed):
    mk, op, fmt = _Maker(seed), case["op"], case["fmt"]
    s = {"case": case}
    train = op.endswith("_train")
    if op in ("linear_decode", "linear_train"):
        s["mods"] = [mk.linear(fmt, case["n"], case["k"], case["r"])]
        s["x"] = mk.acts(case["tokens"], case["k"])
    elif op in ("qkv_decode", "attention_train"):
        s["mods"] = [mk.linear(fmt, n, case["k"], case["r"]) for n in (case["q"], case["kv"], case["kv"])]
        s["x"] = mk.acts(case["tokens"], case["k"])
        if train:
            s["mods"].append(mk.linear(fmt, case["k"], case["q"], case["r"]))
            s["attn"] = mk.acts(case["tokens"], case["q"]).requires_grad_(True)
    elif op in ("mlp_infer", "mlp_train"):
        H, I = case["hidden"], case["inter"]
        s["mods"] = [mk.linear(fmt, n, k, case["r"]) for n, k in ((I, H), (I, H), (H, I))]
        s["x"] = mk.acts(case["tokens"], H)
    elif op in ("moe_infer", "moe_train"):
        s["mods"] = [mk.experts(case)]
        s["x"] = mk.acts(case["tokens"], case["hidden"])
        s["weights"], s["ids"] = mk.routing(case["tokens"], case["experts"], case["topk"])
        s["weights"].requires_grad_(train)
    elif op == "merge":
        s["mods"] = [mk.linear(fmt, case["n"], case["k"], case["r"])]
        s["qw"] = s["mods"][0]._quant_weight()
    else:
        w = mk.randn(case["n"], case["k"], std=0.02, dtype=torch.bfloat16)
        s["w"] = w if op == "quantize" else _quantize(fmt, w, case["experts"])
    if train:
        s["x"].requires_grad_(True)
        if op == "attention_train":
            outs = [case["q"], case["kv"], case["kv"], case["k"]]
        else:
            outs = [case["n"] if op == "linear_train" else case["hidden"]]
        s["dy"] = [mk.acts(case["tokens"], n) for n in outs]
        leaves = [s["x"]] + [s[k] for k in ("attn", "weights") if k in s]
        s["leaves"] = leaves + [p for m in s["mods"] for p in m.get_lora_parameters()]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _forward(s):
    op, mods, x = s["case"]["op"], s["mods"], s["x"]
    if op in ("linear_decode", "linear_train"):
        return [mods[0](x)]
    if op == "qkv_decode":
        return qlora_linears_forward(mods, x)
    if op == "attention_train":
        return [*qlora_linears_forward(mods[:3], x), mods[3](s["attn"])]
    if op in ("mlp_infer", "mlp_train"):
        return [qlora_mlp_forward(*mods, x)]
    return [mods[0](x, s["weights"], s["ids"])]


def _merge(s):
    m, case = s["mods"][0], s["case"]
    if case["publish"]:
        return m.merged_weight()
    qw, args = s["qw"], (m.lora_A, m.lora_B, m.active_r, m.scaling)
    if case["fmt"] == "block_fp8":
        return F.merge_requant_fp8(qw, *args)
    if case["fmt"] == "nvfp4":
        return F.merge_requant_nvfp4(qw, *args, F.merge_amax(qw, *args))
    if case["fmt"] == "nf4":
        return F.merge_requant_nf4(qw, *args)
    return F.merge_requant_int4(qw, *args, symmetric=True)


def run(state):
    case = state["case"]
    op, fmt = case["op"], case["fmt"]
    if op == "quantize":
        return _quantize(fmt, state["w"], case["experts"])
    if op == "dequantize":
        return _dequantize(fmt, state["w"], case["n"], case["k"], case["experts"])
    if op.endswith("_train"):
        ys = _forward(state)
        return {"y": ys, "grads": torch.autograd.grad(ys, state["leaves"], state["dy"])}
    with torch.no_grad():
        return _merge(state) if op == "merge" else _forward(state)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct programs may lie apart
# ---------------------------------------------------------------------------
def _packed_bytes(fmt, elements):
    return elements * ((1 if fmt == "block_fp8" else 0.5) + SCALE_BYTES[fmt])


def work(case):
    op, fmt = case["op"], case["fmt"]
    if op in ("quantize", "dequantize"):
        elements = case["n"] * case["k"]
        return {"bytes": 2 * elements + _packed_bytes(fmt, elements), "flops": 0}
    r = case["r"]
    if op == "merge":
        n, k = case["n"], case["k"]
        out = 2 * n * k if case["publish"] else _packed_bytes(fmt, n * k)
        return {"bytes": _packed_bytes(fmt, n * k) + 4 * r * (n + k) + out, "flops": 2 * n * k * r}
    T, train = case["tokens"], op.endswith("_train")
    if op in ("moe_infer", "moe_train"):
        H, I, rows = case["hidden"], case["inter"], T * case["topk"]
        touched = min(case["experts"], rows)
        if rows < 8 * case["experts"]:            # a handful of rows: how many experts uneven routing touches on average
            p = torch.arange(1, case["experts"] + 1, dtype=torch.float64) ** -1.1
            touched = float((1 - (1 - p / p.sum()) ** rows).sum())
        factors = 3 * r * (H + I) * touched * 4
        flops = rows * (3 * 2 * H * I + 3 * 2 * r * (H + I))
        nbytes = _packed_bytes(fmt, 3 * H * I * touched) + factors + 2 * 2 * T * H + 10 * rows
        return {"bytes": nbytes + (2 * 2 * T * H + factors if train else 0),
                "flops": flops + (rows * (3 * 2 * H * I + 3 * 4 * r * (H + I)) if train else 0)}
    if op in ("linear_decode", "linear_train"):
        shapes, io = [(case["n"], case["k"])], case["n"] + case["k"]
    elif op in ("qkv_decode", "attention_train"):
        q, kv, k = case["q"], case["kv"], case["k"]
        shapes, io = [(q, k), (kv, k), (kv, k)], k + q + 2 * kv
        if train:
            shapes, io = shapes + [(k, q)], io + k + q
    else:
        H, I = case["hidden"], case["inter"]
        shapes, io = [(I, H), (I, H), (H, I)], 2 * H
    factors = 4 * r * sum(n + k for n, k in shapes)
    flops = sum(2.0 * T * n * k + 2.0 * T * r * (n + k) for n, k in shapes)
    nbytes = sum(_packed_bytes(fmt, n * k) for n, k in shapes) + factors + 2 * T * io
    if train:                                      # the other direction: dy in, dx out, factor gradients out
        nbytes += 2 * T * io + factors
        flops = sum(4.0 * T * n * k + 6.0 * T * r * (n + k) for n, k in shapes)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # codes, scales and decoded weights are defined bit for bit; so is the re-encoding, but of a low-rank product whose
    # summation order is free: a value on the boundary between two codes may take either
    if case["op"] in ("quantize", "dequantize"):
        return "exact"
    if case["op"] == "merge":
        return {"rel": 4e-3, "max": 0.15, "differ": 5e-3}
    # bf16 activations and intermediates, fp32 accumulation
    return {"rel": 1e-2, "max": 0.1}
