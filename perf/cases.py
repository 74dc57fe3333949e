"""The work that a user of this engine has it do, as cases that a timer can run.

* `linear`: one FPQuantLinear on a batch of tokens, rotation, quantization, GEMM and bias included: a token's
  decode step, the steps of a serving batch, a chunk of a prompt, a prefill;
* `block`: the engine's share of one decoder block whose producers are fused (fuse_producers): norms, projections,
  gated MLP and skip connections.  Attention over the cache is the model's own and left out: the query stands in for
  its result, and the new keys and values are outputs as a cache would take them;
* `quantize`: the rotate-and-quantize operator alone (what writes weights and calibrates activations);
* `operators`: the reference-named quantize and matmul operators one after the other on row-major tensors, as callers
  of the kernel package below the linear layer use them.

Layer sizes are those of the benchmark's workloads (hidden 4096, intermediate 14336 or 12288, 1024 key/value
features), or generic ones with ragged remainders.
"""
import math
import os
import sys

import torch
from torch import nn

sys.path.insert(0, os.path.abspath("fp-quant_amd"))

import fp_quant  # noqa: E402
from fp_quant.module import hip_ops, linear_fns  # noqa: E402
from fp_quant.utils import fuse_producers  # noqa: E402

LARGEST_TOKENS = 8192
LARGEST_LINEAR = 8192 * 4096 * 14336          # multiply-adds of the largest drawn linear layer
BLOCK_WEIGHTS = 4096 * (4096 + 2 * 1024 + 4096 + 3 * 14336)
LARGEST_BLOCK = 8192 * BLOCK_WEIGHTS


def listed():
    return [
        # one token through an attention output projection: latency, launches and host time
        dict(name="linear_mx_token", kind="linear", fmt="mxfp4", method="abs_max", init="hadamard", g=128,
             m=1, k=4096, n=4096, bias=False),
        # a serving batch of 32 sequences through a down-projection (few output features, a long K)
        dict(name="linear_mx_batch32_down", kind="linear", fmt="mxfp4", method="abs_max", init="hadamard", g=128,
             m=32, k=14336, n=4096, bias=False),
        # a serving batch of 128 sequences, or a short prompt, through an up-projection
        dict(name="linear_mx_batch128_up", kind="linear", fmt="mxfp4", method="abs_max", init="hadamard", g=128,
             m=128, k=4096, n=14336, bias=False),
        # a prompt of 2048 tokens through the same layer: the benchmark's headline workload
        dict(name="linear_mx_prefill_up", kind="linear", fmt="mxfp4", method="abs_max", init="hadamard", g=128,
             m=2048, k=4096, n=14336, bias=False),
        # a ragged layer (K no multiple of 256) with a bias, in the method that trained checkpoints use
        dict(name="linear_mx_ragged", kind="linear", fmt="mxfp4", method="quest", init="hadamard", g=64,
             m=333, k=3200, n=8640, bias=True),
        # a chunk of a prompt through an NVFP4 down-projection
        dict(name="linear_nv_chunk_down", kind="linear", fmt="nvfp4", method="abs_max", init="hadamard", g=16,
             m=512, k=12288, n=4096, bias=False),
        # a long prompt through an NVFP4 gate and up projection
        dict(name="linear_nv_prefill_gate_up", kind="linear", fmt="nvfp4", method="abs_max", init="hadamard", g=16,
             m=4096, k=4096, n=24576, bias=False),
        # one token through a fused decoder block
        dict(name="block_mx_token", kind="block", fmt="mxfp4", g=128, m=1, hidden=4096, kv=1024, inter=14336),
        # prefill of 4 prompts of 2048 tokens through the same block: the largest call
        dict(name="block_mx_prefill", kind="block", fmt="mxfp4", g=128, m=8192, hidden=4096, kv=1024, inter=14336),
        # the quantizer on a prompt's activations with outliers
        dict(name="quantize_mx", kind="quantize", fmt="mxfp4", method="abs_max", init="hadamard", g=128,
             m=2048, k=4096),
        # the quantizer on a long prompt's heavy-tailed activations
        dict(name="quantize_nv", kind="quantize", fmt="nvfp4", method="abs_max", init="hadamard", g=16,
             m=8192, k=4096),
        # quantize and matmul operators on row-major tensors: a serving batch through a q/k/v projection
        dict(name="operators_nv_batch64", kind="operators", fmt="nvfp4", method="abs_max", init="hadamard", g=16,
             m=64, k=4096, n=6144),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(value, of, least=1):
    return max(least, int(round(value / of))) * of


def _tokens(rng):
    m = _log_uniform(rng, 1, LARGEST_TOKENS)
    # a serving batch or a padded prompt is often a power of two
    return 1 << int(round(math.log2(m))) if rng.random() < 0.4 else m


def _format(rng, method=True):
    fmt = rng.choice(("mxfp4", "mxfp4", "nvfp4"))
    g = rng.choice((32, 64, 128, 128) if fmt == "mxfp4" else (16, 16, 32, 64, 128))
    out = dict(fmt=fmt, g=g)
    if method:
        out["method"] = rng.choice(("abs_max", "abs_max", "quest")) if fmt == "mxfp4" else "abs_max"
        out["init"] = rng.choice(("hadamard", "hadamard", "hadamard", "hadamard", "identity", "gsr"))
    return out


def _inner(rng, g, low, high):
    # most layers' inner dimensions are multiples of 256, the others of the rotation's size
    return _multiple(_log_uniform(rng, low, high), 256 if rng.random() < 0.7 else max(g, 32))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "block", "quantize", "operators"))
    if kind == "block":
        case = dict(kind=kind, **_format(rng, method=False))
        hidden = _multiple(_log_uniform(rng, 1024, 5120), rng.choice((128, 256, 256)))
        inter = _multiple(hidden * rng.uniform(2.5, 4.0), 256)
        kv = _multiple(hidden // rng.choice((1, 4, 8)), 128)
        weights = hidden * (2 * hidden + 2 * kv + 3 * inter)
        share = 1 if case["fmt"] == "mxfp4" else 3
        case.update(m=max(1, min(_tokens(rng), LARGEST_BLOCK // (share * weights))), hidden=hidden, kv=kv, inter=inter)
        return case
    case = dict(kind=kind, **_format(rng))
    k = _inner(rng, case["g"], 512, 14336)
    m = _tokens(rng)
    if kind == "quantize":
        case.update(m=m, k=k)
        return case
    n = _multiple(_log_uniform(rng, 256, 28672), rng.choice((256, 256, 32, 8)))
    ragged = k % 256 != 0 or kind == "operators"
    m = max(1, min(m, LARGEST_LINEAR // ((4 if ragged else 1) * (1 if case["fmt"] == "mxfp4" else 2) * n * k)))
    case.update(m=m, k=k, n=n)
    if kind == "linear":
        case["bias"] = rng.random() < 0.3
    return case


def _config(case):
    return fp_quant.FPQuantConfig(
        forward_dtype=fp_quant.FPQuantDtype.MXFP4 if case["fmt"] == "mxfp4" else fp_quant.FPQuantDtype.NVFP4,
        forward_method=case.get("method", "abs_max"), backward_dtype=fp_quant.FPQuantDtype.BF16,
        hadamard_group_size=case["g"], transform_init=case.get("init", "hadamard"))


def _linear(case, k, n, bias, gen):
    layer = fp_quant.FPQuantLinear(k, n, _config(case), bias=bias, device="cuda", dtype=torch.bfloat16)
    layer.weight.data = torch.randn(n, k, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.02)
    if bias:
        layer.bias.data = torch.randn(n, generator=gen, device="cuda", dtype=torch.bfloat16)
    layer.pre_forward()
    return layer


def _activations(case, m, k, gen):
    """Normal values with a few large outliers (MXFP4), or heavy-tailed ones, Student-t with 3 degrees of freedom
    (NVFP4)."""
    x = torch.randn(m, k, generator=gen, device="cuda")
    if case["fmt"] == "mxfp4":
        outliers = torch.rand(m, k, generator=gen, device="cuda") < 0.005
        return torch.where(outliers, x * 25, x).to(torch.bfloat16)
    chi2 = sum(torch.randn(m, k, generator=gen, device="cuda").square() for _ in range(3))
    return (x / (chi2 / 3).sqrt()).to(torch.bfloat16)


class BlockRMSNorm(nn.Module):
    def __init__(self, hidden, gen):
        super().__init__()
        self.weight = nn.Parameter((1 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")).to(torch.bfloat16))
        self.variance_epsilon = 1e-5

    def forward(self, hidden_states):
        x = hidden_states.float()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + self.variance_epsilon)
        return self.weight * x.to(hidden_states.dtype)


class BlockAttention(nn.Module):
    """The projections of an attention module; `cache` receives the new keys and values."""

    def __init__(self, case, gen):
        super().__init__()
        hidden, kv = case["hidden"], case["kv"]
        self.q_proj = _linear(case, hidden, hidden, False, gen)
        self.k_proj = _linear(case, hidden, kv, False, gen)
        self.v_proj = _linear(case, hidden, kv, False, gen)
        self.o_proj = _linear(case, hidden, hidden, False, gen)

    def forward(self, hidden_states, cache=None):
        query = self.q_proj(hidden_states)
        key = self.k_proj(hidden_states)
        value = self.v_proj(hidden_states)
        if cache is not None:
            cache.append((key, value))
        return self.o_proj(query), None


class BlockMLP(nn.Module):
    def __init__(self, case, gen):
        super().__init__()
        hidden, inter = case["hidden"], case["inter"]
        self.gate_proj = _linear(case, hidden, inter, False, gen)
        self.up_proj = _linear(case, hidden, inter, False, gen)
        self.down_proj = _linear(case, inter, hidden, False, gen)
        self.act_fn = nn.SiLU()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))


class Block(nn.Module):
    def __init__(self, case, gen):
        super().__init__()
        self.input_layernorm = BlockRMSNorm(case["hidden"], gen)
        self.self_attn = BlockAttention(case, gen)
        self.post_attention_layernorm = BlockRMSNorm(case["hidden"], gen)
        self.mlp = BlockMLP(case, gen)

    def forward(self, hidden_states, cache=None):
        residual = hidden_states
        hidden_states = self.input_layernorm(hidden_states)
        hidden_states, _ = self.self_attn(hidden_states=hidden_states, cache=cache)
        hidden_states = residual + hidden_states
        residual = hidden_states
        hidden_states = self.post_attention_layernorm(hidden_states)
        hidden_states = self.mlp(hidden_states)
        hidden_states = residual + hidden_states
        return hidden_states


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = dict(case)
    kind = case["kind"]
    if kind == "block":
        state["block"] = Block(case, gen)
        fuse_producers(state["block"])
        state["x"] = _activations(case, case["m"], case["hidden"], gen)
        return state
    state["x"] = _activations(case, case["m"], case["k"], gen)
    if kind == "quantize":
        # a layer's rotation and activation scale
        layer = _linear(case, case["k"], 32, False, gen)
        state["rotation"] = layer.forward_hadamard_matrix
        state["scale"] = layer.act_global_scale.float()
        return state
    layer = _linear(case, case["k"], case["n"], case.get("bias", False), gen)
    if kind == "linear":
        state["layer"] = layer
        return state
    state["rotation"] = layer.forward_hadamard_matrix
    state["scale"] = layer.act_global_scale.float()
    state["alpha"] = (1.0 / (layer.weight_global_scale * layer.act_global_scale)).float()
    state["qweight"], state["scales"] = layer.qweight, layer.scales
    return state


@torch.no_grad()
def run(state):
    x, kind = state["x"], state["kind"]
    if kind == "linear":
        return state["layer"](x.unsqueeze(0))
    if kind == "block":
        cache = []
        hidden = state["block"](x.unsqueeze(0), cache=cache)
        return (hidden, *cache[0])
    mx = state["fmt"] == "mxfp4"
    if mx:
        codes, scales, _ = hip_ops.fused_quantize_mx_op(x, state["rotation"], state["method"], False)
    else:
        codes, scales = hip_ops.fused_quantize_nv_op(x, state["rotation"], state["scale"])
    if kind == "quantize":
        return codes, scales.view(torch.uint8)
    dtype = fp_quant.FPQuantDtype.MXFP4 if mx else fp_quant.FPQuantDtype.NVFP4
    return linear_fns.forward_gemm(codes, state["qweight"], scales, state["scales"], state["alpha"], dtype)


def _weight_bytes(case, n, k):
    return n * k // 2 + n * k // (32 if case["fmt"] == "mxfp4" else 16)


def work(case):
    m, kind = case["m"], case["kind"]
    if kind == "block":
        hidden, kv, inter = case["hidden"], case["kv"], case["inter"]
        weights = hidden * (2 * hidden + 2 * kv + 3 * inter)
        return {"bytes": _weight_bytes(case, 1, weights) + 2 * m * (2 * hidden + 2 * kv), "flops": 2 * m * weights}
    k = case["k"]
    if kind == "quantize":
        group = 32 if case["fmt"] == "mxfp4" else 16
        return {"bytes": m * (2 * k + k // 2 + k // group), "flops": 2 * m * k}
    n = case["n"]
    return {"bytes": 2 * m * k + _weight_bytes(case, n, k) + 2 * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "block":
        # against the same block with torch's norms and products summed in fp64: 2.6e-3 and 0.21 (a statistic that rounds
        # the other way moves a bf16 value, and that a 4-bit code, of the next layer's input)
        return {"rel": 1e-2, "max": 0.8}
    # against sums in fp64, not rounded to bf16: 1.7e-3 and 0.004, with a bias 2.4e-3 and 0.0097
    return {"rel": 7e-3, "max": 0.03}
