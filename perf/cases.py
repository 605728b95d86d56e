"""What a user of the package has it do, as cases that can be timed: the whole-model passes of a quantized Llama
(a decode step, a prompt), single kernel-mode Linears from one activation row to a long prompt, a
Mixture-of-Experts block, and the group quantizer. Everything goes through the public entry points
(`llmquant.oneshot`, `llmquant.runtime.KernelDecoder`, `KernelQuantLinear`, `KernelQuantExperts`,
`fake_quantize_hip`). Weights and inputs are random at the shapes of the Llama-3.2-1B, Llama-3-8B and
OLMoE-1B-7B layers that the benchmark and the tests use.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import torch
import torch.nn as nn

_PACKAGE = os.path.join(os.getcwd(), "llm-quant_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

GROUP = 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

#: (hidden, intermediate, head_dim, layers taken): both architectures have 32 query and 8 key/value heads and a
#: vocabulary of 128256. A few of the 16 / 32 layers are enough to run the launches of a layer on weights that do not
#: stay in a cache, beside the embedding and the lm_head, and keep a case's preparation short.
MODELS = {"1b": (2048, 8192, 64, 4), "8b": (4096, 14336, 128, 2)}
VOCAB, Q_HEADS, KV_HEADS = 128256, 32, 8

#: the Linears of those models: (out, in, head_dim of the output, head_dim of the input); an output head shares one
#: scale per group, an input head is padded to whole groups
LINEARS = {
    "1b_q": (2048, 2048, 64, 0), "1b_kv": (512, 2048, 64, 0), "1b_o": (2048, 2048, 0, 64),
    "1b_gate": (8192, 2048, 0, 0), "1b_down": (2048, 8192, 0, 0), "1b_head": (128256, 2048, 0, 0),
    "8b_q": (4096, 4096, 128, 0), "8b_kv": (1024, 4096, 128, 0), "8b_o": (4096, 4096, 0, 128),
    "8b_gate": (14336, 4096, 0, 0), "8b_down": (4096, 14336, 0, 0), "8b_head": (128256, 4096, 0, 0),
}

#: (experts, experts a token is routed to, hidden, intermediate): the OLMoE-1B-7B block, and a block of few, wider
#: experts
BLOCKS = {"64of8": (64, 8, 2048, 1024), "8of2": (8, 2, 2048, 4096)}

#: no drawn case does more than this (the prompt-sized 8B gate projection, the largest listed case)
MOST_FLOPS = 2.0 * 2048 * 14336 * 4096
MOST_BYTES = 700e6


def listed():
    return [
        # one token of a chat: the step that generation replays, at an ordinary context
        dict(name="decode_step_600", kind="step", model="1b", cached=600, kv_bits=8),
        # the same far into a long document: the attention over the cache is what counts
        dict(name="decode_step_24000", kind="step", model="1b", cached=24000, kv_bits=8),
        # time to first token: an ordinary prompt of no particular length, and the first token after it
        dict(name="prompt_500", kind="prompt", model="1b", tokens=500, kv_bits=8),
        # one row through the smallest Linear of a decoder layer: what a module-by-module decode calls most
        dict(name="linear_1_1b_q", kind="linear", layer="1b_q", rows=1, bits=8, act=16, dtype="bf16"),
        # one row through lm_head: the largest single stream of a decode step
        dict(name="linear_1_1b_head", kind="linear", layer="1b_head", rows=1, bits=8, act=16, dtype="bf16"),
        # a small batch of sequences, each at its next token
        dict(name="linear_16_8b_gate", kind="linear", layer="8b_gate", rows=16, bits=4, act=16, dtype="bf16"),
        # a short prompt in fp16, ragged in rows, through the longest reduction
        dict(name="linear_333_8b_down", kind="linear", layer="8b_down", rows=333, bits=4, act=16, dtype="f16"),
        # a long prompt through the widest projection
        dict(name="linear_2048_8b_gate", kind="linear", layer="8b_gate", rows=2048, bits=4, act=16, dtype="bf16"),
        # the same projection with 8-bit activations (W4A8) on an ordinary prompt
        dict(name="linear_512_8b_gate_a8", kind="linear", layer="8b_gate", rows=512, bits=4, act=8, dtype="bf16"),
        # one token through the experts of a layer
        dict(name="experts_1", kind="experts", block="64of8", tokens=1, bits=4, dtype="bf16"),
        # a prompt through the experts of a layer
        dict(name="experts_300", kind="experts", block="64of8", tokens=300, bits=4, dtype="bf16"),
        # what an accuracy study calls on every weight: quantize-dequantize, with a last axis that is no whole
        # number of groups
        dict(name="fake_quant_ragged", kind="fake", rows=4096, width=5000, bits=4, strategy="group", dtype="bf16"),
    ]


def _spread(rng, low, high):
    """A whole number from low to high, even over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    while True:
        kind = rng.choice(["step", "prompt", "linear", "linear", "linear", "linear", "experts", "experts", "fake"])
        if kind == "step":
            case = dict(kind=kind, model=rng.choice(["1b", "1b", "8b"]), cached=_spread(rng, 40, 24000),
                        kv_bits=rng.choice([8, 8, 4]))
        elif kind == "prompt":
            case = dict(kind=kind, model=rng.choice(["1b", "1b", "8b"]), tokens=_spread(rng, 30, 1100),
                        kv_bits=rng.choice([8, 8, 4]))
        elif kind == "linear":
            case = dict(kind=kind, layer=rng.choice(sorted(LINEARS)), rows=_spread(rng, 1, 2048),
                        bits=rng.choice([4, 8]), act=rng.choice([16, 16, 16, 8]),
                        dtype=rng.choice(["bf16", "bf16", "f16"]))
        elif kind == "experts":
            case = dict(kind=kind, block=rng.choice(["64of8", "64of8", "8of2"]), tokens=_spread(rng, 1, 600),
                        bits=rng.choice([4, 4, 8]), dtype=rng.choice(["bf16", "bf16", "f16"]))
        else:
            strategy = rng.choice(["group", "group", "channel"])
            case = dict(kind=kind, rows=_spread(rng, 16, 8192), width=_spread(rng, 256, 14336),
                        bits=rng.choice([4, 8]), strategy=strategy, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
        need = work(case)
        if need["flops"] <= MOST_FLOPS and need["bytes"] <= MOST_BYTES:
            return case


# ---- what a user's program has in hand before the call -----------------------------------------------------------
class CaseRMSNorm(nn.Module):
    def __init__(self, width, eps=1e-5):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(width))
        self.variance_epsilon = eps

    def forward(self, x):
        wide = x.float()
        wide = wide * torch.rsqrt(wide.pow(2).mean(-1, keepdim=True) + self.variance_epsilon)
        return self.weight * wide.to(x.dtype)


def _modules(**children):
    owner = nn.Module()
    for name, child in children.items():
        setattr(owner, name, child)
    return owner


def _llama(name):
    """A module tree of the Llama shape (what the runtimes walk: its forward is never called)."""
    hidden, inter, head_dim, layers = MODELS[name]
    linear = lambda n, k: nn.Linear(k, n, bias=False)  # noqa: E731

    def layer():
        attn = _modules(q_proj=linear(Q_HEADS * head_dim, hidden), k_proj=linear(KV_HEADS * head_dim, hidden),
                        v_proj=linear(KV_HEADS * head_dim, hidden), o_proj=linear(hidden, Q_HEADS * head_dim))
        mlp = _modules(gate_proj=linear(inter, hidden), up_proj=linear(inter, hidden), down_proj=linear(hidden, inter),
                       act_fn=nn.SiLU())
        return _modules(self_attn=attn, mlp=mlp, input_layernorm=CaseRMSNorm(hidden),
                        post_attention_layernorm=CaseRMSNorm(hidden))

    rope = nn.Module()
    rope.register_buffer("inv_freq", 500000.0 ** (-torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim),
                         persistent=False)
    rope.attention_scaling = 1.0
    body = _modules(embed_tokens=nn.Embedding(VOCAB, hidden), layers=nn.ModuleList(layer() for _ in range(layers)),
                    norm=CaseRMSNorm(hidden), rotary_emb=rope)
    model = _modules(model=body, lm_head=linear(VOCAB, hidden))
    model.config = SimpleNamespace(hidden_size=hidden, num_attention_heads=Q_HEADS, num_key_value_heads=KV_HEADS,
                                   head_dim=head_dim, num_hidden_layers=layers, vocab_size=VOCAB)
    return model


def _quantized_llama(name, gen):
    """The model with random weights in bf16, quantized as the benchmark's recipe does: attention int8, MLP int4,
    lm_head int8."""
    from llmquant import QuantConfig, oneshot

    with torch.device("meta"):
        model = _llama(name)
    inv_freq = 500000.0 ** (-torch.arange(0, model.config.head_dim, 2, dtype=torch.float32) / model.config.head_dim)
    model = model.to(torch.bfloat16).to_empty(device="cuda").eval()
    model.model.rotary_emb.inv_freq = inv_freq.cuda()
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.02, generator=gen) if p.dim() > 1 else p.fill_(1.0)
    recipe = QuantConfig(attn_weight="int8", mlp_weight="int4", head_weight="int8", kv_cache="int8")
    return oneshot(model, recipe.to_modifier("kernel"))


def _linear(case, gen):
    from dataclasses import replace

    from llmquant.core.scheme import QuantizationScheme, preset_name_to_scheme
    from llmquant.quantizers import KernelQuantLinear

    n, k, out_head, in_head = LINEARS[case["layer"]]
    scheme = preset_name_to_scheme(f"W{case['bits']}A{case['act']}")
    weights, acts = scheme.weights, scheme.input_activations
    if out_head:
        weights = replace(weights, out_group=out_head)
    if in_head:
        weights = replace(weights, head_dim=in_head)
        acts = replace(acts, head_dim=in_head) if acts else None
    float_layer = nn.Linear(k, n, bias=False, device="meta").to_empty(device="cuda").to(DTYPES[case["dtype"]])
    with torch.no_grad():
        float_layer.weight.normal_(0.0, 0.02, generator=gen)
    return KernelQuantLinear.from_linear(float_layer, QuantizationScheme(weights=weights, input_activations=acts))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + 17)
    kind = case["kind"]
    if kind in ("step", "prompt"):
        from llmquant.runtime import KernelDecoder

        tokens = case["cached"] if kind == "step" else case["tokens"]
        model = _quantized_llama(case["model"], gen)
        ids = torch.randint(0, VOCAB, (1, tokens + 1), device="cuda", generator=gen)
        decoder = KernelDecoder(model, tokens, 256, kv_bits=case["kv_bits"])
        # a server captures its step once, and has seen a prompt by then; for a step case the cache is what that
        # prompt left
        decoder.prefill(ids[:, :tokens])
        decoder.capture(tokens, ids[:, tokens])
        return dict(kind=kind, decoder=decoder, ids=ids[:, :tokens].contiguous(), token=ids[:, tokens].contiguous(),
                    tokens=tokens)
    dtype = DTYPES[case["dtype"]]
    if kind == "linear":
        layer = _linear(case, gen)
        x = torch.randn(case["rows"], layer.in_features, device="cuda", generator=gen).to(dtype)
        return dict(kind=kind, layer=layer, x=x)
    if kind == "experts":
        from llmquant.core.scheme import preset_name_to_scheme
        from llmquant.quantizers import KernelQuantExperts

        experts, top_k, hidden, inter = BLOCKS[case["block"]]
        source = SimpleNamespace(act_fn=nn.SiLU())
        for name, shape in (("gate_up_proj", (experts, 2 * inter, hidden)), ("down_proj", (experts, hidden, inter))):
            weight = torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, 0.02, generator=gen)
            setattr(source, name, nn.Parameter(weight, requires_grad=False))
        block = KernelQuantExperts.from_experts(source, preset_name_to_scheme(f"W{case['bits']}A16"))
        x = torch.randn(case["tokens"], hidden, device="cuda", generator=gen).to(dtype)
        # a router prefers some experts to others
        scores = (torch.randn(case["tokens"], experts, device="cuda", generator=gen)
                  + 0.5 * torch.randn(1, experts, device="cuda", generator=gen)).softmax(-1)
        weights, index = scores.topk(top_k, dim=-1)
        return dict(kind=kind, block=block, x=x, index=index, weights=weights.to(dtype))
    from llmquant.core.scheme import QuantizationArgs

    args = QuantizationArgs(num_bits=case["bits"], strategy=case["strategy"],
                            group_size=GROUP if case["strategy"] == "group" else None)
    weight = torch.empty(case["rows"], case["width"], device="cuda").normal_(0.0, 0.02, generator=gen).to(dtype)
    return dict(kind=kind, args=args, weight=weight)


# ---- one pass ------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "step":
        # the next token of a sequence whose cache holds `tokens` (a caller that scores, drafts or constrains feeds
        # its own token): the logits, and the scales of the cache rows, the new one among them. (The codes beside them
        # are rounded from 16-bit values and flip wherever such a value does.)
        decoder = state["decoder"]
        decoder.step(state["token"], state["tokens"])
        return dict(logits=decoder.logits, k_scale=decoder.runtime.cache.k_scale, v_scale=decoder.runtime.cache.v_scale)
    if kind == "prompt":
        # a prompt, then the first step after it, from a token that the caller fixes (a reply that has to begin with
        # it): the logits depend on every cache row that the prompt wrote
        decoder = state["decoder"]
        decoder.prefill(state["ids"])
        decoder.capture(state["tokens"], state["token"])
        decoder.step()
        return dict(logits=decoder.logits, k_scale=decoder.runtime.cache.k_scale, v_scale=decoder.runtime.cache.v_scale)
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "experts":
        return state["block"](state["x"], state["index"], state["weights"])
    from llmquant.hip import fake_quantize_hip

    return fake_quantize_hip(state["weight"], state["args"], return_scale=True)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _weight_bytes(n, k, bits, scale_rows=None):
    return n * k * bits / 8 + (scale_rows or n) * math.ceil(k / GROUP) * 4


def work(case):
    kind = case["kind"]
    if kind in ("step", "prompt"):
        hidden, inter, head_dim, layers = MODELS[case["model"]]
        rows = 1 if kind == "step" else case["tokens"]
        qkv = (Q_HEADS + 2 * KV_HEADS) * head_dim
        per_layer = (_weight_bytes(qkv, hidden, 8, qkv // head_dim) + _weight_bytes(hidden, Q_HEADS * head_dim, 8)
                     + _weight_bytes(2 * inter, hidden, 4) + _weight_bytes(hidden, inter, 4))
        head = _weight_bytes(VOCAB, hidden, 8) + VOCAB * 2
        row = 2 * KV_HEADS * (head_dim * case["kv_bits"] / 8 + 4)         # a cached token of one layer
        matmuls = 2.0 * (qkv * hidden + hidden * Q_HEADS * head_dim + 3 * inter * hidden)
        cached = case["cached"] + 1 if kind == "step" else case["tokens"] + 1
        step_flops = layers * (matmuls + 4.0 * cached * Q_HEADS * head_dim) + 2.0 * VOCAB * hidden
        step_bytes = layers * (per_layer + cached * row) + head
        if kind == "step":
            return dict(bytes=step_bytes, flops=step_flops)
        # the prompt reads the weights once and writes the cache, lm_head sees its last row; then the step
        attention = 4.0 * Q_HEADS * head_dim * rows * (rows + 1) / 2
        return dict(bytes=2 * step_bytes + rows * hidden * 2,
                    flops=layers * (rows * matmuls + attention) + 2.0 * VOCAB * hidden + step_flops)
    size = 4 if case["dtype"] == "f32" else 2
    if kind == "linear":
        n, k, out_head, _ = LINEARS[case["layer"]]
        rows = case["rows"]
        return dict(bytes=_weight_bytes(n, k, case["bits"], n // out_head if out_head else n) + rows * (n + k) * size,
                    flops=2.0 * rows * n * k)
    if kind == "experts":
        experts, top_k, hidden, inter = BLOCKS[case["block"]]
        hit = experts * (1 - (1 - top_k / experts) ** case["tokens"])      # experts that some token is routed to
        weights = _weight_bytes(2 * inter, hidden, case["bits"]) + _weight_bytes(hidden, inter, case["bits"])
        return dict(bytes=hit * weights + case["tokens"] * (2 * hidden * size + top_k * (8 + size)),
                    flops=2.0 * case["tokens"] * top_k * 3 * hidden * inter)
    values = case["rows"] * case["width"]
    groups = case["rows"] * (math.ceil(case["width"] / GROUP) if case["strategy"] == "group" else 1)
    return dict(bytes=values * 2 * size + groups * 4, flops=0)


def tolerance(case):
    kind = case["kind"]
    if kind == "fake" or (kind == "linear" and case["act"] == 8):
        # the quantizer is bit-exact, and integer activations keep the rounding points of the group-by-group form
        return "exact"
    # 16-bit values: about four times what two implementations with the same rounding points but another order of the
    # sums, or with the weight rounded to 16 bits before the product, were measured to differ by
    wide = case.get("dtype") == "f16"
    if kind in ("step", "prompt"):
        return {"rel": 0.03, "max": 0.25}       # the fused step against the module walk: 1.2e-2 and 6e-2
    if kind == "experts":                       # against fp32 throughout: 6e-3 and 4e-2, in fp16 6e-4 and 4e-3
        return {"rel": 2.5e-3, "max": 0.016} if wide else {"rel": 0.02, "max": 0.16}
    return {"rel": 1.2e-3, "max": 6e-3} if wide else {"rel": 1e-2, "max": 0.05}     # 3e-4 and 2e-3; 2.5e-3 and 1.2e-2
