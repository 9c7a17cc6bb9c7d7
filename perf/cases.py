"""What a user of kernl_amd has it do, as cases that can be timed and compared: whole models through `optimize_model`
and the operators of `kernl_amd.implementations` called directly.

Kinds of cases and the ranges they stand for (`draw` covers them; `listed` holds the sizes of the repository's own
configurations, tests and benchmark, and a few odd ones between them):

  encoder    BERT-base, fp16, `optimize_model`: batch 1 .. 32, 16 .. 512 tokens, full-length or padded
  prompt     decoder layers of Llama-2-7B width with the output head, fp16, `optimize_model`: causal prefill of one
             prompt of 32 .. 2048 tokens
  decode     one decoding step of such layers, the operators called one after the other: 1 .. 32 sequences over caches
             of 128 .. 4096 positions, fp16 or bf16
  attention  `attention_forward`: head size 64 or 128, 64 .. 2048 positions, no mask / padding mask / causal, fp16 or bf16
  linear     `linear_layer`: 1 .. 16384 rows against the weights of the two models, with and without activation
  norm       `layer_norm`: LayerNorm or RMSNorm, 1 .. 65536 rows of 768 or 4096
"""
import torch
from transformers import BertConfig, BertModel, LlamaConfig, LlamaForCausalLM

from kernl_amd.implementations.attention import attention_forward
from kernl_amd.implementations.attention_skinny import skinny_attention_forward
from kernl_amd.implementations.layer_norm import layer_norm
from kernl_amd.implementations.linear_layer import decode_linear_layer, interleave_glu_rows, linear_layer, rms_linear_layer
from kernl_amd.model_optimization import optimize_model

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

# BERT-base
VOCAB, WIDTH, HEADS, FFN, LAYERS, TYPES = 30522, 768, 12, 3072, 12, 2
# decoder of Llama-2-7B width, four layers deep
D_VOCAB, D_WIDTH, D_HEADS, D_HEAD, D_FFN, D_LAYERS, D_EPS = 32000, 4096, 32, 128, 11008, 4, 1e-5

# [out features, in features] of the projections of the two models
WEIGHTS = [(2304, 768), (768, 768), (3072, 768), (768, 3072), (12288, 4096), (4096, 4096), (4096, 11008)]


def listed():
    return [
        # one short sentence: a query encoder answering a single request, bounded by latency
        {"name": "encoder_b1_s16", "kind": "encoder", "batch": 1, "seq": 16, "padded": False},
        # a handful of sentences of unequal length, the longest of an odd size
        {"name": "encoder_b3_s77_padded", "kind": "encoder", "batch": 3, "seq": 77, "padded": True},
        # an ordinary server batch
        {"name": "encoder_b8_s128", "kind": "encoder", "batch": 8, "seq": 128, "padded": False},
        # offline encoding of documents: the benchmark's end-to-end size
        {"name": "encoder_b32_s512_padded", "kind": "encoder", "batch": 32, "seq": 512, "padded": True},
        # time to the first token of a chat turn, an odd number of tokens
        {"name": "prompt_s333", "kind": "prompt", "seq": 333},
        # the same for a long document: the benchmark's prompt length
        {"name": "prompt_s2048", "kind": "prompt", "seq": 2048},
        # a single user's generation: every weight is read for one token
        {"name": "decode_b1_n700", "kind": "decode", "dtype": "fp16", "batch": 1, "cache": 700},
        # a server's generation, many sequences over long caches
        {"name": "decode_b24_n3000", "kind": "decode", "dtype": "bf16", "batch": 24, "cache": 3000},
        # attention of an encoder batch with the padding mask such a batch comes with: the benchmark's headline
        {"name": "attention_b32_h12_s512_d64_padding", "kind": "attention", "dtype": "fp16", "batch": 32, "heads": 12, "seq": 512,
         "head": 64, "mask": "padding"},
        # causal attention of two prompts in a decoder written around the operators, an odd length
        {"name": "attention_b2_h16_s1111_d128_causal", "kind": "attention", "dtype": "bf16", "batch": 2, "heads": 16, "seq": 1111,
         "head": 128, "mask": "causal"},
        # feed-forward entry of an encoder batch: the benchmark's fused linear layer
        {"name": "linear_16384_3072x768_gelu", "kind": "linear", "dtype": "fp16", "rows": 16384, "out": 3072, "in": 768,
         "activation": "fast_gelu"},
        # the norm between the blocks of such a batch, also the benchmark's
        {"name": "norm_16384_768", "kind": "norm", "dtype": "fp16", "rows": 16384, "width": 768, "rms": False},
    ]


def _log_int(rng, low, high):
    return min(high, int(low * (high / low) ** rng.random() * (1 + 1e-9) + 0.5))


def draw(rng):
    kind = rng.choice(["encoder"] * 4 + ["prompt"] * 2 + ["decode"] * 2 + ["attention"] * 2 + ["linear", "norm"])
    if kind == "encoder":
        return {"kind": kind, "batch": _log_int(rng, 1, 32), "seq": _log_int(rng, 16, 512), "padded": rng.random() < 0.5}
    if kind == "prompt":
        return {"kind": kind, "seq": _log_int(rng, 32, 2048)}
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "decode":
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 1, 32), "cache": _log_int(rng, 128, 4096)}
    if kind == "attention":
        head, mask = rng.choice([64, 128]), rng.choice(["none", "padding", "causal"])
        seq = _log_int(rng, 64, 2048)
        batch = _log_int(rng, 1, max(1, min(32, (1 << 24) // (seq * seq // 2 + 1))))
        return {"kind": kind, "dtype": dtype, "batch": batch, "heads": 12 if head == 64 else 16, "seq": seq, "head": head, "mask": mask}
    if kind == "linear":
        n, k = rng.choice(WEIGHTS)
        return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 1, 16384 if k == 768 or n == 768 else 2048), "out": n, "in": k,
                "activation": rng.choice(["", "", "gelu", "fast_gelu"])}
    return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 1, 65536 if dtype == "fp16" else 16384), "width": rng.choice([768, 4096]),
            "rms": rng.random() < 0.5}


# ---- models and weights a program loads once and then serves every request with

_LOADED = {}


def _encoder_model():
    if "encoder" not in _LOADED:
        torch.manual_seed(0)
        cfg = BertConfig()
        cfg._attn_implementation = "eager"
        with torch.device(DEVICE):
            model = BertModel(cfg).eval().half()
        optimize_model(model)
        _LOADED["encoder"] = model
    return _LOADED["encoder"]


def _prompt_model():
    if "prompt" not in _LOADED:
        torch.manual_seed(0)
        cfg = LlamaConfig(num_hidden_layers=D_LAYERS, hidden_size=D_WIDTH, num_attention_heads=D_HEADS, num_key_value_heads=D_HEADS,
                          intermediate_size=D_FFN, vocab_size=D_VOCAB, rms_norm_eps=D_EPS, max_position_embeddings=4096,
                          rope_theta=10000.0, initializer_range=0.02, tie_word_embeddings=False)
        cfg._attn_implementation = "sdpa"
        before = torch.get_default_dtype()
        torch.set_default_dtype(torch.float16)
        try:
            with torch.device(DEVICE):
                model = LlamaForCausalLM(cfg).eval()
        finally:
            torch.set_default_dtype(before)
        optimize_model(model)
        _LOADED["prompt"] = model
    return _LOADED["prompt"]


def _decode_weights(dtype):
    """Weights of the decoder layers, laid out once for the fused projections, and the rotary tables."""
    key = ("decode", dtype)
    if key not in _LOADED:
        gen = torch.Generator(DEVICE).manual_seed(0)

        def weight(n, k):
            return (torch.randn((n, k), generator=gen, device=DEVICE) * 0.02).to(dtype)

        layers = []
        for _ in range(D_LAYERS):
            layers.append({
                "norm_1": (1 + 0.1 * torch.randn((D_WIDTH,), generator=gen, device=DEVICE)).to(dtype),
                "norm_2": (1 + 0.1 * torch.randn((D_WIDTH,), generator=gen, device=DEVICE)).to(dtype),
                "qkv": weight(3 * D_WIDTH, D_WIDTH),
                "out": weight(D_WIDTH, D_WIDTH),
                "gate_up": interleave_glu_rows(weight(D_FFN, D_WIDTH), weight(D_FFN, D_WIDTH)),
                "down": weight(D_WIDTH, D_FFN),
            })
        angle = torch.outer(torch.arange(4097).float(), 1.0 / (10000.0 ** (torch.arange(0, D_HEAD, 2).float() / D_HEAD)))
        table = torch.cat((angle, angle), dim=-1)[None].to(DEVICE)
        _LOADED[key] = (layers, table.cos().to(dtype), table.sin().to(dtype))
    return _LOADED[key]


# ---- inputs

def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(DEVICE).manual_seed(seed)

    def normal(*shape, std=1.0, dtype=None):
        return (torch.randn(shape, generator=gen, device=DEVICE) * std).to(dtype or DTYPES[case["dtype"]])

    def lengths(batch, seq):
        return torch.randint((seq + 1) // 2, seq + 1, (batch, 1), generator=gen, device=DEVICE)

    if kind == "encoder":
        shape = (case["batch"], case["seq"])
        ids = torch.randint(0, VOCAB, shape, generator=gen, device=DEVICE)
        valid = torch.ones_like(ids)
        if case["padded"]:
            valid = (torch.arange(shape[1], device=DEVICE)[None, :] < lengths(*shape)).long()
        return {"kind": kind, "model": _encoder_model(), "ids": ids, "valid": valid}
    if kind == "prompt":
        ids = torch.randint(0, D_VOCAB, (1, case["seq"]), generator=gen, device=DEVICE)
        return {"kind": kind, "model": _prompt_model(), "ids": ids}
    if kind == "decode":
        dtype, batch, n = DTYPES[case["dtype"]], case["batch"], case["cache"]
        layers, cos, sin = _decode_weights(dtype)
        # caches hold the positions before this step; the step adds one more
        caches = [tuple(normal(batch, D_HEADS, n + 1, D_HEAD) for _ in range(2)) for _ in range(D_LAYERS)]
        return {"kind": kind, "layers": layers, "cos": cos[:, n:n + 1], "sin": sin[:, n:n + 1], "caches": caches, "position": n,
                "hidden": normal(batch, 1, D_WIDTH)}
    if kind == "attention":
        batch, seq, shape = case["batch"], case["seq"], (case["batch"], case["heads"], case["seq"], case["head"])
        mask = None
        if case["mask"] == "padding":
            beyond = torch.arange(seq, device=DEVICE)[None, :] >= lengths(batch, seq)
            mask = torch.zeros((batch, seq), device=DEVICE).masked_fill_(beyond, float("-inf"))[:, None, None, :]
        q, k, v = normal(*shape), normal(*shape), normal(*shape)
        return {"kind": kind, "q": q, "k": k, "v": v, "mask": mask, "causal": case["mask"] == "causal", "scale": case["head"] ** -0.5}
    if kind == "linear":
        return {"kind": kind, "x": normal(case["rows"], case["in"]), "weight": normal(case["out"], case["in"], std=0.02),
                "bias": normal(case["out"], std=0.02), "activation": case["activation"]}
    width = case["width"]
    return {"kind": kind, "x": normal(case["rows"], width), "weight": 1 + normal(width, std=0.1),
            "bias": None if case["rms"] else normal(width, std=0.1), "rms": case["rms"]}


# ---- one pass

def _decode_step(state):
    x, position = state["hidden"], state["position"]
    batch = x.shape[0]
    for layer, (keys, values) in zip(state["layers"], state["caches"]):
        qkv = decode_linear_layer(x, layer["qkv"], None, layer["norm_1"], D_EPS, None, state["cos"], state["sin"],
                                  head_dim=D_HEAD, rope_cols=2 * D_WIDTH)
        q, k, v = qkv.view(batch, 1, 3, D_HEADS, D_HEAD).permute(2, 0, 3, 1, 4)
        keys[:, :, position:position + 1] = k
        values[:, :, position:position + 1] = v
        mixed = torch.empty((batch, 1, D_HEADS, D_HEAD), dtype=x.dtype, device=x.device).transpose(1, 2)
        skinny_attention_forward(q, keys, values, mixed, D_HEAD ** -0.5)
        x = decode_linear_layer(mixed.transpose(1, 2).reshape(batch, 1, D_WIDTH), layer["out"], residual=x)
        inner = rms_linear_layer(x, layer["norm_2"], D_EPS, layer["gate_up"], None, "silu", gated=True)
        x = decode_linear_layer(inner, layer["down"], residual=x)
    return x


def run(state):
    kind = state["kind"]
    with torch.inference_mode():
        if kind == "encoder":
            out = state["model"](input_ids=state["ids"], attention_mask=state["valid"])
            return [out.last_hidden_state, out.pooler_output]
        if kind == "prompt":
            return state["model"](input_ids=state["ids"], use_cache=False).logits
        if kind == "decode":
            hidden = _decode_step(state)
            at = state["position"]
            new = [cache[:, :, at] for pair in state["caches"] for cache in pair]
            return [hidden] + new
        if kind == "attention":
            out = torch.empty_like(state["q"])
            return attention_forward(state["q"], state["k"], state["v"], out, state["scale"], state["causal"], state["mask"])
        if kind == "linear":
            return linear_layer(state["x"], state["weight"], state["bias"], state["activation"])
        return layer_norm(state["x"], state["weight"], state["bias"], 1e-5 if state["rms"] else 1e-12, use_rms_norm=state["rms"])


# ---- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "encoder":
        rows, keys = case["batch"] * case["seq"], case["seq"] * (0.75 if case["padded"] else 1.0)
        weights = LAYERS * (4 * WIDTH * WIDTH + 2 * WIDTH * FFN + 9 * WIDTH + FFN) + WIDTH * (WIDTH + 1) + WIDTH * (case["seq"] + TYPES)
        flops = LAYERS * (2 * rows * (4 * WIDTH * WIDTH + 2 * WIDTH * FFN) + 4 * rows * keys * WIDTH) + 2 * case["batch"] * WIDTH * WIDTH
        return {"bytes": 2 * (weights + min(rows, VOCAB) * WIDTH + rows * WIDTH + case["batch"] * WIDTH) + 16 * rows, "flops": flops}
    if kind == "prompt":
        seq = case["seq"]
        layer = 4 * D_WIDTH * D_WIDTH + 3 * D_WIDTH * D_FFN
        weights = D_LAYERS * (layer + 2 * D_WIDTH) + D_WIDTH + D_VOCAB * D_WIDTH
        flops = D_LAYERS * (2 * seq * layer + 2 * seq * (seq + 1) * D_WIDTH) + 2 * seq * D_VOCAB * D_WIDTH
        return {"bytes": 2 * (weights + seq * D_WIDTH + seq * D_VOCAB) + 8 * seq, "flops": flops}
    if kind == "decode":
        batch, n = case["batch"], case["cache"] + 1
        layer = 4 * D_WIDTH * D_WIDTH + 3 * D_WIDTH * D_FFN
        return {"bytes": D_LAYERS * 2 * (layer + 2 * D_WIDTH + 2 * batch * n * D_WIDTH) + 4 * batch * D_WIDTH,
                "flops": D_LAYERS * (2 * batch * layer + 4 * batch * n * D_WIDTH)}
    if kind == "attention":
        cells = case["batch"] * case["heads"] * case["seq"] * case["head"]
        keys = {"none": case["seq"], "padding": 0.75 * case["seq"], "causal": (case["seq"] + 1) / 2}[case["mask"]]
        mask = 4 * case["batch"] * case["seq"] if case["mask"] == "padding" else 0
        return {"bytes": 2 * 4 * cells + mask, "flops": 4 * cells * keys}
    if kind == "linear":
        m, n, k = case["rows"], case["out"], case["in"]
        return {"bytes": 2 * (m * k + n * k + n + m * n), "flops": 2 * m * n * k}
    return {"bytes": 2 * (2 * case["rows"] * case["width"] + 2 * case["width"]), "flops": 8 * case["rows"] * case["width"]}


def tolerance(case):
    """Inputs, weights and results are 16-bit with fp32 sums: one operator rounds its result (and attention its
    probabilities) once, a model rounds its hidden states some ten times a layer."""
    if case["kind"] in ("encoder", "prompt"):
        return {"rel": 1e-2}
    if case["kind"] == "decode":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3, "max": 0.1}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3}
