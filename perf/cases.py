"""The work a program that serves INT8 OPT models gives this package, as cases that can be timed and compared.

Four kinds, each through public entry points:

* ``prefill``: ``Int8OPTModel`` on a batch of prompts (the decoder stack of ``benchmark/bench_opt.py``), with the KV
  caches that decoding needs; with equal prompts or a padded batch, fp32 or fp16 residual stream.
* ``generate``: ``Int8OPTForCausalLM``, eight greedy tokens after a cached prompt.
* ``linear``: one W8A8 layer of ``torch_int.nn.linear``.
* ``attention_products``: ``BMM_S8T_S8N_F32T`` (scores) and ``BMM_S8T_S8N_S8T`` (context) for callers that run the
  softmax between them themselves.
* ``dq_add_layernorm_q``: the fused dequantise + residual + LayerNorm + quantise operator.

Weights and activations are drawn as rounded normal values: a weight quantised by its largest magnitude has a standard
deviation of some 20 steps, and the scales below keep every activation tensor at some 30 steps, as calibrated models do.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "torch-int_amd"))

import torch_int._CUDA as ops  # noqa: E402
from torch_int.models.opt import Int8OPTForCausalLM, OPTConfigLite  # noqa: E402
from torch_int.nn.bmm import BMM_S8T_S8N_F32T, BMM_S8T_S8N_S8T  # noqa: E402
from torch_int.nn.linear import (W8A8B8O8Linear, W8A8B8O8LinearReLU, W8A8B32O32Linear,  # noqa: E402
                                 W8A8B32O32LinearWithoutScaling, W8A8BFP32OFP32Linear)

DEV = "cuda:0"
# hidden size, heads, layers of the stack that is run: all of them up to 1.3B, a stage of 12 or 16 beyond
MODELS = {"opt-125m": (768, 12, 12), "opt-1.3b": (2048, 32, 24), "opt-2.7b": (2560, 32, 16),
          "opt-6.7b": (4096, 32, 16), "opt-13b": (5120, 40, 12)}
VOCAB = 50272
NEW_TOKENS = 8
DTYPES = {"fp32": torch.float32, "fp16": torch.float16}
LINEARS = {"b8_o8": W8A8B8O8Linear, "relu_b8_o8": W8A8B8O8LinearReLU, "b32_o32": W8A8B32O32LinearWithoutScaling,
           "b32_o32_scaled": W8A8B32O32Linear, "bfp32_ofp32": W8A8BFP32OFP32Linear}


def listed():
    return [
        # A chat turn on the smallest model: one short prompt, where the launches and the host count.
        {"name": "prefill_125m_1x33", "kind": "prefill", "model": "opt-125m", "batch": 1, "tokens": 33, "padded": False,
         "dtype": "fp16"},
        # A batch of prompts of different lengths on a mid-sized model, padded to the longest.
        {"name": "prefill_1.3b_8x256", "kind": "prefill", "model": "opt-1.3b", "batch": 8, "tokens": 256, "padded": True,
         "dtype": "fp16"},
        # A large model on a few prompts whose rows are not whole tiles (2112), fp32 residual stream: large products.
        {"name": "prefill_13b_4x528", "kind": "prefill", "model": "opt-13b", "batch": 4, "tokens": 528, "padded": False,
         "dtype": "fp32"},
        # One long prompt (a document) near the model's 2048 positions: long attention.
        {"name": "prefill_6.7b_1x1900", "kind": "prefill", "model": "opt-6.7b", "batch": 1, "tokens": 1900, "padded": False,
         "dtype": "fp16"},
        # Token by token on the smallest model: launches and host time.
        {"name": "generate_125m_1", "kind": "generate", "model": "opt-125m", "batch": 1, "cached": 100, "dtype": "fp16"},
        # One user on a large model: the weights are read once a token.
        {"name": "generate_13b_1", "kind": "generate", "model": "opt-13b", "batch": 1, "cached": 500, "dtype": "fp16"},
        # A served batch of users with long contexts: weights and KV caches.
        {"name": "generate_6.7b_24", "kind": "generate", "model": "opt-6.7b", "batch": 24, "cached": 900, "dtype": "fp16"},
        # One layer by itself: a decode step of 8 sequences, a batch of an odd few hundred rows, a large prefill.
        {"name": "linear_relu_8x20480x5120", "kind": "linear", "layer": "relu_b8_o8", "m": 8, "n": 20480, "k": 5120},
        {"name": "linear_fp32_300x5120x20480", "kind": "linear", "layer": "bfp32_ofp32", "m": 300, "n": 5120, "k": 20480},
        {"name": "linear_relu_8192x20480x5120", "kind": "linear", "layer": "relu_b8_o8", "m": 8192, "n": 20480, "k": 5120},
        # Scores and context of 4 sequences x 40 heads at 512 tokens.
        {"name": "attention_160x512x512x128", "kind": "attention_products", "heads": 160, "t": 512, "s": 512, "d": 128},
        # The LayerNorm between two int8 products of a 2048-token prefill.
        {"name": "layernorm_2048x5120", "kind": "dq_add_layernorm_q", "rows": 2048, "width": 5120, "dtype": "fp32"},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw(rng):
    kind = rng.choice(["prefill", "prefill", "generate", "generate", "linear", "linear", "attention_products",
                       "dq_add_layernorm_q"])
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "batch": _log_int(rng, 1, 16),
                "tokens": _log_int(rng, 17, 1900), "padded": rng.random() < 0.3, "dtype": rng.choice(sorted(DTYPES))}
    if kind == "generate":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "batch": _log_int(rng, 1, 48),
                "cached": _log_int(rng, 17, 1900), "dtype": rng.choice(sorted(DTYPES))}
    width = rng.choice([m[0] for m in MODELS.values()])
    if kind == "linear":
        n, k = rng.choice([(width, width), (4 * width, width), (width, 4 * width)])
        return {"kind": kind, "layer": rng.choice(sorted(LINEARS)), "m": _log_int(rng, 1, 8192), "n": n, "k": k}
    if kind == "attention_products":
        t, s = rng.choice([(1, _log_int(rng, 16, 2048)), (_log_int(rng, 17, 2048), 0), (_log_int(rng, 17, 2048), 0)])
        return {"kind": kind, "heads": _log_int(rng, 12, 320), "t": t, "s": s or t, "d": rng.choice([64, 80, 128])}
    return {"kind": kind, "rows": _log_int(rng, 1, 8192), "width": width, "dtype": rng.choice(sorted(DTYPES))}


def draw(rng):
    """One more case of the same ranges, no larger than the largest listed one."""
    works = [work(c) for c in listed()]
    most = {m: max(w[m] for w in works) for m in ("bytes", "flops")}
    while True:
        case = _draw(rng)
        w = work(case)
        if all(w[m] <= most[m] for m in most):
            return case


# ------------------------------------------------------------------------------------ inputs

def _int8(gen, shape, std):
    return torch.randn(shape, device=DEV, generator=gen).mul_(std).round_().clamp_(-127, 127).to(torch.int8)


def _model(case, gen):
    """A random-weight model whose scales keep every tensor in the range that calibration would."""
    width, heads, layers = MODELS[case["model"]]
    d, act, wstd = width // heads, 30.0, 20.0
    cfg = OPTConfigLite(vocab_size=VOCAB, hidden_size=width, num_attention_heads=heads, ffn_dim=4 * width,
                        num_hidden_layers=layers)
    with torch.device(DEV):
        lm = Int8OPTForCausalLM(cfg)
    dec = lm.model.decoder
    with torch.no_grad():
        for emb, std in ((dec.embed_tokens, 0.5), (dec.embed_positions, 0.1)):
            emb.weight.copy_(torch.randn(emb.weight.shape, device=DEV, generator=gen).mul_(std))
        dec.final_layer_norm.weight.copy_(1 + 0.1 * torch.randn(width, device=DEV, generator=gen))
        for layer in dec.layers:
            at = layer.self_attn
            for ln in (layer.self_attn_layer_norm, layer.final_layer_norm):
                ln.weight.copy_(act * (1 + 0.1 * torch.randn(width, device=DEV, generator=gen)))
                ln.bias.copy_(torch.randn(width, device=DEV, generator=gen))
            for lin in (at.q_proj, at.k_proj, at.v_proj, layer.fc1):
                lin.weight = _int8(gen, (lin.out_features, width), wstd)
                lin.bias = _int8(gen, (1, lin.out_features), wstd)
                lin.a.fill_(1.0 / (math.sqrt(width) * wstd))
                lin.b.fill_(0.1)
            for lin, out in ((at.out_proj, 0.2), (layer.fc2, 0.2)):
                lin.weight = _int8(gen, (width, lin.in_features), wstd)
                lin.bias = 0.05 * torch.randn((1, width), device=DEV, generator=gen)
                lin.a.fill_(out / (math.sqrt(lin.in_features) * wstd * act))
            at.qk_bmm.a.fill_(2.0 / (math.sqrt(d) * act * act))
            at.pv_bmm.a.fill_(2.0 / 127)
    lm = lm.to(DTYPES[case["dtype"]])
    return lm.eval()


def _ids(gen, batch, tokens):
    return torch.randint(2, VOCAB, (batch, tokens), device=DEV, generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "prefill":
        mask = None
        if case["padded"]:   # at least half of every row is prompt, the rest padding on the right
            lengths = torch.randint((case["tokens"] + 1) // 2, case["tokens"] + 1, (case["batch"], 1), device=DEV,
                                    generator=gen)
            mask = torch.arange(case["tokens"], device=DEV)[None, :] < lengths
        return {"kind": kind, "model": _model(case, gen).model, "ids": _ids(gen, case["batch"], case["tokens"]), "mask": mask}
    if kind == "generate":
        lm = _model(case, gen)
        with torch.no_grad():
            out = lm.model(_ids(gen, case["batch"], case["cached"]), use_cache=True)
        past = [tuple(t[:, :, :case["cached"]].contiguous() for t in kv) for kv in out.past_key_values]
        return {"kind": kind, "model": lm, "past": past, "token": _ids(gen, case["batch"], 1)}
    if kind == "linear":
        n, k = case["n"], case["k"]
        with torch.device(DEV):
            layer = LINEARS[case["layer"]](k, n)
        layer.weight = _int8(gen, (n, k), 20.0)
        if case["layer"] == "bfp32_ofp32":
            layer.bias = 0.05 * torch.randn((1, n), device=DEV, generator=gen)
            layer.a.fill_(0.2 / (math.sqrt(k) * 600.0))
        else:
            layer.bias = (_int8(gen, (1, n), 20.0) if "b8" in case["layer"]
                          else torch.randint(-65535, 65536, (1, n), dtype=torch.int32, device=DEV, generator=gen))
            if case["layer"] != "b32_o32":
                layer.a.fill_(1.0 / (math.sqrt(k) * 20.0))
                layer.b.fill_(0.1)
        x = _int8(gen, (case["m"], k), 30.0)
        if k == 4 * n:
            x = x.clamp_(min=0)   # the input of a down projection has passed a ReLU
        return {"kind": kind, "layer": layer, "x": x}
    if kind == "attention_products":
        b, t, s, d = case["heads"], case["t"], case["s"], case["d"]
        with torch.device(DEV):
            qk, pv = BMM_S8T_S8N_F32T(2.0 / (math.sqrt(d) * 900.0)), BMM_S8T_S8N_S8T(2.0 / 127)
        probs = torch.softmax(2 * torch.randn((b, t, s), device=DEV, generator=gen), -1).mul_(127).round_().to(torch.int8)
        return {"kind": kind, "qk": qk, "pv": pv, "q": _int8(gen, (b, t, d), 30.0), "k": _int8(gen, (b, s, d), 30.0),
                "p": probs, "vt": _int8(gen, (b, d, s), 30.0)}
    dtype, width, rows = DTYPES[case["dtype"]], case["width"], case["rows"]
    return {"kind": kind, "x": torch.randint(-30000, 30001, (rows, width), dtype=torch.int32, device=DEV, generator=gen),
            "residual": torch.randn((rows, width), device=DEV, generator=gen).to(dtype),
            "gamma": (30 * (1 + 0.1 * torch.randn(width, device=DEV, generator=gen))).to(dtype),
            "beta": torch.randn(width, device=DEV, generator=gen).to(dtype)}


# ------------------------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "prefill":
        out = state["model"](state["ids"], attention_mask=state["mask"], use_cache=True)
        return [out.last_hidden_state, *(t for kv in out.past_key_values for t in kv)]
    if kind == "generate":
        token, past, logits, tokens = state["token"], state["past"], [], []
        for _ in range(NEW_TOKENS):
            out = state["model"](token, past_key_values=past, use_cache=True)
            past = out.past_key_values
            token = out.logits[:, -1].argmax(-1, keepdim=True)
            logits.append(out.logits)
            tokens.append(token)
        return [torch.cat(tokens, 1), *logits, *(t for kv in past for t in kv)]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "attention_products":
        return [state["qk"](state["q"], state["k"]), state["pv"](state["p"], state["vt"])]
    return ops.dq_add_layernorm_q(state["x"], 1e-5, state["residual"], state["gamma"], state["beta"], 1e-5)


# ------------------------------------------------------------------------------------ what it cannot do without

def work(case):
    """Each weight, input, cache entry and output once (a weight once a token when generating); products as 2 m n k."""
    kind = case["kind"]
    if kind in ("prefill", "generate"):
        width, heads, layers = MODELS[case["model"]]
        b, size = case["batch"], 2 if case["dtype"] == "fp16" else 4
        weights = layers * 12 * width * width
        if kind == "prefill":
            t = case["tokens"]
            # causal attention: half of the t x t products of scores and context
            return {"bytes": weights + 2 * layers * b * t * width + 3 * size * b * t * width,
                    "flops": 2 * b * t * weights + 2 * layers * b * t * t * width}
        s, n = case["cached"], NEW_TOKENS
        head = VOCAB * width
        return {"bytes": n * (weights + size * head + size * b * VOCAB + 2 * layers * b * (s + n // 2) * width),
                "flops": n * (2 * b * (weights + head) + 4 * layers * b * (s + n // 2) * width)}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        bias, out = (1, 1) if "b8" in case["layer"] else (4, 4)
        return {"bytes": m * k + n * k + bias * n + out * m * n, "flops": 2 * m * n * k}
    if kind == "attention_products":
        b, t, s, d = case["heads"], case["t"], case["s"], case["d"]
        return {"bytes": b * (2 * t * d + 2 * s * d + 5 * t * s), "flops": 4 * b * t * s * d}
    size = 2 if case["dtype"] == "fp16" else 4
    rows, width = case["rows"], case["width"]
    return {"bytes": rows * width * (4 + 2 * size + 1) + 2 * size * width, "flops": 10 * rows * width}


def tolerance(case):
    """The operators are integer sums with one rounding at the end, or a LayerNorm whose order of summation is part of
    its contract: exact.  A model ends in a floating LayerNorm (and a floating ``lm_head``): against the same in fp64
    the final LayerNorm is off by 2.1e-4 (fp16) and 6e-8 (fp32) relative, the fp32 sums of ``lm_head`` by a few 1e-7;
    its caches and tokens are whole numbers and stay the same."""
    if case["kind"] in ("prefill", "generate"):
        return {"rel": 1e-3 if case["dtype"] == "fp16" else 2e-6, "differ": 0.0}
    return "exact"
