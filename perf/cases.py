"""What the speed of this framework is measured on: the calls that a program which runs a Llama model makes.

A case is one call (or one short loop of calls) through the public classes `Llama3` and `Transformer`, on a model of one of
the shapes in `denograd_amd.synthetic.CONFIGS` with seeded random weights.  Five kinds of work:

* `generate`: greedy decoding of one sequence with the token fed back on the device (`Llama3.generate`), the conversation
  so far being in the KV cache.
* `chat`: the loop of a chat (`Llama3.chat_tokens`): one sequence, the token read by the host after every step because it
  looks for a stop token; at temperature 0.95 (the default of `Llama3`) the token is drawn by the device sampler.
* `prefill`: a prompt, or the next message of a conversation, in one pass (`Transformer.forward_rows` with tokens [B, S]).
* `batch`: decoding of several sequences at once (`forward_rows` with one position each, tokens fed back on the device, the
  loop of `Llama3.generate_batch`).
* `ingest`: a bfloat16 checkpoint in Hugging Face names turned into int8 or NF4 weights of the model.

Outputs are the tokens, the logits of the last step and the KV cache of every layer (the state that a step updates), the last
two as views of the device buffers.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from denograd_amd import ffi, synthetic
from denograd_amd.llama import convert_from_huggingface, fix_bf16
from denograd_amd.llama3 import Int8Linear, Llama3, NF4Linear
from denograd_amd.tensor import Tensor


def listed() -> list[dict]:
    return [
        # the smallest calls: a two-layer model, where nothing but launches and the host's read of each token takes time
        {"name": "chat-tiny16", "kind": "chat", "model": "tiny16", "layers": 2, "prompt": 16, "new": 8, "temperature": 0.0, "context": 64},
        # the benchmark's own workload: 1B in fp16 behind a 512-token prompt, decoded greedily
        {"name": "generate-1B", "kind": "generate", "model": "1B", "layers": 16, "prompt": 512, "new": 32, "context": 1024},
        # what `Llama3(...)` does by default: a short question, every token drawn at temperature 0.95 and read by the host
        {"name": "chat-1B-sampled", "kind": "chat", "model": "1B", "layers": 16, "prompt": 131, "new": 16, "temperature": 0.95, "context": 1024},
        # the 8B model with int8 weights at the positions of an ordinary conversation
        {"name": "generate-8B-int8", "kind": "generate", "model": "8B-int8", "layers": 32, "prompt": 517, "new": 16, "context": 2304},
        # the 8B model with NF4 weights at the end of a long document
        {"name": "generate-8B-nf4-long", "kind": "generate", "model": "8B-nf4", "layers": 32, "prompt": 4099, "new": 16, "context": 4352},
        # the first prompt of a conversation with the 1B model: a few hundred tokens, not a round number of them
        {"name": "prefill-1B-371", "kind": "prefill", "model": "1B", "layers": 16, "batch": 1, "start": 0, "seq": 371, "context": 1024},
        # the next message of a conversation: a few dozen new positions behind a thousand old ones
        {"name": "prefill-3B-int8-57-more", "kind": "prefill", "model": "3B-int8", "layers": 28, "batch": 1, "start": 1024, "seq": 57, "context": 1536},
        # one long document as a prompt
        {"name": "prefill-8B-nf4-4096", "kind": "prefill", "model": "8B-nf4", "layers": 32, "batch": 1, "start": 0, "seq": 4096, "context": 4352},
        # the largest: sixteen long prompts at once
        {"name": "prefill-8B-int8-16x2048", "kind": "prefill", "model": "8B-int8", "layers": 32, "batch": 16, "start": 0, "seq": 2048, "context": 2304},
        # a serving loop over sixteen sequences
        {"name": "batch-8B-int8-16", "kind": "batch", "model": "8B-int8", "layers": 32, "batch": 16, "start": 2048, "new": 8, "context": 2304},
        # a lightly loaded server: five sequences on the small model
        {"name": "batch-1B-5", "kind": "batch", "model": "1B", "layers": 16, "batch": 5, "start": 300, "new": 8, "context": 1024},
        # loading a checkpoint: three layers of the 8B model, bfloat16 in, int8 codes and scales out
        {"name": "ingest-8B-int8", "kind": "ingest", "model": "8B-int8", "layers": 3},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """A whole number between lo and hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng) -> dict:
    """One more case: any of the shapes, with fewer layers or all of them, at any length up to those listed."""
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["generate", "generate", "chat", "prefill", "prefill", "batch", "batch", "ingest"])
        if kind == "ingest":
            case = {"kind": kind, "model": rng.choice(["8B-int8", "8B-nf4", "3B-int8"]), "layers": rng.randint(1, 3)}
            return case
        model = rng.choice(["tiny16", "1B", "3B-int8", "8B-nf4", "8B-int8"])
        full = synthetic.CONFIGS[model]["n_layers"]
        case = {"kind": kind, "model": model, "layers": _log(rng, 2, full)}
        if kind in ("generate", "chat"):
            if kind == "chat" and rng.random() < 0.2:
                case["model"] = "tiny"                        # the float32 model: one position per call only
                case["layers"] = 2
            case["prompt"] = _log(rng, 2, 4200)
            case["new"] = rng.randint(4, 24)
            if kind == "chat":
                # the device sampler takes vocabularies of more than 512 entries: all of these
                case["temperature"] = rng.choice([0.0, 0.95])
            last = case["prompt"] + case["new"]
        elif kind == "prefill":
            case["batch"] = rng.choice([1, 1, 1, 2, 3, 4, 8, 16])
            case["start"] = rng.choice([0, 0, _log(rng, 1, 2048)])
            case["seq"] = _log(rng, 2, 4096)
            last = case["start"] + case["seq"]
            if case["batch"] * case["seq"] > 32768:
                continue
        else:
            case["batch"] = _log(rng, 2, 32)
            case["start"] = _log(rng, 4, 2048)
            case["new"] = rng.randint(3, 10)
            last = case["start"] + case["new"]
            if case["batch"] * case["start"] > 32768:
                continue
        case["context"] = (last + 255) // 256 * 256
        if _cost(case) <= most:
            return case


# ---- models and inputs

def _cfg(case: dict) -> dict:
    return synthetic.config(case["model"], n_layers=case["layers"], max_context=case.get("context", 64))


def _view(t: Tensor) -> torch.Tensor:
    """The device buffer of a Tensor as a torch tensor, without a copy."""
    kind = {"float32": "<f4", "float16": "<f2", "bfloat16": "<i2", "int8": "|i1", "uint8": "|u1", "int32": "<i4"}[t.dtype]

    class _Device:
        __cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": kind, "data": (t.ptr, False), "version": 2}

    v = torch.as_tensor(_Device(), device="cuda")
    return v.view(torch.bfloat16) if t.dtype == "bfloat16" else v


def _weights(cfg: dict, seed: int) -> dict:
    """Seeded weights made on the device: every matrix N(0, 1 / columns), the two that write into the residual stream smaller
    by the square root of their number, embeddings N(0, 1), and a final norm that gives logits of the size that trained
    models have.  The lm_head of an untied model is the embedding table shifted by one row.  So the residual stream keeps
    the size that it has in trained models, attention scores are of order one, and the best token is ahead of the others by
    more than rounding can make up."""
    act = cfg["act_dtype"]
    n = 0

    def randn(shape, std):
        nonlocal n
        n += 1
        return Tensor.randn(shape, act, seed * 1009 + n, std)

    sd = {"tok_embeddings.weight": randn((cfg["vocab_size"], cfg["dim"]), 1.0)}
    for l in range(cfg["n_layers"]):
        for name, (out_f, in_f) in synthetic.linear_shapes(cfg).items():
            std = in_f ** -0.5 * ((2 * cfg["n_layers"]) ** -0.5 if name.endswith(("wo", "w2")) else 1.0)
            sd[f"layers.{l}.{name}.weight"] = randn((out_f, in_f), std)
        sd[f"layers.{l}.attention_norm.weight"] = Tensor.ones((cfg["dim"],), act)
        sd[f"layers.{l}.ffn_norm.weight"] = Tensor.ones((cfg["dim"],), act)
    sd["norm.weight"] = Tensor.full((cfg["dim"],), 25.0 / cfg["dim"], act)
    if cfg["tied"]:
        sd["output.weight"] = sd["tok_embeddings.weight"]
    else:
        head = Tensor.empty(sd["tok_embeddings.weight"].shape, act)
        row = head.nbytes // cfg["vocab_size"]
        lib = ffi.load()
        ffi.check(lib.jsgrad_hip_copy(head.ptr + row, sd["tok_embeddings.weight"].ptr, head.nbytes - row))
        ffi.check(lib.jsgrad_hip_copy(head.ptr, sd["tok_embeddings.weight"].ptr + head.nbytes - row, row))
        sd["output.weight"] = head
    return sd


def _model(cfg: dict, seed: int, temperature: float) -> Llama3:
    return Llama3.from_config(cfg, temperature=temperature).load_weights(_weights(cfg, seed))


def _tokens(cfg: dict, seed: int, shape) -> np.ndarray:
    return np.random.default_rng(seed).integers(0, cfg["vocab_size"], size=shape, dtype=np.int32)


def _checkpoint(cfg: dict, seed: int) -> dict:
    """Layers of a bfloat16 checkpoint under their Hugging Face names, on the device."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    names = {"attention.wq": "self_attn.q_proj", "attention.wk": "self_attn.k_proj", "attention.wv": "self_attn.v_proj", "attention.wo": "self_attn.o_proj",
             "feed_forward.w1": "mlp.gate_proj", "feed_forward.w2": "mlp.down_proj", "feed_forward.w3": "mlp.up_proj"}
    out = {}
    for l in range(cfg["n_layers"]):
        shapes = {names[k]: v for k, v in synthetic.linear_shapes(cfg).items()}
        shapes.update({"input_layernorm": (cfg["dim"],), "post_attention_layernorm": (cfg["dim"],)})
        for name, shape in shapes.items():
            t = Tensor.empty(shape, "bfloat16")
            _view(t).copy_(torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).mul_(0.02))
            out[f"model.layers.{l}.{name}.weight"] = t
    torch.cuda.synchronize()
    return out


def prepare(case: dict, seed: int) -> dict:
    """A loaded model that has served a call before, the conversation so far in its KV cache, and the tokens of the next call."""
    cfg = _cfg(case)
    if case["kind"] == "ingest":
        return {"case": case, "cfg": cfg, "checkpoint": _checkpoint(cfg, seed)}
    llm = _model(cfg, seed, case.get("temperature", 0.0))
    model, st = llm.model, {"case": case, "cfg": cfg, "llm": llm}
    if case["kind"] in ("generate", "chat"):
        prompt = [int(t) for t in _tokens(cfg, seed, case["prompt"])]
        llm.batched_prefill = cfg["act_dtype"] == "float16"
        # an earlier answer to the same conversation, to another last token: the step has been captured
        llm.chat_tokens(prompt[:-1] + [prompt[0]], 3)
        st["prompt"] = prompt
        logits = model.logits
    else:
        b, start = case["batch"], case["start"]
        seq = case["seq"] if case["kind"] == "prefill" else 1
        toks = _tokens(cfg, seed, (b, start + seq))
        st["tokens"] = np.ascontiguousarray(toks[:, start:])
        if start:
            model.forward_rows(np.ascontiguousarray(toks[:, :start]), 0)
        model.forward_rows(np.ascontiguousarray(st["tokens"][:, ::-1] if seq > 1 else (st["tokens"] + 1) % cfg["vocab_size"]), start)   # an earlier message
        if case["kind"] == "batch":
            st["history"] = Tensor.empty((case["new"], b), "int32")
        logits = model.rows_logits()
    st["outputs"] = {"logits": _view(logits), "cache": [_view(layer.attention.cache_kv) for layer in model.layers]}
    return st


def run(st: dict) -> dict:
    case = st["case"]
    kind = case["kind"]
    if kind == "generate":
        llm = st["llm"]
        llm.start_pos = 0
        return {"tokens": llm.generate(st["prompt"], case["new"]), **st["outputs"]}
    if kind == "chat":
        llm = st["llm"]
        llm.start_pos = 0
        return {"tokens": np.array(llm.chat_tokens(st["prompt"], case["new"])["tokens"], np.int32), **st["outputs"]}
    if kind == "prefill":
        return {"tokens": st["llm"].model.forward_rows(st["tokens"], case["start"]).numpy(), **st["outputs"]}
    if kind == "batch":
        model, hist, b, lib = st["llm"].model, st["history"], case["batch"], ffi.load()
        tok = model.forward_rows(st["tokens"], case["start"])
        for i in range(case["new"]):
            ffi.check(lib.jsgrad_hip_copy(hist.ptr + i * b * 4, tok.ptr, b * 4))
            if i + 1 < case["new"]:
                tok = model.forward_rows(tok, case["start"] + 1 + i)
        return {"tokens": hist.numpy(), **st["outputs"]}
    cfg = st["cfg"]
    weights = fix_bf16(convert_from_huggingface(st["checkpoint"], cfg["n_layers"], cfg["n_heads"], cfg["n_kv_heads"]))
    linear = Int8Linear if cfg["quantize"] == "int8" else NF4Linear(64)
    st["weights"] = linear.quantize(weights)
    return {k: _view(t) for k, t in st["weights"].items()}


# ---- what a pass cannot do without

def _cost(case: dict) -> float:
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def work(case: dict) -> dict:
    cfg = _cfg(case)
    shapes = synthetic.linear_shapes(cfg).values()
    matrices = cfg["n_layers"] * sum(o * i for o, i in shapes)
    if case["kind"] == "ingest":
        norms = cfg["n_layers"] * 2 * cfg["dim"]
        rows = cfg["n_layers"] * sum(o for o, _ in shapes)
        out = matrices + 2 * rows if cfg["quantize"] == "int8" else matrices // 2 + matrices // 64 * 2
        return {"bytes": 2 * matrices + out + 4 * norms, "flops": 0}
    weights, row = synthetic.weight_bytes_per_token(cfg), synthetic.kv_bytes_per_position(cfg)
    head, width = cfg["vocab_size"] * cfg["dim"], cfg["dim"]
    attention = lambda positions: 4.0 * positions * width * cfg["n_layers"]   # noqa: E731  q.K and P.V of one row
    if case["kind"] in ("generate", "chat"):
        first, n, b = case["prompt"], case["new"], 1
    elif case["kind"] == "batch":
        first, n, b = case["start"] + 1, case["new"], case["batch"]
    else:
        b, s, start = case["batch"], case["seq"], case["start"]
        seen = s * start + s * (s + 1) // 2                                   # positions seen by the rows of one sequence
        return {"bytes": weights + b * (start + s) * row + b * s * 4, "flops": 2.0 * b * s * matrices + 2.0 * b * head + b * attention(seen)}
    seen = sum(first + i for i in range(n))
    return {"bytes": n * weights + b * (seen + n) * row, "flops": n * b * 2.0 * (matrices + head) + b * attention(seen)}


def tolerance(case: dict):
    """Codes and scales of a checkpoint are whole numbers and single roundings.  For the rest the one-row kernels and the
    several-row kernels were compared on the same 100-token prompt: sums in another order, and one more rounding of a
    quantised weight.  Largest over the shapes at full depth: relative 1.5e-3, 1.1e-2 of the r.m.s. value for a single
    element; four times that is allowed.  float32 sums in another order: 2e-6."""
    if case["kind"] == "ingest":
        return "exact"
    if case["model"] == "tiny":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 6e-3, "max": 0.045}
