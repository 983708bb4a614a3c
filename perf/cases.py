"""The work that programs give this library, as cases that can be timed and compared.

A case goes through the public entry points of ``llmops`` the way a program calls them: single operators on the current
stream, a decode step as a replayed graph, a prompt through ``LlamaDecoder.forward``.  Widths are those of the 7B-shape
model that the benchmark and the tests use (hidden 4096, FFN 11008, 32 heads of 128); weights are ~N(0, 0.02) and
activations ~N(0, 1), the distributions of the benchmark.

Kinds:
  fc         one fully connected call on [1, rows, K]: one row while a token is generated, a few for a batch of
             sequences, hundreds and thousands for a prompt; Q4_1 groups of 128 and of 32 (the library's default)
  layer_fcs  the seven projections of one decoder layer (q, k, v, o, gate, up, down) on the same rows: what a batch
             of sequences does per layer and token when the program calls operator by operator
  attention  rotary + cache update + attention of ``tokens`` new tokens behind ``past`` cached ones, in place as the
             operator works (q and k are put back before each call); fp32 cache or fp16 cache
  pack       a weight matrix to Q4_1 blocks, as every linear layer goes through once when a model is loaded
  unpack     the blocks back to fp32
  decode     one token through a captured decode graph: embedding, layers, final norm, logits
  prompt     a prompt (or a later turn of a chat, with ``past`` tokens cached) through ``LlamaDecoder.forward``
"""
import functools
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("llama.cl_amd"))

import llmops  # noqa: E402
from llmops.decode import LLAMA_7B, LlamaDecoder  # noqa: E402
from llmops.opset import KVCache  # noqa: E402

HIDDEN, FFN, HEADS, HEAD = 4096, 11008, 32, 128
#: the projections of one layer: (outputs, inputs)
LAYER = ((HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (FFN, HIDDEN), (FFN, HIDDEN), (HIDDEN, FFN))
#: layers of the models below.  All layers of a model do the same work, and with two the weights of a step (0.34 GB with
#: the logits' projection) come from memory and not from the 256 MB cache in front of it.  More would make outputs
#: incomparable: see tolerance()
MODEL_LAYERS = 2


def listed():
    return [
        # the smallest call: one row, a square projection, the default group
        {"name": "fc_row1_g32", "kind": "fc", "rows": 1, "n": HIDDEN, "k": HIDDEN, "group": 32},
        # sixteen sequences generating in step: weights are still read once per step and the rows are few
        {"name": "layer_fcs_rows16", "kind": "layer_fcs", "rows": 16, "group": 128},
        # a short prompt
        {"name": "fc_rows128", "kind": "fc", "rows": 128, "n": HIDDEN, "k": FFN, "group": 128},
        # a prompt of no particular length, outputs that do not fill the last strip
        {"name": "fc_rows300_ragged", "kind": "fc", "rows": 300, "n": 4090, "k": FFN, "group": 128},
        # the longest prompt the benchmark has
        {"name": "fc_rows2048", "kind": "fc", "rows": 2048, "n": FFN, "k": HIDDEN, "group": 128},
        # a prompt through a model packed with the default group
        {"name": "fc_rows512_g32", "kind": "fc", "rows": 512, "n": FFN, "k": HIDDEN, "group": 32},
        # one token behind a full cache of halves
        {"name": "attn_decode_fp16", "kind": "attention", "batch": 1, "tokens": 1, "past": 2047, "half": True},
        # a short user turn in a chat that already has 1500 tokens
        {"name": "attn_turn16", "kind": "attention", "batch": 1, "tokens": 16, "past": 1500, "half": False},
        # a whole prompt
        {"name": "attn_prompt2048", "kind": "attention", "batch": 1, "tokens": 2048, "past": 0, "half": False},
        # loading a model: one projection
        {"name": "pack_g128", "kind": "pack", "n": FFN, "k": HIDDEN, "group": 128},
        # generating a token, the whole step
        {"name": "decode_step", "kind": "decode", "past": 2047, "half": False},
        # reading a prompt, the whole pass
        {"name": "prompt512", "kind": "prompt", "tokens": 512, "past": 0, "half": False},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fc", "fc", "fc", "layer_fcs", "attention", "attention", "pack", "unpack", "decode", "prompt"])
    if kind == "fc":
        group = rng.choice([128, 128, 32])
        n = rng.choice([HIDDEN, FFN, _log(rng, 512, 12288)])
        k = rng.choice([HIDDEN, FFN, group * _log(rng, 512 // group, 11008 // group)])
        top = 2048 * HIDDEN * FFN // (n * k)
        return {"kind": kind, "rows": _log(rng, 1, min(2048, top)), "n": n, "k": k, "group": group}
    if kind == "layer_fcs":
        return {"kind": kind, "rows": _log(rng, 1, 256), "group": rng.choice([128, 128, 32])}
    if kind == "attention":
        batch = rng.choice([1, 1, 2, 4, 8])
        tokens = _log(rng, 1, 2048 // batch)
        return {"kind": kind, "batch": batch, "tokens": tokens, "past": rng.choice([0, _log(rng, 1, 4096 - tokens)]) // batch,
                "half": rng.random() < 0.5}
    if kind in ("pack", "unpack"):
        group = rng.choice([128, 32])
        return {"kind": kind, "n": _log(rng, 512, 11008), "k": group * _log(rng, 512 // group, 4096 // group), "group": group}
    if kind == "decode":
        return {"kind": kind, "past": _log(rng, 1, 4095), "half": rng.random() < 0.5}
    tokens = _log(rng, 2, 1024)
    return {"kind": kind, "tokens": tokens, "past": rng.choice([0, _log(rng, 1, 2048)]), "half": rng.random() < 0.5}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * std


def _cache_rows(tokens):
    """programs allocate caches in round sizes"""
    return max(256, -(-tokens // 256) * 256)


def _filled_cache(gen, layers, batch, rows, past, half):
    cfg = {"layer_num": layers, "head_num": HEADS, "head_size": HEAD}
    kv = KVCache(cfg, batch, rows, dtype=torch.float16 if half else torch.float32)
    for plane in range(2 * layers):  # (plane by plane: no second copy of the whole cache)
        kv.cache[plane, :, :, :past] = _normal(gen, batch, HEADS, past, HEAD).to(kv.cache.dtype)
    return kv


@functools.lru_cache(None)
def _decode_stream():
    """the one stream on which a program generates: a token's step waits for the step before it"""
    return torch.cuda.Stream()


class _State:
    pass


def prepare(case, seed):
    gen, kind, s = _gen(seed), case["kind"], _State()
    s.case = case
    if kind in ("fc", "layer_fcs"):
        shapes = ((case["n"], case["k"]),) if kind == "fc" else LAYER
        s.n = [n for n, _ in shapes]
        s.w = [llmops.offline_FC_quant_Q4A(_normal(gen, n, k, std=0.02), case["group"]) for n, k in shapes]
        by_k = {k: _normal(gen, 1, case["rows"], k) for k in sorted({k for _, k in shapes})}
        s.x = [by_k[k] for _, k in shapes]
    elif kind == "attention":
        b, t, past = case["batch"], case["tokens"], case["past"]
        s.kv = _filled_cache(gen, 1, b, _cache_rows(past + t), past, case["half"])
        s.fresh = _normal(gen, 2, b, t, HEADS * HEAD)  # q and k as the projections leave them
        s.qk = torch.empty_like(s.fresh)
        s.v = _normal(gen, b, t, HEADS * HEAD)
        s.inv_freq = 1.0 / (10000.0 ** (torch.arange(0, HEAD, 2, device="cuda").float() / HEAD))
        s.slots = torch.arange(past, past + t, dtype=torch.int32, device="cuda")
    elif kind == "pack":
        s.w = _normal(gen, case["n"], case["k"], std=0.02)
    elif kind == "unpack":
        s.w = llmops.offline_FC_quant_Q4A(_normal(gen, case["n"], case["k"], std=0.02), case["group"])
    else:
        past, t = case["past"], case.get("tokens", 1)
        s.model = LlamaDecoder(dict(LLAMA_7B, layer_num=MODEL_LAYERS), group_k=128, seed=seed, embed_rows=1024, device_rng=True)
        # In a trained model what one layer adds to the hidden state is a few percent of it; with the constructor's
        # random weights it is as large, so the embedding is scaled to stand for the layers before these.
        s.model.embed_tokens.scales.mul_(64.0)
        s.kv = _filled_cache(gen, MODEL_LAYERS, 1, _cache_rows(past + t), past, case["half"])
        s.ids = torch.randint(0, 1024, (1, t), generator=gen, device="cuda")
        s.slots = torch.arange(past, past + t, dtype=torch.int32, device="cuda")
        if kind == "decode":
            s.token = int(s.ids[0, 0])
            s.graph = s.model.capture_decode(s.kv.cache, past, past, stream=_decode_stream())
    return s


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind in ("fc", "layer_fcs"):
        return [llmops.fc_Q4A(x, w, n) for x, w, n in zip(s.x, s.w, s.n)]
    if kind == "attention":
        s.qk.copy_(s.fresh)
        q, k = s.qk[0], s.qk[1]
        llmops.attention_rope2(q, k, s.v, s.inv_freq, s.kv.cache, s.slots, case["past"], 0)
        return [q, k, s.kv.cache]
    if kind == "pack":
        return llmops.offline_FC_quant_Q4A(s.w, case["group"])
    if kind == "unpack":
        return llmops.offline_FC_dequant_Q4A(s.w)
    if kind == "decode":
        return [s.graph.step(s.token, case["past"], case["past"]), s.kv.cache]
    return [s.model.forward(s.ids, s.kv.cache, s.slots, case["past"]), s.kv.cache]


def _packed_bytes(n, k, group):
    return -(-n // 32) * -(-k // group) * (16 * group + 128)


def _fc_work(rows, n, k, group):
    return _packed_bytes(n, k, group) + 4 * rows * (n + k), 2 * rows * n * k


def _attention_work(batch, tokens, past, half):
    """q, k, v and the past cache read, q, k and the new cache rows written; each token sees the past and the tokens up
    to itself"""
    e = 2 if half else 4
    width = HEADS * HEAD
    return (batch * width * (tokens * (3 * 4 + 2 * 4 + 2 * e) + 2 * past * e),
            4 * batch * width * tokens * (past + (tokens + 1) / 2))


def work(case):
    kind = case["kind"]
    if kind == "fc":
        b, f = _fc_work(case["rows"], case["n"], case["k"], case["group"])
    elif kind == "layer_fcs":
        parts = [_fc_work(case["rows"], n, k, case["group"]) for n, k in LAYER]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "attention":
        b, f = _attention_work(case["batch"], case["tokens"], case["past"], case["half"])
    elif kind in ("pack", "unpack"):
        b, f = _packed_bytes(case["n"], case["k"], case["group"]) + 4 * case["n"] * case["k"], 0
    else:
        t, vocab = case.get("tokens", 1), LLAMA_7B["vocab_size"]
        e = 2 if case["half"] else 4
        # the packed weights, the past cache rows and the new ones once, the embedding's rows, the logits
        weights = sum(_packed_bytes(n, k, 128) for n, k in LAYER) * MODEL_LAYERS + _packed_bytes(vocab, HIDDEN, 128)
        b = weights + MODEL_LAYERS * 2 * HIDDEN * e * (case["past"] + t) + t * (HIDDEN + 4 * vocab)
        f = 2 * t * (sum(n * k for n, k in LAYER) * MODEL_LAYERS + vocab * HIDDEN)
        f += MODEL_LAYERS * _attention_work(1, t, case["past"], case["half"])[1]
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pack", "unpack"):
        return "exact"  # bytes; and d * code + m, whose product is exact, rounded once
    if kind in ("fc", "layer_fcs"):
        # fp32 sums of exact int32 group sums: against the same codes in 64 bits 2 to 3e-7, largest 1.5e-6
        return {"rel": 1.2e-6, "max": 8e-6}
    if kind == "attention":
        # against 64 bits: up to 5.7e-7, largest 9.3e-6 (2048 tokens).  A new row that is stored as halves can fall on
        # the other side of a rounding: one unit of a half is up to 9.8e-4 of the value
        return {"rel": 1e-5, "max": 2e-3} if case["half"] else {"rel": 2.4e-6, "max": 4e-5}
    # A difference of 1e-7 flips an 8-bit activation code now and then, a flipped code moves the next output by 4e-4,
    # which flips 3 % of the next codes: two correct evaluations of the layers end up apart by the rounding of the
    # activations.  Separate and fused operators on the same weights: 0.4 to 1 %, largest 6 % (two layers; 0.7 to 1.7 %
    # with four, 3 % with thirty-two)
    return {"rel": 0.03, "max": 0.25}
