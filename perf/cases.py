"""The work a program has this framework do, as cases to be timed: the driver loop, the generation loop, the operator
path and the batched prefill, at the shapes of lighterpp_amd.CONFIGS, over the context lengths, prompt lengths and
options those are used with.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) model with weights in HBM, prompt and cache contents, made from the seed
    run(state)          one pass through the public entry points; returns its outputs
    work(case)          bytes and floating-point operations one pass cannot do without
    tolerance(case)     how far two correct implementations of the same precision may be apart

A case is a dict: "kind" (below), "config" (key of CONFIGS) and the kind's own sizes.

    drive     lpp_run: a prompt read by decode steps, then generation (main.cpp's loop)   prompt, reply
    generate  lpp_generate on the persistent path from a cache that holds `start` positions     start, tokens, sampled
    operators lpp_generate on the operator path (the twelve wrappers of kernels.cuh)            start, tokens, sampled
    answer    lpp_run_batched_prefill: prompt in one batch, then generation                     prompt, reply
    prefill   lpp_prefill of `tokens` ids behind a cache that holds `start` positions           start, tokens, fast
"""
import math

import numpy as np
import torch

from lighterpp_amd import CONFIGS, Model, capi

C1, C2, C3, C4, C5 = ("c1_llama2c_15m_fp32", "c2_tinyllama_1b_fp16", "c3_llama32_1b_fp16", "c4_llama32_1b_longctx_fp16",
                      "c5_llama3_8b_fp16")


def listed():
    return [
        # A story model of a few million parameters in the driver loop: nothing but latency.  Prompt of 8 ids, greedy.
        {"name": "drive_15m", "kind": "drive", "config": C1, "prompt": 8, "reply": 32},
        # The driver's default way through a 16-id prompt and into the reply, on a 1B model.
        {"name": "drive_tinyllama", "kind": "drive", "config": C2, "prompt": 16, "reply": 16},
        # Chat decoding with the sampler on (temperature, repetition penalty, window), short context.
        {"name": "generate_1b", "kind": "generate", "config": C3, "start": 0, "tokens": 16, "sampled": True},
        # Decoding behind a long document.
        {"name": "generate_1b_8k", "kind": "generate", "config": C4, "start": 8192, "tokens": 16, "sampled": False},
        # Decoding with the largest model, in the middle of its context.
        {"name": "generate_8b", "kind": "generate", "config": C5, "start": 500, "tokens": 8, "sampled": False},
        # A program that calls the operator wrappers itself, as the reference's forward() does.
        {"name": "operators_1b", "kind": "operators", "config": C3, "start": 100, "tokens": 8, "sampled": True},
        # A short question: how long until the first two ids of the answer.
        {"name": "answer_tinyllama", "kind": "answer", "config": C2, "prompt": 23, "reply": 2},
        # A page of text into the cache: the length the prefill is benchmarked with.
        {"name": "prefill_1b_512", "kind": "prefill", "config": C3, "start": 0, "tokens": 512, "fast": False},
        # The opt-in fast mode on a few pages, odd length.
        {"name": "prefill_1b_fast_2011", "kind": "prefill", "config": C3, "start": 0, "tokens": 2011, "fast": True},
        # A whole document: attention over thousands of positions.
        {"name": "prefill_1b_6000", "kind": "prefill", "config": C4, "start": 0, "tokens": 6000, "fast": False},
        # The next message of a conversation that is already in the cache.
        {"name": "prefill_1b_append", "kind": "prefill", "config": C4, "start": 3000, "tokens": 150, "fast": False},
        # A long prompt through the largest model.
        {"name": "prefill_8b_1024", "kind": "prefill", "config": C5, "start": 0, "tokens": 1024, "fast": False},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("drive", "generate", "generate", "operators", "answer", "prefill", "prefill", "prefill"))
    if kind == "drive":
        config = rng.choice((C1, C2, C3))
        prompt = _log_uniform(rng, 1, 48 if config == C1 else 28)
        return {"kind": kind, "config": config, "prompt": prompt, "reply": rng.randint(4, 48 if config == C1 else 16)}
    if kind in ("generate", "operators"):
        config = rng.choice((C1, C2, C3, C4, C5) if kind == "generate" else (C2, C3, C4))
        tokens = rng.randint(2, 7 if config == C5 else 16)
        room = min(CONFIGS[config].seq_len, 9000) - tokens
        return {"kind": kind, "config": config, "start": _log_uniform(rng, 1, room), "tokens": tokens, "sampled": rng.random() < 0.5}
    config = rng.choice((C2, C3, C5))
    if kind == "answer":
        return {"kind": kind, "config": config, "prompt": _log_uniform(rng, 9, 400), "reply": rng.randint(1, 3)}
    config = rng.choice((config, C4))
    longest = {C2: 1800, C3: 2000, C4: 5000, C5: 1000}[config]
    tokens = _log_uniform(rng, 9, longest)
    start = 0 if rng.random() < 0.5 else _log_uniform(rng, 1, min(CONFIGS[config].seq_len, 7000) - tokens)
    return {"kind": kind, "config": config, "start": start, "tokens": tokens, "fast": rng.random() < 0.3}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

class _DeviceMemory:
    """Device memory of a model as torch sees it (no copy).  Keeps the model alive."""

    def __init__(self, model, ptr, shape, typestr):
        self.model = model
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 3, "strides": None}


def _view(model, ptr, shape, typestr):
    return torch.as_tensor(_DeviceMemory(model, ptr, shape, typestr), device="cuda")


def _load_weights(model, gen):
    """The benchmark's weights, N(0, 0.02) with norm gains 1, made on the device from the generator; a binary16 model's
    embedding holds binary16 values, as a GGUF file gives it.  A tensor counts as loaded once its end has been uploaded."""
    shape = model.shape
    for t in range(12):
        if t == capi.T_WCLS and shape.tied:
            continue
        gain, embedding = t in (capi.T_RMS_ATT, capi.T_RMS_FFN, capi.T_RMS_FINAL), t == capi.T_TOKEN_EMBEDDING
        wide = gain or embedding or not shape.fp16
        dims = shape.tensor_shape(t)
        w = _view(model, model.tensor_ptr(t), dims, "<f4" if wide else "<f2")
        if gain:
            w.fill_(1.0)
        else:
            w.normal_(0.0, 0.02, generator=gen)
            if embedding and shape.fp16:
                for rows in w.split(16384):
                    rows.copy_(rows.half())
        flat = w.view(-1)
        tail = flat[-16:].cpu().numpy()
        model.upload(t, tail, byte_offset=(flat.numel() - tail.size) * tail.itemsize)
    torch.cuda.synchronize()
    if shape.tied:
        model.tie_classifier()


def prepare(case, seed):
    shape = CONFIGS[case["config"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    model = Model(shape)
    _load_weights(model, gen)
    model.set_path(capi.PATH_OPS if case["kind"] == "operators" else capi.PATH_PERSISTENT)
    cache_shape = (shape.n_layers, shape.n_kv_heads, shape.seq_len, shape.head_size)
    caches = [_view(model, model.buffer_ptr(b), cache_shape, "<f2") for b in (capi.B_KEY_CACHE, capi.B_VALUE_CACHE)]
    start = case.get("start", 0)
    if start > 0:
        for cache in caches:
            cache[:, :, :start].normal_(0.0, 1.0, generator=gen)
    torch.cuda.synchronize()
    if case["kind"] == "prefill":
        model.set_prefill_mode(capi.PREFILL_FAST if case["fast"] else capi.PREFILL_EXACT)
    n = case.get("prompt", case.get("tokens"))
    return {
        "case": case,
        "model": model,
        "ids": rng.integers(3, shape.vocab_size, n).astype(np.int32),
        "uniforms": rng.random(n + 1, dtype=np.float32),
        "logits": _view(model, model.buffer_ptr(capi.B_LOGITS), (shape.vocab_size,), "<f4"),
        "keys": caches[0],
        "values": caches[1],
    }


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(state):
    case, model, ids = state["case"], state["model"], state["ids"]
    if case["kind"] == "prefill":
        model.prefill(ids, case["start"])
        return {"keys": state["keys"], "values": state["values"]}
    if case["kind"] in ("drive", "answer"):
        tokens, _ = model.run(ids, case["prompt"] - 1 + case["reply"], batched_prefill=case["kind"] == "answer")
    else:
        first = int(ids[0])
        if case["sampled"]:
            tokens, _, _ = model.generate(first, case["start"], case["tokens"], temperature=0.8, penalty=1.1, history=[first],
                                          history_cap=64, uniforms=state["uniforms"])
        else:
            tokens, _, _ = model.generate(first, case["start"], case["tokens"])
    return {"tokens": tokens, "logits": state["logits"], "keys": state["keys"], "values": state["values"]}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def _decode(shape, positions):
    """Decode steps one after the other: every weight matrix once a step, the cache up to the step's position."""
    attended = sum(p + 1 for p in positions)
    return (sum(shape.bytes_per_token(p) for p in positions),
            2.0 * shape.matrix_params() * len(positions) + 4.0 * shape.n_layers * shape.dim * attended)


def _prefill(shape, start, n):
    """Cache entries of n ids: every layer's Wk and Wv, and Wq, attention, Wo and the feed-forward block of all layers
    but the last, whose output nothing reads; each weight once, the cache read and written once, the embedding rows."""
    L, dim, kv, hidden = shape.n_layers, shape.dim, shape.kv_dim, shape.hidden_dim
    weights = L * 2 * kv * dim + (L - 1) * (2 * dim * dim + 3 * hidden * dim)
    size = (2.0 if shape.fp16 else 4.0) * weights + 4.0 * dim * n + 2.0 * 2 * kv * (L * n + (L - 1) * (start + n))
    attended = n * start + n * (n + 1) / 2
    return size, 2.0 * weights * n + 4.0 * (L - 1) * dim * attended


def work(case):
    shape = CONFIGS[case["config"]]
    kind = case["kind"]
    if kind == "prefill":
        size, flops = _prefill(shape, case["start"], case["tokens"])
    elif kind == "answer":
        size, flops = _prefill(shape, 0, case["prompt"] - 1)
        more = _decode(shape, range(case["prompt"] - 1, case["prompt"] - 1 + case["reply"]))
        size, flops = size + more[0], flops + more[1]
    elif kind == "drive":
        # (the ids sampled behind the prompt's other ids are dropped: no classifier there)
        size, flops = _decode(shape, range(case["prompt"] - 1 + case["reply"]))
        classifier = float(shape.vocab_size * shape.dim * (case["prompt"] - 1))
        size, flops = size - (2.0 if shape.fp16 else 4.0) * classifier, flops - 2.0 * classifier
    else:
        size, flops = _decode(shape, range(case["start"], case["start"] + case["tokens"]))
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # K and V are rounded to binary16 in the cache: a different order of fp32 sums moves some entries by one step
    # (2^-11 of their value), and the layers after it read them.  Measured between the fused and the persistent path
    # and between the prefill's kernels: 2.1e-4 and 6.5e-3; in the fast mode, which rounds every GEMM input as well,
    # 1.5e-3 and 1.1e-2.  About four times that.
    if case["kind"] == "prefill" and case["fast"]:
        return {"rel": 5e-3, "max": 0.05}
    return {"rel": 1e-3, "max": 0.03}
