"""Performance cases: what programs that use this framework have it do, through its public entry points.

A case is a dict of plain values. `kind` says which entry point it goes through:

  accept     sh_accept_sample over logits that are on the device (a server's batched acceptance)
  gemv       sh_gemv_quant, the f32-level quantized matrix-vector product of narrow calls
  wide       sh_gemm_wide16, the f16 matrix product of calls of 32 columns or more
  forward    Engine.forward_full_readback over a cache that holds `ctx` positions (decode, verify, prefill)
  unified    Engine.verify_unified of B sequences: chains of `cols` tokens, or trees
  spec       Engine.decode_speculative (REJECTION) and the readback of the step's logits

Models are synthetic (seeker_amd.synth): the layer shapes of this repository's named configurations with
fewer layers, so that a pass is some layers of the real thing and the exact result can be computed.
Weights are random but the same for every seed, as a model file is; tokens, cached keys and values,
activations, logits and drafts are made from the seed.
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import math
import struct

import numpy as np
import torch

from seeker_amd import Engine, synth
from seeker_amd import _native as native
from seeker_amd.inference import DeviceBuffer, QTensor, SamplerConfig

# Layer shapes of the named configurations (seeker_amd/synth.py). "8b_mix" is the Q4_K_M recipe of the 8B
# shape: Q6_K attn_v and ffn_down in even layers and a Q6_K output matrix.
SHAPES = {
    "tiny": synth.TINY_TARGET,
    "8b": synth.L8B_TARGET,
    "8b_mix": dataclasses.replace(synth.L8B_TARGET, mix=1, out_type=native.GGML_Q6_K),
    "1b": synth.L1B_DRAFT,
    "qwen_06b": synth.Q06B_DRAFT,
    "moe_30b": synth.Q30B_A3B_TARGET,
}
QTYPES = {"q8_0": native.GGML_Q8_0, "q4_k": native.GGML_Q4_K, "q5_k": native.GGML_Q5_K, "q6_k": native.GGML_Q6_K}
BLOCK = {0: (1, 4), native.GGML_Q8_0: (32, 34), native.GGML_Q4_K: (256, 144), native.GGML_Q5_K: (256, 176),
         native.GGML_Q6_K: (256, 210)}
TREE = (4, 3, 2)  # 4 x 3 x 2 branches: 1 + 4 + 12 + 24 = 41 nodes


def listed():
    return [
        # one sequence's acceptance after a short draft: the smallest call, a few kernels long
        dict(name="accept_one", kind="accept", mode="compare", batch=1, k=4, vocab=32000),
        # a server's batch of 32 sequences, rejection sampling over a Llama-3 vocabulary
        dict(name="accept_batch", kind="accept", mode="rejection", batch=32, k=8, vocab=128256),
        # the tiny Q8_0 model's gate/up over k + 1 = 5 verify columns: the smallest product
        dict(name="gemv_q8_tiny", kind="gemv", qtype="q8_0", rows=2816, inner=512, cols=5),
        # the 8B gate/up over the 8 verify columns of k = 7: the largest product of the headline path
        dict(name="gemv_q4k_verify", kind="gemv", qtype="q4_k", rows=28672, inner=4096, cols=8),
        # the same matrix in a tree verify of 4 x 41 columns (f16 wide arithmetic)
        dict(name="wide_q4k_tree", kind="wide", qtype="q4_k", rows=28672, inner=4096, cols=164),
        # the Q6_K ffn_down of a Q4_K_M file in a prefill of 512 tokens
        dict(name="wide_q6k_prefill", kind="wide", qtype="q6_k", rows=4096, inner=14336, cols=512),
        # one token through layers of the 1B draft at context 2048: single-sequence decode
        dict(name="decode_1b", kind="forward", shape="1b", layers=4, ctx=2048, cols=1, logits=True, residual=False),
        # the 8B verify of k = 7 at context 4096 with its logits of all positions: a whole call
        dict(name="verify_8b", kind="forward", shape="8b", layers=8, ctx=4096, cols=8, logits=True, residual=True),
        # a prompt of 2048 tokens through layers of the 8B target: prefill
        dict(name="prefill_8b", kind="forward", shape="8b", layers=2, ctx=0, cols=2048, logits=False, residual=False),
        # four trees of 41 nodes at context 8192 through 8B layers
        dict(name="tree_8b", kind="unified", shape="8b", layers=2, ctx=8192, batch=4, cols=41, tree=True),
        # eight sequences of k + 1 = 7 columns at context 8192 through a MoE layer
        dict(name="verify_moe", kind="unified", shape="moe_30b", layers=1, ctx=8192, batch=8, cols=7, tree=False),
        # a whole speculative step (7 drafts, verify, rejection sampling) with 1B draft and 8B target layers
        dict(name="spec_step", kind="spec", target="8b", draft="1b", layers=4, ctx=4096, k=7, vocab=32000),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["accept", "gemv", "wide", "decode", "verify", "prefill", "unified", "tree", "moe", "spec"])
    if kind == "accept":
        vocab = rng.choice([32000, 50257, 128256, 151936])
        k = rng.randint(1, 8)
        batch = min(_spread(rng, 1, 32), 32 * 9 * 128256 // ((k + 1) * vocab))
        return dict(kind="accept", mode=rng.choice(["compare", "rejection"]), batch=batch, k=k, vocab=vocab)
    if kind in ("gemv", "wide"):
        qtype = rng.choice(["q4_k", "q4_k", "q6_k", "q5_k", "q8_0"])
        unit = 32 if qtype == "q8_0" else 256
        inner = max(1, _spread(rng, 512, 14336) // unit) * unit
        rows = _spread(rng, 500, 28672)
        rows = max(1, min(rows, 28672 * 4096 // inner))
        cols = _spread(rng, 1, 24) if kind == "gemv" else _spread(rng, 32, 512)
        return dict(kind=kind, qtype=qtype, rows=rows, inner=inner, cols=cols)
    if kind == "decode":
        shape = rng.choice(["tiny", "1b", "8b", "8b_mix", "qwen_06b"])
        ctx = _spread(rng, 16, 800 if shape == "tiny" else 6000)
        return dict(kind="forward", shape=shape, layers=2, ctx=ctx, cols=1, logits=True, residual=rng.random() < 0.5)
    if kind == "verify":
        shape = rng.choice(["tiny", "1b", "8b", "8b_mix", "qwen_06b"])
        ctx = _spread(rng, 16, 800 if shape == "tiny" else 6000)
        return dict(kind="forward", shape=shape, layers=2, ctx=ctx, cols=rng.randint(2, 9), logits=True,
                    residual=rng.random() < 0.5)
    if kind == "prefill":
        shape = rng.choice(["tiny", "1b", "8b", "8b_mix", "qwen_06b"])
        top = 900 if shape == "tiny" else 1800
        cols = _spread(rng, 10, top)
        ctx = 0 if rng.random() < 0.5 else _spread(rng, 8, 100 if shape == "tiny" else 2000)
        return dict(kind="forward", shape=shape, layers=2, ctx=ctx, cols=cols, logits=False, residual=rng.random() < 0.25)
    if kind == "tree":
        return dict(kind="unified", shape=rng.choice(["8b", "1b"]), layers=2, ctx=_spread(rng, 64, 6000),
                    batch=rng.randint(1, 4), cols=rng.choice([13, 29, 41]), tree=True)
    if kind == "moe":
        return dict(kind="unified", shape="moe_30b", layers=1, ctx=_spread(rng, 64, 6000), batch=rng.randint(1, 8),
                    cols=rng.randint(1, 7), tree=False)
    if kind == "unified":
        return dict(kind="unified", shape=rng.choice(["8b", "1b", "8b_mix", "qwen_06b"]), layers=2,
                    ctx=_spread(rng, 64, 4000), batch=rng.randint(2, 8), cols=rng.randint(1, 8), tree=False)
    return dict(kind="spec", target="8b", draft="1b", layers=2, ctx=_spread(rng, 64, 4000), k=rng.randint(1, 7),
                vocab=32000)


# ------------------------------------------------------------------ inputs


class State:
    """What a program has in hand before a call; its handles are given back with it."""

    def __init__(self, case):
        self.case, self.handles = case, []

    def own(self, handle):
        self.handles.append(handle)
        return handle

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


@functools.lru_cache(maxsize=1)
def _engine():
    return Engine(0)


@functools.lru_cache(maxsize=2)
def _image(shape, layers, vocab):
    """A model file's bytes in host memory."""
    s = dataclasses.replace(SHAPES[shape], n_layer=layers)
    return synth.GgufImage(dataclasses.replace(s, n_vocab=vocab) if vocab else s, 41)


@functools.lru_cache(maxsize=2)
def _blocks(qtype, rows, inner):
    """A quantized matrix as a file holds it."""
    w = synth.normal_f32(43, 0, rows * inner, 0.0, 0.02)
    return synth.quantize(QTYPES[qtype], w)


def _device(tensor):
    """A torch tensor as one of the engine's device buffers (it stays torch's)."""
    return DeviceBuffer(_engine(), ctypes.c_void_p(tensor.data_ptr()), tensor.numel() * tensor.element_size())


def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) & 0x7FFFFFFF)


def _cached(shape, layers, ctx, seed, seq):
    """Keys and values of `ctx` cached positions, per layer (K, V) as f16 bits [ctx][n_kv][hd]."""
    hd = shape.head_dim or shape.n_embd // shape.n_head
    # a unit-RMS input against N(0, weight_std) weights; qwen3 keys are normalized per head
    std = shape.weight_std * math.sqrt(shape.n_embd)
    g = _generator(seed * 1000 + seq * 16 + 7)
    kv = torch.randn((layers, 2, ctx, shape.n_head_kv, hd), generator=g, device="cuda")
    kv[:, 0] *= 1.0 if shape.arch else std
    kv[:, 1] *= std
    return kv.half().cpu().numpy().view(np.uint16)


def _fill(cache, rows):
    ctx = rows.shape[2]
    if ctx:
        for layer in range(rows.shape[0]):
            cache.write_layer(layer, False, rows[layer, 0])
            cache.write_layer(layer, True, rows[layer, 1])
    cache.set_position(ctx)
    return cache


def _tree_parents():
    parents, level = [-1], [0]
    for width in TREE:
        nxt = []
        for p in level:
            for _ in range(width):
                nxt.append(len(parents))
                parents.append(p)
        level = nxt
    return parents


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_accept(c, seed):
    s, eng, g = State(c), _engine(), _generator(seed)
    B, k, V = c["batch"], c["k"], c["vocab"]
    # logits of a unit-RMS hidden state against a random head, and a draft model near the target
    s.p = torch.randn((B, k + 1, V), generator=g, device="cuda") * 2.0
    noise = torch.randn((B, k, V), generator=g, device="cuda")
    s.q = s.p[:, :k] * 0.9 + noise * 0.5
    if c["mode"] == "rejection":  # drafts drawn from the draft distribution
        u = torch.rand((B, k, V), generator=g, device="cuda").clamp_(1e-9, 1 - 1e-7)
        s.drafts = (s.q / 0.8 - (-u.log()).log()).argmax(-1).to(torch.int32)
    else:
        s.drafts = s.q.argmax(-1).to(torch.int32)
    s.accepted = torch.zeros(B, dtype=torch.int32, device="cuda")
    s.next = torch.zeros(B, dtype=torch.int32, device="cuda")
    s.sampler = SamplerConfig(0.8, seed, native.SH_SAMPLE_REJECTION if c["mode"] == "rejection"
                              else native.SH_SAMPLE_COMPARE)
    s.buffers = [_device(s.p), _device(s.q) if c["mode"] == "rejection" else None, _device(s.drafts),
                 _device(s.accepted), _device(s.next)]
    s.engine = eng
    return s


def _prepare_gemv(c, seed):
    s, eng, g = State(c), _engine(), _generator(seed)
    # a normalized hidden state: unit variance
    s.x = torch.randn((c["cols"], c["inner"]), generator=g, device="cuda")
    s.y = torch.zeros((c["cols"], c["rows"]), device="cuda")
    s.w = s.own(QTensor(eng, QTYPES[c["qtype"]], _blocks(c["qtype"], c["rows"], c["inner"]), c["rows"], c["inner"]))
    s.buffers = [_device(s.x), _device(s.y)]
    s.engine = eng
    return s


_prepare_wide = _prepare_gemv


def _prepare_forward(c, seed):
    s, eng = State(c), _engine()
    shape = SHAPES[c["shape"]]
    s.model = s.own(eng.upload_weights(_image(c["shape"], c["layers"], 0)))
    s.cache = s.own(eng.allocate_kv_cache(s.model, c["ctx"] + c["cols"] + 64))
    _fill(s.cache, _cached(shape, c["layers"], c["ctx"], seed, 0))
    s.tokens = synth.tokens(seed, c["cols"], shape.n_vocab)
    s.engine = eng
    return s


def _prepare_unified(c, seed):
    s, eng = State(c), _engine()
    shape = SHAPES[c["shape"]]
    s.model = s.own(eng.upload_weights(_image(c["shape"], c["layers"], 32000)))
    s.caches = []
    for b in range(c["batch"]):
        cache = s.own(eng.allocate_kv_cache(s.model, c["ctx"] + c["cols"] + 64))
        s.caches.append(_fill(cache, _cached(shape, c["layers"], c["ctx"], seed, b)))
    s.tokens = synth.tokens(seed, c["batch"] * c["cols"], 32000)
    s.parents = _tree_parents()[: c["cols"]] * c["batch"] if c["tree"] else None
    s.engine = eng
    return s


def _prepare_spec(c, seed):
    s, eng = State(c), _engine()
    for name, i in (("target", 0), ("draft", 1)):
        model = s.own(eng.upload_weights(_image(c[name], c["layers"], c["vocab"])))
        cache = s.own(eng.allocate_kv_cache(model, c["ctx"] + 64))
        _fill(cache, _cached(SHAPES[c[name]], c["layers"], c["ctx"], seed, i))
        setattr(s, name, (model, cache))
    s.last = int(synth.tokens(seed, 1, c["vocab"])[0])
    s.sampler = SamplerConfig(0.8, seed, native.SH_SAMPLE_REJECTION)
    s.engine = eng
    return s


# ------------------------------------------------------------------ one pass


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


def _run_accept(s):
    c = s.case
    p, q, drafts, accepted, nxt = s.buffers
    s.engine.accept_sample(p, q, drafts, c["batch"], c["k"], c["vocab"], s.sampler.to_c(), accepted, nxt)
    return {"accepted": s.accepted, "next": s.next}


def _run_gemv(s):
    s.engine.gemv(s.w, s.buffers[0], s.case["cols"], s.buffers[1])
    return {"y": s.y}


def _run_wide(s):
    s.engine.gemm_wide16(s.w, s.buffers[0], s.case["cols"], s.buffers[1])
    return {"y": s.y}


def _run_forward(s):
    c = s.case
    s.cache.truncate(c["ctx"])  # the rollback of the tokens fed before
    logits, residual = s.engine.forward_full_readback(s.model, s.cache, s.tokens, c["ctx"], full_logits=c["logits"],
                                                      want_residual=c["residual"])
    return {"logits": logits, "residual": residual}


def _run_unified(s):
    c = s.case
    for cache in s.caches:
        cache.truncate(c["ctx"])
    out = s.engine.verify_unified(s.model, s.caches, s.tokens, [c["cols"]] * c["batch"], parents=s.parents,
                                  want_residual=True)
    return {"residual": out.residual, "sampled": out.sampled}


def _run_spec(s):
    c = s.case
    for _, cache in (s.target, s.draft):
        cache.truncate(c["ctx"])
    step = s.engine.decode_speculative(s.target[0], s.draft[0], s.target[1], s.draft[1], s.last, c["k"],
                                       s.sampler.to_c())
    p, q = s.engine.spec_step_logits()
    emitted = np.full(c["k"] + 1, -1, np.int64)
    emitted[: len(step.emitted)] = step.emitted
    return {"drafts": np.asarray(step.drafts, np.int64), "emitted": emitted, "p": p, "q": q}


# ------------------------------------------------------------------ work


def _layer_params(s):
    """(dense matrix weights, weights of one routed expert) of a layer."""
    hd = s.head_dim or s.n_embd // s.n_head
    attn = s.n_embd * hd * (2 * s.n_head + 2 * s.n_head_kv)
    return attn + (0 if s.n_expert else 3 * s.n_embd * s.n_ff), 3 * s.n_embd * s.expert_ff


def _forward_work(s, layers, seqs, cols, ctx, vocab, logit_cols):
    """One forward of seqs x cols columns: the weights once, the cached K/V once, the logits written."""
    hd = s.head_dim or s.n_embd // s.n_head
    bpw = BLOCK[s.wtype][1] / BLOCK[s.wtype][0]
    dense, expert = _layer_params(s)
    n = seqs * cols
    active = s.n_expert * (1 - (1 - s.n_expert_used / s.n_expert) ** n) if s.n_expert else 0
    kv = 2 * s.n_head_kv * hd * 2
    nbytes = layers * ((dense + active * expert) * bpw + seqs * (ctx + cols) * kv)
    nbytes += (vocab * s.n_embd * bpw if logit_cols else 0) + 4 * logit_cols * vocab
    flops = layers * 2.0 * n * (dense + s.n_expert_used * expert)
    flops += layers * 4.0 * s.n_head * hd * n * (ctx + (cols + 1) / 2) + 2.0 * logit_cols * vocab * s.n_embd
    return nbytes, flops


def work(case):
    c, kind = case, case["kind"]
    if kind == "accept":
        rows = c["batch"] * (2 * c["k"] + 1 if c["mode"] == "rejection" else c["k"] + 1)
        return {"bytes": 4.0 * rows * c["vocab"], "flops": 2.0 * rows * c["vocab"]}
    if kind in ("gemv", "wide"):
        elems, nbytes = BLOCK[QTYPES[c["qtype"]]]
        w = c["rows"] * c["inner"]
        return {"bytes": w * nbytes / elems + 4.0 * c["cols"] * (c["rows"] + c["inner"]), "flops": 2.0 * w * c["cols"]}
    if kind == "forward":
        s = SHAPES[c["shape"]]
        b, f = _forward_work(s, c["layers"], 1, c["cols"], c["ctx"], s.n_vocab, c["cols"] if c["logits"] else 1)
        return {"bytes": b + (4.0 * c["cols"] * s.n_embd if c["residual"] else 0), "flops": f}
    if kind == "unified":
        s = SHAPES[c["shape"]]
        n = c["batch"] * c["cols"]
        b, f = _forward_work(s, c["layers"], c["batch"], c["cols"], c["ctx"], 32000, n)
        return {"bytes": b - 4.0 * n * 32000 + 4.0 * n * s.n_embd, "flops": f}
    b, f = _forward_work(SHAPES[c["target"]], c["layers"], 1, c["k"] + 1, c["ctx"], c["vocab"], c["k"] + 1)
    bd, fd = _forward_work(SHAPES[c["draft"]], c["layers"], 1, 1, c["ctx"], c["vocab"], 1)
    return {"bytes": b + c["k"] * bd, "flops": f + c["k"] * fd}


# ------------------------------------------------------------------ tolerance


def tolerance(case):
    """Largest differences of another correct implementation of the same precision: about four times what the
    same calls give with their sums in another order."""
    kind = case["kind"]
    if kind == "accept":  # whole numbers decided by f64 probabilities
        return "exact"
    if kind == "gemv":  # f32-level sums
        return {"rel": 1e-5}
    if kind == "wide":  # f16 weights and activations, f32 sums: only the order of the sums is free
        return {"rel": 1e-5, "max": 2e-3}
    if kind == "forward" and case["cols"] == 1:  # f32-level (measured 9e-7, largest 4e-6)
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "spec" or kind == "forward" and case["cols"] < 32:
        # f16 scores and probabilities of the causal attention (measured 7e-5, largest 3e-4)
        return {"rel": 3e-4, "max": 2e-3}
    if kind == "unified" and SHAPES[case["shape"]].n_expert:
        # a routed expert at a near tie: a tenth of one column's layer output
        return {"rel": 0.015, "max": 0.5, "differ": 0.01}
    # f16 operands of every matrix product: an input's f16 rounding flips with the order of the sums before it
    return {"rel": 2e-3, "max": 0.03, "differ": 0.01}


# ------------------------------------------------------------------ exact results


def _dequant(blocks, qtype, rows, inner):
    """GGML blocks (uint8) as float64 [rows][inner] on the GPU."""
    if qtype == 0:
        return torch.from_numpy(blocks.view(np.float32).astype(np.float64)).cuda().reshape(rows, inner)
    elems, nbytes = BLOCK[qtype]
    b = torch.from_numpy(blocks).cuda().reshape(-1, nbytes)

    def half(i):
        return b[:, i:i + 2].contiguous().view(torch.float16).double()

    if qtype == native.GGML_Q8_0:
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, inner)
    if qtype == native.GGML_Q6_K:
        ql, qh = b[:, :128].reshape(-1, 2, 1, 64), b[:, 128:192].reshape(-1, 2, 32)
        low = torch.cat([ql & 15, ql >> 4], 2).reshape(-1, 2, 4, 32)
        high = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (low | (high << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
        return (half(208) * sc * q.reshape(-1, 256)).reshape(rows, inner)
    s = b[:, 4:16].int()  # Q4_K and Q5_K: 6-bit scales and minimums of 8 groups of 32
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, nbytes - 128:].reshape(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if qtype == native.GGML_Q5_K:
        qh = b[:, 16:48].reshape(-1, 1, 32)
        q = q | torch.cat([((qh >> i) & 1) << 4 for i in range(8)], 1)
    w = (half(0) * sc)[:, :, None] * q.double() - (half(2) * mn)[:, :, None]
    return w.reshape(rows, inner)


def _tensors(image):
    """name -> (type, dimensions, bytes) of a GGUF v3 image."""
    raw, at = image.bytes(), 8

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, raw, at)
        at += struct.calcsize("<" + fmt)
        return v[0]

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(raw[at - n:at]).decode()

    n_tensors, n_meta = take("Q"), take("Q")
    for _ in range(n_meta):
        text()
        vt = take("I")
        text() if vt == 8 else take("I")
    infos = []
    for _ in range(n_tensors):
        name = text()
        dims = [take("Q") for _ in range(take("I"))]
        infos.append((name, take("I"), dims, take("Q")))
    base = (at + 31) // 32 * 32
    out = {}
    for name, qt, dims, off in infos:
        elems, nbytes = BLOCK[qt]
        out[name] = (qt, dims, raw[base + off: base + off + math.prod(dims) // elems * nbytes])
    return out


def _rope(x, pos, base, neox):
    """x [n][heads][hd] rotated at pos [n]."""
    hd = x.shape[-1]
    th = pos[:, None].double() * base ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    cos, sin = th.cos()[:, None], th.sin()[:, None]
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    u, v = a * cos - b * sin, a * sin + b * cos
    return torch.cat([u, v], -1) if neox else torch.stack([u, v], -1).flatten(-2)


def _exact_forward(image, shape, layers, tokens, seqs, logit_cols):
    """(residual, logits of the columns logit_cols) in 64 bits. seqs: per sequence (columns, cached K/V rows
    [layer][2][ctx][n_kv][hd] as f16 bits, parents or None)."""
    t = _tensors(image)
    hd = shape.head_dim or shape.n_embd // shape.n_head
    nh, nkv = shape.n_head, shape.n_head_kv

    def w(name, e=None):
        qt, dims, raw = t[name]
        if e is not None:
            raw = raw[len(raw) // dims[2] * e: len(raw) // dims[2] * (e + 1)]
        return _dequant(raw, qt, dims[1] if len(dims) > 1 else 1, dims[0])

    def norm(x, name):
        return x / (x.square().mean(-1, keepdim=True) + shape.rms_eps).sqrt() * w(name)

    qt, dims, raw = t["token_embd.weight"]
    row = dims[0] // BLOCK[qt][0] * BLOCK[qt][1]
    rows = raw.reshape(-1, row)[np.asarray(tokens, np.int64)]
    x = _dequant(np.ascontiguousarray(rows).reshape(-1), qt, len(tokens), dims[0])
    pos, masks, at = torch.zeros(len(tokens), device="cuda"), [], 0
    for n, kv, parents in seqs:
        ctx = kv.shape[2]
        seen = torch.tril(torch.ones((n, n), dtype=torch.bool, device="cuda"))
        depth = list(range(n))
        if parents is not None:
            seen = torch.eye(n, dtype=torch.bool, device="cuda")
            for i, p in enumerate(parents):
                depth[i] = depth[p] + 1 if p >= 0 else 0
                if p >= 0:
                    seen[i] |= seen[p]
        pos[at:at + n] = torch.tensor(depth, device="cuda") + ctx
        masks.append(torch.cat([torch.ones((n, ctx), dtype=torch.bool, device="cuda"), seen], 1))
        at += n
    for layer in range(layers):
        p = f"blk.{layer}."
        h = norm(x, p + "attn_norm.weight")
        q, k, v = ((h @ w(p + f"attn_{m}.weight").T).reshape(len(tokens), -1, hd) for m in "qkv")
        if shape.arch:
            q, k = norm(q, p + "attn_q_norm.weight"), norm(k, p + "attn_k_norm.weight")
        q, k = _rope(q, pos, shape.rope_base, shape.arch > 0), _rope(k, pos, shape.rope_base, shape.arch > 0)
        outs, at = [], 0
        for (n, kv, _), mask in zip(seqs, masks):
            old = torch.from_numpy(kv[layer].view(np.float16)).cuda().double()
            kk = torch.cat([old[0], k[at:at + n]])
            vv = torch.cat([old[1], v[at:at + n]])
            o = torch.empty((n, nh, hd), dtype=torch.float64, device="cuda")
            for g in range(nkv):  # the query heads of one key head
                qq = q[at:at + n, g * nh // nkv:(g + 1) * nh // nkv].transpose(0, 1).contiguous()
                s = (qq.reshape(-1, hd) @ kk[:, g].contiguous().T).reshape(-1, n, kk.shape[0]) / math.sqrt(hd)
                a = s.masked_fill(~mask, -math.inf).softmax(-1)
                o[:, g * nh // nkv:(g + 1) * nh // nkv] = (
                    (a.reshape(-1, kk.shape[0]) @ vv[:, g].contiguous()).reshape(-1, n, hd).transpose(0, 1))
            outs.append(o.reshape(n, -1))
            at += n
        x = x + torch.cat(outs) @ w(p + "attn_output.weight").T
        h = norm(x, p + "ffn_norm.weight")
        if shape.n_expert:
            prob = (h @ w(p + "ffn_gate_inp.weight").T).softmax(-1)
            top, ids = prob.topk(shape.n_expert_used, -1)
            top = top / top.sum(-1, keepdim=True)
            for e in range(shape.n_expert):
                col, j = (ids == e).nonzero(as_tuple=True)
                if col.numel():
                    he = h[col]
                    f = torch.nn.functional.silu(he @ w(p + "ffn_gate_exps.weight", e).T)
                    f = f * (he @ w(p + "ffn_up_exps.weight", e).T)
                    x.index_add_(0, col, (f @ w(p + "ffn_down_exps.weight", e).T) * top[col, j][:, None])
        else:
            f = torch.nn.functional.silu(h @ w(p + "ffn_gate.weight").T) * (h @ w(p + "ffn_up.weight").T)
            x = x + f @ w(p + "ffn_down.weight").T
    head = "output.weight" if "output.weight" in t else "token_embd.weight"
    return x, norm(x[logit_cols], "output_norm.weight") @ w(head).T if logit_cols else None


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("gemv", "wide"):
        x = torch.randn((c["cols"], c["inner"]), generator=_generator(seed), device="cuda").double()
        w = _dequant(_blocks(c["qtype"], c["rows"], c["inner"]), QTYPES[c["qtype"]], c["rows"], c["inner"])
        return {"y": x @ w.T}
    if kind == "forward":
        shape = SHAPES[c["shape"]]
        kv = _cached(shape, c["layers"], c["ctx"], seed, 0)
        cols = list(range(c["cols"])) if c["logits"] else [c["cols"] - 1]
        x, logits = _exact_forward(_image(c["shape"], c["layers"], 0), shape, c["layers"],
                                   synth.tokens(seed, c["cols"], shape.n_vocab), [(c["cols"], kv, None)], cols)
        return {"logits": logits, "residual": x if c["residual"] else None}
    if kind == "unified":
        shape = SHAPES[c["shape"]]
        parents = _tree_parents()[: c["cols"]] if c["tree"] else None
        seqs = [(c["cols"], _cached(shape, c["layers"], c["ctx"], seed, b), parents) for b in range(c["batch"])]
        x, _ = _exact_forward(_image(c["shape"], c["layers"], 32000), shape, c["layers"],
                              synth.tokens(seed, c["batch"] * c["cols"], 32000), seqs, None)
        return {"residual": x, "sampled": None}
    return None  # drawn tokens, and logits that follow from them
