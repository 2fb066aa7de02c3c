"""The measured cases of the prefix-LM attention library.

Each case is one call path that a training or serving program takes through the
public entry points of ``mimir_amd``:

* ``step``  -- ``flash_attn_varlen_prefixlm`` and its gradients (a training step's
  attention), returning O, dQ, dK and dV;
* ``eval``  -- the same forward without gradients (validation), returning O;
* ``layer`` -- ``gated_attention`` and the gradient of the fused projection;
* ``cache`` -- ``attention_with_cache`` (decode and chunked prefill), returning the
  attention output and the updated cache.

A case holds everything that shapes the work: the packing (``docs`` and its
seed), head counts, head dimension, data type and options.  ``prepare`` draws
the values from its own seed.
"""

from __future__ import annotations

import math
import random

import torch

import mimir_amd
from mimir_amd.cache import Cache, attention_with_cache

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # Serving, one user: a new token against a few hundred cached ones. Launch latency.
        dict(name="decode_single", kind="cache", batch=1, new=1, hq=16, hkv=4, d=128, positions=4096, min_len=700,
             max_len=700, len_seed=1, causal=True, rows=False),
        # Serving, a small batch of conversations of mixed length.
        dict(name="decode_batch", kind="cache", batch=8, new=1, hq=16, hkv=4, d=128, positions=4096, min_len=1024,
             max_len=3583, len_seed=2, causal=True, rows=False),
        # Serving, a full batch addressed through row indices: the cache read is the work.
        dict(name="decode_wide", kind="cache", batch=64, new=1, hq=16, hkv=4, d=128, positions=8192, min_len=512,
             max_len=8000, len_seed=3, causal=True, rows=True),
        # Chunked prefill: 512 new tokens per row onto a filled cache.
        dict(name="prefill_chunk", kind="cache", batch=8, new=512, hq=16, hkv=4, d=128, positions=4096, min_len=1536,
             max_len=1536, len_seed=4, causal=True, rows=False),
        # Fine-tuning on a few short ragged documents with padding rows: launches and host time.
        dict(name="step_short", kind="step", dtype="bf16", tokens=1000, pad=24, hq=2, hkv=2, d=128, doc_min=17,
             doc_max=400, doc_seed=5, prefix="uniform", causal=False, outlier=0.0),
        # The XXS model's training row: two heads over packed documents.
        dict(name="step_xxs", kind="step", dtype="bf16", tokens=24576, pad=0, hq=2, hkv=2, d=128, doc_min=128,
             doc_max=4096, doc_seed=6, prefix="uniform", causal=False, outlier=0.0),
        # The headline training shape: 8 sequences of 2048, grouped heads.
        dict(name="step_gqa", kind="step", dtype="bf16", tokens=16384, pad=0, hq=16, hkv=4, d=128, doc_min=2048,
             doc_max=2048, doc_seed=7, prefix="uniform", causal=False, outlier=0.0),
        # Many sequences at head_dim 64, each either all prefix or all causal.
        dict(name="step_small_head", kind="step", dtype="bf16", tokens=65536, pad=0, hq=8, hkv=8, d=64, doc_min=1024,
             doc_max=1024, doc_seed=8, prefix="ends", causal=False, outlier=0.0),
        # One long document whose keys hold an outlier channel (P and dS carried as two halves).
        dict(name="step_long", kind="step", dtype="bf16", tokens=32768, pad=0, hq=32, hkv=8, d=128, doc_min=32768,
             doc_max=32768, doc_seed=9, prefix="quarter", causal=False, outlier=20.0),
        # Full-precision training on a small batch.
        dict(name="step_fp32", kind="step", dtype="fp32", tokens=2048, pad=0, hq=8, hkv=8, d=64, doc_min=512,
             doc_max=512, doc_seed=10, prefix="uniform", causal=False, outlier=0.0),
        # Validation: the forward alone, plain causal, over ragged documents.
        dict(name="eval_causal", kind="eval", dtype="bf16", tokens=8191, pad=100, hq=16, hkv=4, d=128, doc_min=64,
             doc_max=3000, doc_seed=11, prefix="uniform", causal=True, outlier=0.0),
        # The attention layer from the fused projection: split, RoPE, attention, output gate, and back.
        dict(name="layer_packed", kind="layer", dtype="bf16", tokens=16384, pad=0, hq=16, hkv=4, d=128, doc_min=128,
             doc_max=4096, doc_seed=12, prefix="uniform", causal=False, outlier=0.0, rope=True),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 0.5 / hi))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "cache", "cache", "eval", "layer", "fp32"])
    if kind == "cache":
        hq, hkv, d = rng.choice([(16, 4, 128), (8, 8, 64), (2, 2, 128), (32, 8, 128), (8, 2, 64)])
        new = 1 if rng.random() < 0.6 else _log(rng, 2, 1024)
        batch = _log(rng, 1, 64 if new == 1 else 8)
        positions = max(new + 64, _log(rng, 256, 8192))
        hi = rng.randint(1, positions - new)
        return dict(kind="cache", batch=batch, new=new, hq=hq, hkv=hkv, d=d, positions=positions,
                    min_len=rng.randint(0, hi), max_len=hi, len_seed=rng.randrange(1 << 20),
                    causal=rng.random() < 0.8, rows=rng.random() < 0.3)
    if kind == "fp32":
        hq, hkv, d = rng.choice([(8, 8, 64), (2, 2, 128), (8, 2, 64), (4, 1, 128), (4, 4, 32)])
        tokens = _log(rng, 128, 4096)
        case = dict(kind=rng.choice(["step", "step", "eval"]), dtype="fp32")
    else:
        hq, hkv, d = rng.choice([(16, 4, 128), (2, 2, 128), (8, 8, 64), (32, 8, 128), (4, 1, 128), (6, 6, 128)])
        tokens = _log(rng, 256, 32768)
        case = dict(kind=kind, dtype="bf16")
    doc_max = min(tokens, _log(rng, 64, 32768 if case["kind"] == "step" and case["dtype"] == "bf16" else 4096))
    case.update(tokens=tokens, pad=rng.choice([0, 0, rng.randint(1, 63)]), hq=hq, hkv=hkv, d=d,
                doc_min=rng.randint(1, doc_max), doc_max=doc_max, doc_seed=rng.randrange(1 << 20),
                prefix=rng.choice(["uniform", "uniform", "ends", "quarter"]), causal=rng.random() < 0.2,
                outlier=20.0 if case["dtype"] == "bf16" and kind != "layer" and rng.random() < 0.1 else 0.0)
    if kind == "layer":
        case["rope"] = rng.random() < 0.8
    while work(case)["flops"] > 2e13:  # one document of the whole row, all prefix: less than the longest listed
        case["tokens"] //= 2
    return case


# ---------------------------------------------------------------- metadata

def _documents(case):
    """Document and prefix lengths of one packed row."""
    rng = random.Random(case["doc_seed"])
    left, lens, prefixes = case["tokens"], [], []
    while left > 0:
        n = min(left, rng.randint(case["doc_min"], case["doc_max"]))
        p = {"uniform": rng.randint(0, n), "ends": n * rng.randint(0, 1), "quarter": n // 4}[case["prefix"]]
        lens.append(n)
        prefixes.append(p)
        left -= n
    return lens, prefixes


def _seq_info(case, device):
    """The metadata keywords as a training loop passes them (device tensors, CPU scalars)."""
    lens, prefixes = _documents(case)
    rows = max(case["tokens"] + case["pad"], len(lens) + 1)
    pad = lambda x: torch.tensor(x + [0] * (rows - len(x)), dtype=torch.int32, device=device)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    causal = [n - p for n, p in zip(lens, prefixes)]
    scalar = lambda x: torch.tensor(x, dtype=torch.int64)
    return dict(prefix_lens=pad(prefixes), causal_lens=pad(causal), cu_seqlens=pad(cu), total_seqlen=scalar(cu[-1]),
                numseqs=scalar(len(lens)), max_seqlen_prefix=scalar(max(prefixes)),
                max_seqlen_causal=scalar(max(causal)), max_seqlen_all=scalar(max(lens)))


def _lengths(case):
    rng = random.Random(case["len_seed"])
    return [rng.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"])]


def _row_indices(case):
    rows = list(range(case["batch"]))
    if case["rows"]:
        random.Random(case["len_seed"] + 1).shuffle(rows)
    return rows


# ---------------------------------------------------------------- inputs and calls

def _normal(gen, *shape):
    # projections of normalised activations: near normal, without far tails
    return torch.randn(shape, generator=gen, device=gen.device).clamp_(-5.0, 5.0)


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    if case["kind"] == "cache":
        b, s, n = case["batch"], case["new"], case["positions"]
        bf = lambda *shape: _normal(gen, *shape).to(torch.bfloat16)
        cache = Cache(bf(b, n, hkv, d), bf(b, n, hkv, d))
        rows = torch.tensor(_row_indices(case), device=device) if case["rows"] else None
        return dict(case=case, q=bf(b, s, hq, d), k=bf(b, s, hkv, d), v=bf(b, s, hkv, d), cache=cache,
                    lengths=torch.tensor(_lengths(case), device=device), rows=rows)
    dtype = _DTYPES[case["dtype"]]
    t = case["tokens"] + case["pad"]
    state = dict(case=case, info=_seq_info(case, device))
    if case["kind"] == "layer":
        x = _normal(gen, t, (2 * hq + 2 * hkv) * d).to(dtype)
        state.update(gqkv=x.requires_grad_(True), dout=_normal(gen, t, hq * d).to(dtype), cos_sin=None)
        if case["rope"]:
            state["cos_sin"] = _rope_tables(case, t, device)
        return state
    q, k, v = _normal(gen, t, hq, d), _normal(gen, t, hkv, d), _normal(gen, t, hkv, d)
    if case["outlier"]:
        channel = seed % d
        q[..., channel] *= case["outlier"]
        k[..., channel] *= case["outlier"]
    grad = case["kind"] == "step"
    q, k, v = (x.to(dtype).requires_grad_(grad) for x in (q, k, v))
    state.update(q=q, k=k, v=v)
    if grad:
        state["dout"] = _normal(gen, t, hq, d).to(dtype)
    return state


def _rope_tables(case, t, device):
    """cos and sin [tokens, head_dim], positions counted from each document's start."""
    pos = [i for n in _documents(case)[0] for i in range(n)] + [0] * case["pad"]
    d = case["d"]
    freq = 10000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)
    angle = torch.tensor(pos, dtype=torch.float64)[:, None] * freq[None, :]
    angle = torch.cat((angle, angle), dim=1)
    return angle.cos().float().to(device), angle.sin().float().to(device)


def run(state):
    case = state["case"]
    if case["kind"] == "cache":
        out = attention_with_cache(state["q"], state["k"], state["v"], state["cache"], state["lengths"],
                                   case["causal"], state["rows"])
        return out, state["cache"].keys, state["cache"].values
    if case["kind"] == "layer":
        y = mimir_amd.gated_attention(state["gqkv"], state["cos_sin"], case["hq"], case["hkv"], case["causal"],
                                      **state["info"])
        return y, torch.autograd.grad(y, state["gqkv"], state["dout"])[0]
    q, k, v = state["q"], state["k"], state["v"]
    if case["kind"] == "eval":
        with torch.no_grad():
            return mimir_amd.flash_attn_varlen_prefixlm(q, k, v, case["causal"], **state["info"])
    out = mimir_amd.flash_attn_varlen_prefixlm(q, k, v, case["causal"], **state["info"])
    return (out, *torch.autograd.grad(out, (q, k, v), state["dout"]))


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    if case["kind"] == "cache":
        b, s = case["batch"], case["new"]
        lens = _lengths(case)
        kv = sum(n + s for n in lens)
        pairs = sum(n * s + (s * (s + 1) // 2 if case["causal"] else s * s) for n in lens)
        # the cached keys and values, the new rows in and into the cache, q and the output
        return dict(bytes=2 * (2 * (kv - b * s) * hkv * d + 4 * b * s * hkv * d + 2 * b * s * hq * d),
                    flops=4 * d * hq * pairs)
    lens, prefixes = _documents(case)
    if case["causal"]:
        prefixes = [0] * len(lens)
    pairs = sum((n * n + n + p * p - p) // 2 for n, p in zip(lens, prefixes))
    t, e = case["tokens"] + case["pad"], 2 if case["dtype"] == "bf16" else 4
    q, kv = e * t * hq * d, e * t * hkv * d
    if case["kind"] == "eval":
        return dict(bytes=2 * q + 2 * kv, flops=4 * d * hq * pairs)
    if case["kind"] == "layer":
        # gqkv and the output; then the same with its gradient and the output's
        return dict(bytes=(3 * q + 2 * kv) + (2 * (2 * q + 2 * kv) + 2 * q) + (16 * t * d if case["rope"] else 0),
                    flops=14 * d * hq * pairs)
    return dict(bytes=(2 * q + 2 * kv) + (4 * q + 4 * kv), flops=14 * d * hq * pairs)


def tolerance(case):
    # about four times the relative error against `exact`: 4e-7 to 8e-7 in fp32, 2.0e-3 to 2.5e-3 in
    # bf16, and 4e-3 to 5e-3 for the layer, which rounds to bf16 after RoPE, attention and gate as well
    if case["kind"] != "cache" and case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 2e-2 if case["kind"] == "layer" else 1e-2, "max": 0.3}


# ---------------------------------------------------------------- 64-bit results

def _attend(q, k, v, start, prefix, dout=None):
    """All heads of one document in 64 bits: queries [Hq, n, D] at key positions start.., each
    seeing the keys [Hkv, m, D] before max(prefix, its position + 1). O or (O, dQ, dK, dV)."""
    scale = 1.0 / math.sqrt(q.shape[2])
    group = q.shape[0] // k.shape[0]
    k, v = (x.repeat_interleave(group, dim=0) for x in (k, v))
    keys = torch.arange(k.shape[1], device=q.device)
    out = torch.empty_like(q)
    if dout is not None:
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    heads = max(1, min(q.shape[0], (1 << 27) // (min(q.shape[1], 2048) * k.shape[1])))  # 1 GiB of scores at a time
    for h in range(0, q.shape[0], heads):
        h = slice(h, h + heads)
        for a in range(0, q.shape[1], 2048):
            b = min(q.shape[1], a + 2048)
            kend = (start + 1 + torch.arange(a, b, device=q.device)).clamp_(min=prefix)
            n = max(prefix, start + b)
            p = (q[h, a:b] @ k[h, :n].mT).mul_(scale)
            p.masked_fill_(keys[None, :n] >= kend[:, None], -math.inf)
            p = torch.softmax(p, dim=2)
            out[h, a:b] = p @ v[h, :n]
            if dout is not None:
                do = dout[h, a:b]
                dv[h, :n] += p.mT @ do
                ds = (do @ v[h, :n].mT).sub_((do * out[h, a:b]).sum(2, keepdim=True)).mul_(p).mul_(scale)
                dq[h, a:b] = ds @ k[h, :n]
                dk[h, :n] += ds.mT @ q[h, a:b]
    if dout is None:
        return out
    return out, dq, *(x.unflatten(0, (-1, group)).sum(1) for x in (dk, dv))


def _attention(case, q, k, v, dout=None):
    """A packed row [T, H, D], document by document."""
    rows = (q, k, v) if dout is None else (q, k, v, dout)
    outs = [torch.zeros_like(x) for x in ((q,) if dout is None else (q, q, k, v))]
    at = 0
    for n, p in zip(*_documents(case)):
        q_, k_, v_, *do = (x[at:at + n].transpose(0, 1) for x in rows)
        got = _attend(q_, k_, v_, 0, 0 if case["causal"] else p, *do)
        for o, x in zip(outs, got if do else (got,)):
            o[at:at + n] = x.transpose(0, 1)
        at += n
    return outs[0] if dout is None else tuple(outs)


def _rotate(x, cos, sin, inverse=False):
    half = x.shape[-1] // 2
    if inverse:
        y = x * sin[:, None]
        return x * cos[:, None] + torch.cat((y[..., half:], -y[..., :half]), dim=-1)
    return x * cos[:, None] + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin[:, None]


def exact(case, seed):
    state = prepare(case, seed)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    with torch.no_grad():
        if case["kind"] == "cache":
            keys, values = state["cache"].keys, state["cache"].values
            q = state["q"].double()
            out, s = torch.empty_like(q), case["new"]
            for b, (n, row) in enumerate(zip(_lengths(case), _row_indices(case))):
                keys[row, n:n + s], values[row, n:n + s] = state["k"][b], state["v"][b]
                out[b] = _attend(*(x.double().transpose(0, 1) for x in (q[b], keys[row, :n + s], values[row, :n + s])),
                                 n, 0 if case["causal"] else n + s).transpose(0, 1)
            return out, keys.double(), values.double()
        if case["kind"] == "layer":
            t = case["tokens"] + case["pad"]
            x = state["gqkv"].double().view(t, 2 * hq + 2 * hkv, d)
            gate, q, k, v = x.split((hq, hq, hkv, hkv), dim=1)
            if case["rope"]:
                cos, sin = (c.double() for c in state["cos_sin"])
                q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
            s, dy = torch.sigmoid(gate), state["dout"].double().view(t, hq, d)
            out, dq, dk, dv = _attention(case, q, k, v, dy * s)
            if case["rope"]:
                dq, dk = _rotate(dq, cos, sin, True), _rotate(dk, cos, sin, True)
            return (s * out).view(t, hq * d), torch.cat((dy * out * s * (1 - s), dq, dk, dv), dim=1).view(t, -1)
        q, k, v = (state[x].double() for x in "qkv")
        if case["kind"] == "eval":
            return _attention(case, q, k, v)
        return _attention(case, q, k, v, state["dout"].double())
