"""The attention work that users of this package give it, as measurable cases.

Three kinds of pass, each through the public entry points:

  forward  ``flash_attn_forward_gqa``: inference.  Decode steps against a KV
           cache, chunks of a long prompt against the cache built so far, and
           whole-prompt prefill; q and k / v come from different projections,
           so head counts differ (grouped queries).
  train    ``flash_attn`` (equal heads, the reference's signature) or
           ``flash_attn_gqa``, forward and backward through autograd: the
           attention of a training step, causal (decoders) and not
           (encoders, cross-attention), contiguous or as the transposed
           (B, H, S, D) views that HuggingFace models pass.
  rope     ``apply_rotary_qk``, forward and backward through autograd: the
           QK-norm + rotary prologue before the attention of a layer.

Inputs are N(0, 1), as activations after a norm are, on the GPU, from the
seed alone.
"""
from __future__ import annotations

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "flash-attn-volta_amd"))

from flash_attn_volta import (apply_rotary_qk, flash_attn, flash_attn_forward_gqa,  # noqa: E402
                              flash_attn_gqa)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _attn(kind, B, Sq, Sk, H, Hk, D, causal, dtype, layout="bshd"):
    return {"kind": kind, "B": B, "Sq": Sq, "Sk": Sk, "H": H, "Hk": Hk, "D": D,
            "causal": causal, "dtype": dtype, "layout": layout}


def listed():
    cases = {
        # one user's next token against a 4k cache: the smallest call, where
        # launches and latency are the time
        "decode_one": _attn("forward", 1, 1, 4096, 32, 8, 128, True, "bf16"),
        # the same step for a batch of 32 users, caches of some 3000 tokens:
        # reading the cache is the time
        "decode_batch": _attn("forward", 32, 1, 3001, 32, 8, 128, True, "bf16"),
        # the next 256 tokens of a long prompt against the 8k already cached
        "prefill_chunk": _attn("forward", 1, 256, 8448, 32, 8, 128, True, "bf16"),
        # a whole prompt of odd length
        "prefill": _attn("forward", 1, 6001, 6001, 32, 8, 128, True, "bf16"),
        # the smallest training step of the repository's configurations
        "train_small": _attn("train", 4, 512, 512, 4, 4, 32, True, "fp16"),
        # an image encoder's layer: 14 x 14 patches and a class token
        "train_encoder": _attn("train", 32, 197, 197, 12, 12, 64, False, "fp16"),
        # a 12-head decoder at its full context, tensors as transposed views
        "train_12_heads": _attn("train", 8, 1024, 1024, 12, 12, 64, True, "fp16", "bhsd"),
        # the repository's benchmark
        "train_bench": _attn("train", 1, 4096, 4096, 16, 16, 64, True, "fp16"),
        # the repository's D = 128 configuration, every key visible
        "train_full_128": _attn("train", 1, 4096, 4096, 8, 8, 128, False, "fp16"),
        # a grouped-query decoder layer (28 query heads on 4 key/value
        # heads) at a ragged length
        "train_gqa": _attn("train", 1, 4000, 4000, 28, 4, 128, True, "bf16"),
        # the longest context of the repository's benchmark: the largest call
        "train_long": _attn("train", 1, 16384, 16384, 16, 16, 128, True, "fp16"),
        # the normed rotary prologue of a 4k grouped-query layer
        "rope_norm": {"kind": "rope", "B": 1, "S": 4096, "H": 32, "Hk": 8, "D": 128,
                      "norm": True, "dtype": "bf16"},
    }
    return [dict(c, name=n) for n, c in cases.items()]


# Head counts (query, key/value) that models use.
GQA_HEADS = ((32, 8), (28, 4), (16, 8), (14, 2), (64, 8), (32, 4), (32, 32))
MHA_HEADS = (4, 6, 8, 12, 16, 20, 25, 32)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """One more case: a family of listed(), its sizes anew."""
    most = max((work(c)["flops"], work(c)["bytes"]) for c in listed())
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= most[0] and w["bytes"] <= 2e9:
            return c


def _draw(rng):
    family = rng.choice(("decode", "chunk", "prefill", "small", "encoder", "decoder", "decoder",
                         "gqa", "rope"))
    dtype = rng.choice(("fp16", "bf16"))
    if family in ("decode", "chunk", "prefill"):
        H, Hk = rng.choice(GQA_HEADS)
        D = 64 if H == 14 else rng.choice((64, 128, 128))
        if family == "decode":
            Sq = rng.choice((1, 1, 1, 2, 4, 8))
            return _attn("forward", _log_int(rng, 1, 64), Sq, _log_int(rng, 256, 32768), H, Hk, D,
                         True, dtype)
        if family == "chunk":
            Sq = _log_int(rng, 16, 2048)
            return _attn("forward", _log_int(rng, 1, 4), Sq, Sq + _log_int(rng, 256, 16384), H, Hk,
                         D, True, dtype)
        S = _log_int(rng, 100, 16384)
        return _attn("forward", _log_int(rng, 1, 4), S, S, H, Hk, D, True, dtype)
    if family == "rope":
        H, Hk = rng.choice(GQA_HEADS)
        return {"kind": "rope", "B": _log_int(rng, 1, 4), "S": _log_int(rng, 64, 8192), "H": H,
                "Hk": Hk, "D": 64 if H == 14 else 128, "norm": rng.random() < 0.5, "dtype": dtype}
    if family == "gqa":
        H, Hk = rng.choice(GQA_HEADS[:6])
        S = _log_int(rng, 256, 8192)
        return _attn("train", _log_int(rng, 1, 4), S, S, H, Hk, 64 if H == 14 else 128, True,
                     dtype)
    # equal heads: the reference's own signature, fp16
    if family == "small":
        S, D = _log_int(rng, 32, 512), rng.choice((16, 32, 64))
        return _attn("train", _log_int(rng, 1, 8), S, S, rng.choice((2, 4, 8)), 0, D,
                     rng.random() < 0.7, "fp16", rng.choice(("bshd", "bhsd")))
    if family == "encoder":
        S = _log_int(rng, 50, 1600)
        Sk = S if rng.random() < 0.6 else _log_int(rng, 50, 1600)
        return _attn("train", _log_int(rng, 4, 64), S, Sk, rng.choice((6, 8, 12, 16)), 0, 64, False,
                     "fp16", rng.choice(("bshd", "bhsd")))
    S = _log_int(rng, 512, 12288)
    return _attn("train", _log_int(rng, 1, 8), S, S, rng.choice(MHA_HEADS), 0,
                 rng.choice((32, 64, 64, 128)), rng.random() < 0.75, "fp16",
                 rng.choice(("bshd", "bhsd")))


def _heads(c):
    return c["H"], c["Hk"] or c["H"]


def _randn(shape, dtype, gen):
    return torch.randn(shape, dtype=torch.float32, device="cuda", generator=gen).to(dtype)


def _tensor(c, S, heads, gen):
    """(B, S, heads, D) of the case's dtype and layout."""
    if c["layout"] == "bhsd":
        return _randn((c["B"], heads, S, c["D"]), DTYPES[c["dtype"]], gen).transpose(1, 2)
    return _randn((c["B"], S, heads, c["D"]), DTYPES[c["dtype"]], gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    c = case
    H, Hk = _heads(c)
    if c["kind"] == "rope":
        dt, B, S, D = DTYPES[c["dtype"]], c["B"], c["S"], c["D"]
        q, k = _randn((B, S, H, D), dt, gen), _randn((B, S, Hk, D), dt, gen)
        gq, gk = _randn((B, S, H, D), dt, gen), _randn((B, S, Hk, D), dt, gen)
        # the rotary tables of positions 0 .. S - 1, base 10000
        inv = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float32, device="cuda") / D)
        ang = torch.arange(S, dtype=torch.float32, device="cuda")[:, None] * inv
        ang = torch.cat((ang, ang), dim=-1)[None]
        wq = wk = None
        if c["norm"]:
            wq, wk = ((1 + 0.1 * _randn((D,), torch.float32, gen)).to(dt).requires_grad_()
                      for _ in range(2))
        return {"kind": "rope", "q": q.requires_grad_(), "k": k.requires_grad_(), "gq": gq,
                "gk": gk, "cos": ang.cos().to(dt), "sin": ang.sin().to(dt), "wq": wq, "wk": wk}
    q = _tensor(c, c["Sq"], H, gen)
    k = _tensor(c, c["Sk"], Hk, gen)
    v = _tensor(c, c["Sk"], Hk, gen)
    state = {"kind": c["kind"], "causal": c["causal"], "q": q, "k": k, "v": v}
    if c["kind"] == "train":
        state["do"] = _tensor(c, c["Sq"], H, gen)
        state["fn"] = (flash_attn if Hk == H and c["Sq"] == c["Sk"] and c["dtype"] == "fp16"
                       else flash_attn_gqa)
        for t in (q, k, v):
            t.requires_grad_()
    return state


def run(state):
    s = state
    if s["kind"] == "forward":
        return flash_attn_forward_gqa(s["q"], s["k"], s["v"], causal=s["causal"])
    if s["kind"] == "train":
        out = s["fn"](s["q"], s["k"], s["v"], causal=s["causal"])
        dq, dk, dv = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["do"])
        return {"out": out, "dq": dq, "dk": dk, "dv": dv}
    q, k = apply_rotary_qk(s["q"], s["k"], s["cos"], s["sin"], s["wq"], s["wk"], 1e-6)
    wanted = [t for t in (s["q"], s["k"], s["wq"], s["wk"]) if t is not None]
    grads = torch.autograd.grad((q, k), wanted, (s["gq"], s["gk"]))
    return {"q": q, "k": k, "grads": list(grads)}


def _pairs(c):
    """(query, key) pairs that see each other, per head (bottom-right mask)."""
    Sq, Sk = c["Sq"], c["Sk"]
    if not c["causal"]:
        return Sq * Sk
    off = Sk - Sq
    first = max(0, -off)               # queries before it see no key
    n = Sq - first
    return n * (first + off + 1) + n * (n - 1) // 2


def work(case):
    c = case
    H, Hk = _heads(c)
    B, D = c["B"], c["D"]
    if c["kind"] == "rope":
        qk = B * c["S"] * (H + Hk) * D * 2
        tables = 2 * c["S"] * D * 2
        # forward: q, k in and out; backward: their gradients in and out
        # (and, with norms, q and k again)
        return {"bytes": (5 if c["norm"] else 4) * qk + 2 * tables,
                "flops": B * c["S"] * (H + Hk) * D * (20 if c["norm"] else 6)}
    q = B * c["Sq"] * H * D * 2
    kv = 2 * B * c["Sk"] * Hk * D * 2
    pairs = B * H * _pairs(c)
    if c["kind"] == "forward":
        return {"bytes": 2 * q + kv, "flops": 4 * D * pairs}
    # out, dO and dQ beside q; the gradients of k and v; 2 products forward, 5 backward
    return {"bytes": 4 * q + 2 * kv, "flops": 14 * D * pairs}


def tolerance(case):
    # Probabilities, dS and results are rounded to 16 bits (11 significant
    # bits in fp16, 8 in bf16) between sums in 32 bits.  Measured against
    # exact(): at most 4.2e-4 (fp16) and 2.5e-3 (bf16) over the outputs of
    # the listed cases and of a few drawn ones; four times that.
    return {"rel": 1.7e-3 if case["dtype"] == "fp16" else 1e-2}


def _exact_head(q, k, v, do, causal):
    """One head in 64 bits: q (Sq, D), k, v (Sk, D) -> out and, with do, dq, dk, dv."""
    Sq, Sk, scale = q.shape[0], k.shape[0], 1.0 / math.sqrt(q.shape[1])
    rows = max(1, (1 << 26) // Sk)
    out = torch.empty_like(q)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    keys = torch.arange(Sk, device=q.device)
    for i in range(0, Sq, rows):
        j = min(Sq, i + rows)
        s = (q[i:j] @ k.T).mul_(scale)
        if causal:
            last = torch.arange(i, j, device=q.device)[:, None] + (Sk - Sq)
            s.masked_fill_(keys[None] > last, -math.inf)
        p = torch.softmax(s, dim=-1)
        out[i:j] = p @ v
        if do is not None:
            dv += p.T @ do[i:j]
            ds = do[i:j] @ v.T
            ds -= (do[i:j] * out[i:j]).sum(-1, keepdim=True)
            ds *= p
            ds *= scale
            dq[i:j] = ds @ k
            dk += ds.T @ q[i:j]
    return out, dq, dk, dv


def exact(case, seed):
    c, s = case, prepare(case, seed)
    if c["kind"] == "rope":
        return _exact_rope(c, s)
    H, Hk = _heads(c)
    train = c["kind"] == "train"
    q, k, v = (s[n].detach().double() for n in "qkv")
    do = s["do"].double() if train else None
    out, dq = torch.empty(q.shape, dtype=q.dtype, device=q.device), None
    if train:
        dq, dk, dv = (torch.zeros(t.shape, dtype=t.dtype, device=t.device) for t in (q, k, v))
    for b in range(c["B"]):
        for h in range(H):
            g = h // (H // Hk)
            r = _exact_head(q[b, :, h], k[b, :, g], v[b, :, g], do[b, :, h] if train else None,
                            c["causal"])
            out[b, :, h] = r[0]
            if train:
                dq[b, :, h] = r[1]
                dk[b, :, g] += r[2]
                dv[b, :, g] += r[3]
    return {"out": out, "dq": dq, "dk": dk, "dv": dv} if train else out


def _exact_rope(c, s):
    cos, sin = s["cos"].double()[:, :, None], s["sin"].double()[:, :, None]

    def side(x, w):
        if w is not None:
            x = w * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
        lo, hi = x.chunk(2, dim=-1)
        return x * cos + torch.cat((-hi, lo), dim=-1) * sin

    leaf = {n: s[n].detach().double().requires_grad_() for n in ("q", "k", "wq", "wk")
            if s[n] is not None}
    q, k = side(leaf["q"], leaf.get("wq")), side(leaf["k"], leaf.get("wk"))
    grads = torch.autograd.grad((q, k), list(leaf.values()), (s["gq"].double(), s["gk"].double()))
    return {"q": q.detach(), "k": k.detach(), "grads": list(grads)}
