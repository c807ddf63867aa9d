"""The attention work a user of this package has it do, as timed cases.

Each case is one call (or one training step) through the public entry points:
``kotflash_amd.attention`` with and without autograd, and the two K/V caches.
``listed()`` gives the fixed cases, ``draw()`` more of the same ranges:

- prefill: causal self-attention without gradients, 64 to 16384 tokens;
- decode: 1 to 16 query tokens against a long K/V sequence, on plain tensors
  and through the caches (append one token and attend; append a few draft
  tokens to sequences of different lengths, attend, and drop them again);
- cross: query and key sequences of different lengths, non-causal;
- train: forward and backward of each of these masks through autograd.

Head dims 64 to 128, fp16 and bf16, MHA to MQA; tensors are either contiguous
[B, H, S, D] or the transposed views that a model's projections give
(``layout="bshd"``). Values are N(0, 1), the scale of normalised projections.
"""
from __future__ import annotations

import math
import random

import torch

from kotflash_amd import attention
from kotflash_amd.cache import PreallocatedKVCache, RaggedKVCache

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(kind, b, hq, hkv, sq, sk, d, dtype, causal=False, layout="bhsd", capacity=0, name=None):
    case = {"kind": kind, "b": b, "hq": hq, "hkv": hkv, "sq": sq, "sk": sk, "d": d,
            "dtype": dtype, "causal": causal, "layout": layout, "capacity": capacity}
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # One generated token of a small model in an interactive session: the
        # smallest call there is, append and attention over 2000 tokens.
        _case("step", 2, 8, 2, 1, 2000, 64, "fp16", capacity=4096, name="step_2k"),
        # The same model deep into a long document, cache read in place.
        _case("infer", 2, 8, 2, 1, 16384, 64, "fp16", name="decode_16k"),
        # A serving batch of a larger GQA model: all K/V bytes come from HBM.
        _case("infer", 16, 32, 8, 1, 8192, 128, "bf16", name="decode_batch"),
        # Speculative decoding of eight sequences of their own lengths: four
        # draft tokens each are appended, attended to, and dropped again.
        _case("verify", 8, 32, 8, 4, 8000, 64, "fp16", capacity=8192, name="verify_ragged"),
        # A short prompt.
        _case("infer", 2, 8, 2, 512, 512, 64, "fp16", causal=True, name="prefill_512"),
        # One ordinary prompt of a GQA model, of no round length, on the
        # transposed views its projections give.
        _case("infer", 1, 32, 8, 1777, 1777, 128, "bf16", causal=True, layout="bshd",
              name="prefill_1777"),
        # A long document's prompt: the largest call.
        _case("infer", 1, 16, 4, 16384, 16384, 128, "fp16", causal=True, name="prefill_16k"),
        # A block of decoder tokens over an encoder's output.
        _case("infer", 2, 16, 16, 100, 3000, 64, "bf16", name="cross_100x3000"),
        # A layer of an ordinary language-model training step.
        _case("train", 4, 12, 12, 1000, 1000, 64, "bf16", causal=True, layout="bshd",
              name="train_1000"),
        # Long-context GQA training.
        _case("train", 2, 16, 4, 4096, 4096, 128, "bf16", causal=True, name="train_4k"),
        # An image encoder's layer: bidirectional, head dim 72.
        _case("train", 4, 12, 12, 2048, 2048, 72, "fp16", name="train_d72"),
        # Cross-attention training, decoder tokens over an encoder's output.
        _case("train", 4, 8, 8, 300, 1500, 80, "fp16", name="train_cross"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above, no larger than the largest listed
    one of its kind."""
    kind = rng.choice(["step", "decode", "verify", "prefill", "cross", "train", "train",
                       "train_cross"])
    dtype = rng.choice(["fp16", "bf16"])
    d = rng.choice([64, 64, 72, 80, 96, 112, 128, 128])
    layout = rng.choice(["bhsd", "bshd"])
    while True:
        hkv = rng.choice([1, 2, 4, 8, 12, 16])
        hq = hkv * rng.choice([1, 1, 2, 4, 8])
        b = rng.choice([1, 2, 3, 4, 8, 16])
        if hq > 32:
            continue
        if kind == "step":
            sk = _log(rng, 1024, 16384)
            case = _case("step", b, hq, hkv, 1, sk, d, dtype, capacity=sk + rng.randint(1, 2048))
        elif kind == "verify":
            sk = _log(rng, 1100, 8000)
            n = rng.randint(1, 16)
            case = _case("verify", b, hq, hkv, n, sk, d, dtype, capacity=sk + n + rng.randint(0, 512))
        elif kind == "decode":
            case = _case("infer", b, hq, hkv, rng.choice([1, 1, 1, 2, 4, 16]),
                         _log(rng, 1024, 32768), d, dtype)
        elif kind == "prefill":
            s = _log(rng, 64, 16384)
            case = _case("infer", b, hq, hkv, s, s, d, dtype, causal=True, layout=layout)
        elif kind == "cross":
            case = _case("infer", b, hq, hkv, _log(rng, 20, 2048), _log(rng, 64, 8192), d, dtype,
                         layout=layout)
        elif kind == "train":
            s = _log(rng, 256, 4096)
            case = _case("train", b, hq, hkv, s, s, d, dtype, causal=rng.random() < 0.6,
                         layout=layout)
        else:
            case = _case("train", b, hq, hkv, _log(rng, 64, 2048), _log(rng, 256, 4096), d, dtype,
                         layout=layout)
        w = work(case)
        limit = 5.0e11 if kind.startswith("train") else 1.1e12
        if w["flops"] <= limit and w["bytes"] <= 5.4e8:
            return case


def _lengths(case, seed):
    """Populated lengths of a ragged cache: evenly spread from an eighth of
    the longest up, in the seed's order."""
    b, top = case["b"], case["sk"]
    lens = [top - (top - top // 8) * i // b for i in range(b)]
    random.Random(seed).shuffle(lens)
    return lens


def _inputs(case, seed):
    """The call's tensors, made on the GPU from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, b, d = DTYPES[case["dtype"]], case["b"], case["d"]

    def make(heads, s):
        if case["layout"] == "bshd":
            return torch.randn((b, s, heads, d), device="cuda", dtype=dt, generator=g).transpose(1, 2)
        return torch.randn((b, heads, s, d), device="cuda", dtype=dt, generator=g)

    t = {"q": make(case["hq"], case["sq"])}
    if case["kind"] in ("step", "verify"):
        t["k"] = make(case["hkv"], case["capacity"])
        t["v"] = make(case["hkv"], case["capacity"])
        t["new_k"] = make(case["hkv"], case["sq"])
        t["new_v"] = make(case["hkv"], case["sq"])
    else:
        t["k"] = make(case["hkv"], case["sk"])
        t["v"] = make(case["hkv"], case["sk"])
        if case["kind"] == "train":
            t["do"] = make(case["hq"], case["sq"])
    return t


def prepare(case, seed):
    """What the program holds before the call: the tensors, and for the cache
    cases a filled cache."""
    t = _inputs(case, seed)
    state = {"case": case, **t}
    if case["kind"] in ("step", "verify"):
        cls = PreallocatedKVCache if case["kind"] == "step" else RaggedKVCache
        cache = cls(case["b"], case["hkv"], case["capacity"], case["d"], device="cuda",
                    dtype=DTYPES[case["dtype"]])
        cache.k.copy_(state.pop("k"))
        cache.v.copy_(state.pop("v"))
        state["cache"] = cache
        if case["kind"] == "verify":
            state["lengths"] = _lengths(case, seed)
            cache.set_lengths(state["lengths"])
        else:
            cache.length = case["sk"]
    elif case["kind"] == "train":
        for name in ("q", "k", "v"):
            state[name] = state[name].detach().requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "infer":
        return attention(state["q"], state["k"], state["v"], causal=case["causal"])
    if case["kind"] == "train":
        q, k, v = state["q"], state["k"], state["v"]
        out = attention(q, k, v, causal=case["causal"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["do"])
        return {"out": out, "dq": dq, "dk": dk, "dv": dv}
    cache = state["cache"]
    out = cache.append_and_attend(state["q"], state["new_k"], state["new_v"])
    # Back to the lengths before the step: the tokens are dropped.
    if case["kind"] == "verify":
        cache.set_lengths(state["lengths"])
    else:
        cache.length = case["sk"]
    return {"out": out, "k": cache.k, "v": cache.v}


def _pairs(case):
    """Visible (query, key) pairs of one head, over the whole batch."""
    b, sq, sk = case["b"], case["sq"], case["sk"]
    if case["kind"] == "step":
        return b * (sk + 1)
    if case["kind"] == "verify":
        return sq * sum(x + sq for x in _lengths(case, 0))
    if case["causal"]:
        n = min(sq, sk)
        return b * (n * (n + 1) // 2 + max(0, sq - sk) * sk)
    return b * sq * sk


def work(case):
    """Each input read once, each output written once; the products of the
    visible pairs (two forward, five backward)."""
    b, hq, hkv, sq, sk, d = (case[x] for x in ("b", "hq", "hkv", "sq", "sk", "d"))
    flops = 4.0 * d * hq * _pairs(case)
    rows, keys = b * hq * sq * d * 2, b * hkv * sk * d * 2
    if case["kind"] == "train":
        return {"bytes": 4 * rows + 4 * keys, "flops": 3.5 * flops}
    if case["kind"] in ("step", "verify"):
        seen = 2 * hkv * d * 2 * (_pairs(case) // sq)
        return {"bytes": 2 * rows + seen + 2 * b * hkv * sq * d * 2, "flops": flops}
    return {"bytes": 2 * rows + 2 * keys, "flops": flops}


def tolerance(case):
    """Four times the error against 64-bit sums measured for this path (fp16
    2.5e-4 to 3.1e-4, bf16 1.9e-3 to 2.5e-3 over the listed and drawn cases):
    the rounding of P, dS and the outputs to 16 bits."""
    return {"rel": 1.2e-3 if case["dtype"] == "fp16" else 1e-2}


def _attend(q, k, v, visible, scale):
    """One head in 64 bits, dense: O and P. visible(rows, keys) masks."""
    s = (q @ k.t()) * scale
    if visible is not None:
        s = s.masked_fill(~visible, float("-inf"))
    p = torch.softmax(s, dim=-1)
    return p @ v, p


def exact(case, seed):
    t = _inputs(case, seed)
    b, hq, hkv, sq, d = (case[x] for x in ("b", "hq", "hkv", "sq", "d"))
    scale, group = 1.0 / math.sqrt(d), hq // hkv
    out = torch.zeros((b, hq, sq, d), device="cuda", dtype=torch.float64)
    lens = [case["sk"]] * b
    if case["kind"] in ("step", "verify"):
        if case["kind"] == "verify":
            lens = _lengths(case, seed)
        for i, n in enumerate(lens):
            t["k"][i, :, n:n + sq] = t["new_k"][i]
            t["v"][i, :, n:n + sq] = t["new_v"][i]
        lens = [n + sq for n in lens]
    grads = None
    if case["kind"] == "train":
        grads = [torch.zeros((b, h, n, d), device="cuda", dtype=torch.float64)
                 for h, n in ((hq, sq), (hkv, case["sk"]), (hkv, case["sk"]))]
    for i in range(b):
        keys = torch.arange(lens[i], device="cuda")
        for h in range(hq):
            q = t["q"][i, h].double()
            k, v = (t[x][i, h // group, :lens[i]].double() for x in ("k", "v"))
            for r0 in range(0, sq, 2048):
                rows = torch.arange(r0, min(sq, r0 + 2048), device="cuda")
                seen = keys[None, :] <= rows[:, None] if case["causal"] else None
                o, p = _attend(q[rows], k, v, seen, scale)
                out[i, h, rows] = o
                if grads is not None:
                    do = t["do"][i, h, rows].double()
                    ds = p * (do @ v.t() - (o * do).sum(-1, keepdim=True)) * scale
                    grads[0][i, h, rows] = ds @ k
                    grads[1][i, h // group] += ds.t() @ q[rows]
                    grads[2][i, h // group] += p.t() @ do
    if case["kind"] == "train":
        return {"out": out, "dq": grads[0], "dk": grads[1], "dv": grads[2]}
    if case["kind"] in ("step", "verify"):
        return {"out": out, "k": t["k"].double(), "v": t["v"].double()}
    return out
