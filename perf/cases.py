"""Attention workloads of this package: what a user's program calls, at the
sizes it calls it with, for timing and for checking results.

A case is a dict of plain values:

  kind    "infer" (forward without gradients) or "train" (forward + backward)
  B, Tq, Tk, Hq, Hk, D, dtype ("bf16" / "fp16"), layout ("bhsd" / "bshd")
  causal  is_causal of the call
  mask    "none"      no mask
          "padding"   a left-padded batch: bool [B, 1, Tq, Tk], sequence b
                      starts at its own key (the adapter's attention_mask)
          "chunk"     a prompt chunk behind a cache: bool [1, 1, Tq, Tk], row i
                      keeps keys up to Tk - Tq + i
          "packed"    packed documents of 128 .. 1024 tokens: bool [B, 1, T, T],
                      block-diagonal causal
          "sparse"    per-head bool [B, Hq, T, T], a tenth of the keys dropped
  score   "none"
          "alibi"     fp32 [B, Hq, T, T]: -slope_h |i - j| plus noise
          "additive"  the model code's float mask in the inputs' type,
                      [B, 1, T, T]: 0 or the type's lowest value, causal over a
                      right-padded batch (the adapter's attention_mask)
  atomic  use_atomic_backward ("train")
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fa2-with-4d-mask_amd"))

from tilelang_fa2_4d_mask import tilelang_attention_forward, tilelang_flash_attention  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
DOC_LO, DOC_HI = 128, 1024     # document lengths of a packed sequence
SPARSE_DROP = 0.1


def _case(kind, B, Tq, Tk, Hq, Hk, D, dtype="bf16", layout="bhsd", causal=False, mask="none", score="none",
          atomic=True, name=None):
    c = dict(kind=kind, B=B, Tq=Tq, Tk=Tk, Hq=Hq, Hk=Hk, D=D, dtype=dtype, layout=layout, causal=causal, mask=mask,
             score=score, atomic=atomic)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # one token generated for one long conversation: the smallest query,
        # the cache of 16384 tokens is all there is to read
        _case("infer", 1, 1, 16384, 32, 8, 128, name="decode_one_16k"),
        # one token for each sequence of a left-padded batch, through the
        # model adapter with its bool mask
        _case("infer", 16, 1, 3001, 32, 8, 128, mask="padding", name="decode_batch_padded"),
        # the next chunk of a long prompt, behind what the cache already holds
        _case("infer", 1, 512, 8704, 32, 8, 128, mask="chunk", name="prefill_chunk_cached"),
        # the prompts of a right-padded batch, through the model adapter with
        # the additive float mask of eager-attention model code
        _case("infer", 4, 1000, 1000, 32, 8, 128, dtype="fp16", score="additive", name="prefill_padded_float"),
        # a unit-test sized training step: launches and host time
        _case("train", 1, 256, 256, 4, 2, 64, causal=True, name="train_small"),
        # odd sizes, a head dim between the kernels', fp16, token-major layout
        _case("train", 2, 1999, 1999, 16, 16, 96, dtype="fp16", layout="bshd", causal=True, name="train_ragged_d96"),
        # the ordinary causal language-model training step
        _case("train", 2, 4096, 4096, 32, 8, 128, causal=True, name="train_causal"),
        # the headline size, both directions, deterministic backward
        _case("train", 1, 8192, 8192, 32, 8, 128, atomic=False, name="train_full_8k"),
        # packed documents behind a block-diagonal mask
        _case("train", 2, 4096, 4096, 32, 8, 128, mask="packed", name="train_packed_docs"),
        # a position bias per head and a sparse mask per head
        _case("train", 1, 4096, 4096, 16, 16, 128, mask="sparse", score="alibi", name="train_score_mask"),
        # one key/value head for 32 query heads over a long context, head dim 64
        _case("train", 1, 2048, 16384, 32, 1, 64, layout="bshd", name="train_mqa_long_kv"),
        # the largest head dim
        _case("train", 1, 4096, 4096, 16, 4, 256, causal=True, name="train_d256"),
    ]


HEADS = [(32, 8), (16, 4), (32, 32), (16, 16), (24, 8), (8, 1), (32, 1), (4, 2)]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm: a round one or
    any."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and n >= 128:
        n = max(lo, n // 64 * 64)
    return n


def _draw_one(rng):
    family = rng.choice(["decode", "decode", "chunk", "float", "train", "train", "train", "packed", "score", "long_kv"])
    Hq, Hk = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    layout = rng.choice(["bhsd", "bhsd", "bshd"])
    D = rng.choice([64, 128, 128])
    if family == "decode":
        return _case("infer", _log(rng, 1, 32), 1, _log(rng, 256, 32768), Hq, Hk, D, dtype,
                     mask=rng.choice(["none", "padding"]))
    if family == "chunk":
        Tq = _log(rng, 16, 2048)
        return _case("infer", 1, Tq, Tq + _log(rng, 256, 16384), Hq, Hk, D, dtype, layout, mask="chunk")
    if family == "float":
        T = _log(rng, 64, 2048)
        return _case("infer", _log(rng, 1, 8), T, T, Hq, Hk, D, dtype, score="additive")
    if family == "packed":
        T = _log(rng, 1024, 8192)
        return _case("train", _log(rng, 1, 4), T, T, Hq, Hk, D, dtype, layout, mask="packed",
                     atomic=rng.random() < 0.5)
    if family == "score":
        T = _log(rng, 256, 4096)
        return _case("train", 1, T, T, 16, rng.choice([4, 16]), D, dtype, layout, score="alibi",
                     mask=rng.choice(["none", "sparse"]), causal=rng.random() < 0.3, atomic=rng.random() < 0.5)
    if family == "long_kv":
        return _case("train", 1, _log(rng, 128, 2048), _log(rng, 2048, 16384), Hq, Hk, D, dtype, layout,
                     atomic=rng.random() < 0.5)
    T = _log(rng, 128, 8192)
    return _case("train", _log(rng, 1, 4), T, T, Hq, Hk, rng.choice([64, 80, 96, 128, 128, 256]), dtype, layout,
                 causal=rng.random() < 0.7, atomic=rng.random() < 0.5)


def _cost(case):
    """Dense operations of a case, with the slower forms weighted: what bounds
    a drawn case."""
    f = (14.0 if case["kind"] == "train" else 4.0) * case["B"] * case["Hq"] * case["Tq"] * case["Tk"] * case["D"]
    if case["D"] > 128:
        f *= 4.0
    if case["score"] != "none":
        f *= 4.0
    return f


def draw(rng: random.Random):
    top = _cost(_case("train", 1, 8192, 8192, 32, 8, 128))
    while True:
        c = _draw_one(rng)
        cache = 4 * c["B"] * c["Tk"] * c["Hk"] * c["D"]
        if _cost(c) <= 0.8 * top and cache <= 2 << 30:
            return c


# ---- inputs ---------------------------------------------------------------------


def _pads(case):
    """First kept key (left padding) or kept length (right padding) of each
    sequence: up to half of it is padding."""
    T, B = case["Tk"], case["B"]
    return [(T // 2) * ((7 * b) % 8) // 8 for b in range(B)]


def _packed_segments(B, T, seed, device):
    rng = random.Random(seed)
    seg = torch.empty((B, T), dtype=torch.int32)
    for b in range(B):
        pos = sid = 0
        while pos < T:
            n = rng.randint(DOC_LO, DOC_HI)
            seg[b, pos:pos + n] = sid
            pos, sid = pos + n, sid + 1
    return seg.to(device)


def _side(case, seed, gen, dev):
    """(mask, score, attention_mask) of a case."""
    B, Hq, Tq, Tk = case["B"], case["Hq"], case["Tq"], case["Tk"]
    i = torch.arange(Tq, device=dev)[:, None]
    j = torch.arange(Tk, device=dev)[None, :]
    mask = score = additive = None
    if case["mask"] == "padding":
        start = torch.tensor(_pads(case), device=dev).view(B, 1, 1, 1)
        additive = (j >= start).expand(B, 1, Tq, Tk).contiguous()
    elif case["mask"] == "chunk":
        mask = (j <= i + (Tk - Tq)).view(1, 1, Tq, Tk)
    elif case["mask"] == "packed":
        seg = _packed_segments(B, Tk, seed, dev)
        mask = ((seg[:, :, None] == seg[:, None, :]) & (j <= i)).unsqueeze(1).contiguous()
    elif case["mask"] == "sparse":
        mask = torch.rand((B, Hq, Tq, Tk), generator=gen, device=dev) >= SPARSE_DROP
        n = torch.arange(min(Tq, Tk), device=dev)
        mask[:, :, n, n] = True
    if case["score"] == "alibi":
        slope = torch.tensor([2.0 ** (-8.0 * (h + 1) / Hq) for h in range(Hq)], device=dev).view(1, Hq, 1, 1)
        score = torch.randn((B, Hq, Tq, Tk), generator=gen, device=dev).mul_(0.1).sub_(slope * (i - j).abs())
    elif case["score"] == "additive":
        dt = DTYPES[case["dtype"]]
        end = torch.tensor([Tk - p for p in _pads(case)], device=dev).view(B, 1, 1, 1)
        keep = (j <= i) & (j < end)
        additive = torch.zeros(keep.shape, dtype=dt, device=dev).masked_fill_(~keep, torch.finfo(dt).min)
    return mask, score, additive


class _Module:
    """What the model adapter reads of an attention module."""

    is_causal = True


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, Tq, Tk, Hq, Hk, D = (case[n] for n in ("B", "Tq", "Tk", "Hq", "Hk", "D"))

    def rnd(T, H):
        x = torch.randn((B, T, H, D), generator=gen, device=dev).to(dt)
        return x if case["layout"] == "bshd" else x.transpose(1, 2)

    q, k, v = rnd(Tq, Hq), rnd(Tk, Hk), rnd(Tk, Hk)
    if case["layout"] == "bhsd" and Tq < Tk and case["kind"] == "infer":
        k, v = k.contiguous(), v.contiguous()    # a cache is kept head by head
    state = {"case": case, "q": q, "k": k, "v": v}
    if case["kind"] == "train":
        state["do"] = rnd(Tq, Hq)
        for n in "qkv":
            state[n] = state[n].detach().requires_grad_(True)
    state["mask"], state["score"], state["attention_mask"] = _side(case, seed, gen, dev)
    return state


# ---- one pass ---------------------------------------------------------------------


def _attention(state):
    case = state["case"]
    if state["attention_mask"] is not None:
        return tilelang_attention_forward(_Module, state["q"], state["k"], state["v"], state["attention_mask"],
                                          case["D"] ** -0.5, layout=case["layout"])[0]
    return tilelang_flash_attention(state["q"], state["k"], state["v"], mask=state["mask"], score=state["score"],
                                    is_causal=case["causal"], layout=case["layout"],
                                    use_atomic_backward=case["atomic"])


def run(state):
    if state["case"]["kind"] == "infer":
        with torch.no_grad():
            return {"out": _attention(state)}
    out = _attention(state)
    dq, dk, dv = torch.autograd.grad(out, (state["q"], state["k"], state["v"]), state["do"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


# ---- what a pass cannot do without, and its result in 64 bits ------------------------


def _kept_pairs(case):
    """(row, key) pairs kept, over the batch, for one head (expected where the
    seed decides)."""
    B, Tq, Tk = case["B"], case["Tq"], case["Tk"]
    pads = _pads(case)
    lower = sum(min(i + 1, Tk) for i in range(Tq))
    if case["mask"] == "padding":
        return float(Tq * sum(Tk - p for p in pads))
    if case["mask"] == "chunk":
        return float(sum(Tk - Tq + i + 1 for i in range(Tq)))
    if case["mask"] == "packed":
        mean, square = (DOC_LO + DOC_HI) / 2, (DOC_HI ** 3 - DOC_LO ** 3) / (3.0 * (DOC_HI - DOC_LO))
        return B * Tq * min(Tk / 2, square / (2 * mean))
    if case["score"] == "additive":
        return float(sum(sum(min(i + 1, Tk - p) for i in range(Tq)) for p in pads))
    pairs = B * float(lower if case["causal"] else Tq * Tk)
    return pairs * (1 - SPARSE_DROP) if case["mask"] == "sparse" else pairs


def work(case):
    B, Tq, Tk, Hq, Hk, D = (case[n] for n in ("B", "Tq", "Tk", "Hq", "Hk", "D"))
    train = case["kind"] == "train"
    operands = 2 * D * B * (2 * Tq * Hq + 2 * Tk * Hk)            # Q, K, V, O
    if train:
        operands += 2 * D * B * (2 * Tq * Hq + 2 * Tk * Hk)      # dO, dQ, dK, dV
    side = {"none": 0, "padding": B, "chunk": 1, "packed": B, "sparse": B * Hq}[case["mask"]] * Tq * Tk
    side += {"none": 0, "alibi": 4 * B * Hq, "additive": 2 * B}[case["score"]] * Tq * Tk
    return {"bytes": float(operands + side), "flops": (14.0 if train else 4.0) * Hq * D * _kept_pairs(case)}


def tolerance(case):
    """Rounding of the 16-bit results and, without a mask or a score, of P and
    dS before their products: four times the largest error against 64 bits
    over the listed cases (bf16 2.6e-3, fp16 3.2e-4)."""
    return {"rel": 1.05e-2 if case["dtype"] == "bf16" else 1.3e-3}


def exact(case, seed):
    s = prepare(case, seed)
    dev, f64 = s["q"].device, torch.float64
    B, Tq, Tk, Hq, Hk, D = (case[n] for n in ("B", "Tq", "Tk", "Hq", "Hk", "D"))
    group, scale, train = Hq // Hk, D ** -0.5, case["kind"] == "train"

    def heads(x):   # [B, H, T, D] view
        x = x.detach()
        return x if case["layout"] == "bhsd" else x.transpose(1, 2)

    q, k, v = heads(s["q"]), heads(s["k"]), heads(s["v"])
    out = torch.empty((B, Hq, Tq, D), dtype=f64, device=dev)
    if train:
        do = heads(s["do"])
        dq = torch.empty((B, Hq, Tq, D), dtype=f64, device=dev)
        dk = torch.zeros((B, Hk, Tk, D), dtype=f64, device=dev)
        dv = torch.zeros((B, Hk, Tk, D), dtype=f64, device=dev)

    def pick(x, b, h):   # one [Tq, Tk] plane of a broadcast side input
        return x[min(b, x.shape[0] - 1), min(h, x.shape[1] - 1)]

    for b in range(B):
        for h in range(Hq):
            n = h // group
            qh, kh, vh = q[b, h].to(f64), k[b, n].to(f64), v[b, n].to(f64)
            x = qh @ kh.T
            if s["score"] is not None:
                x += pick(s["score"], b, h)
            x *= scale
            extra = s["attention_mask"]
            if extra is not None and extra.dtype == torch.bool:
                x.masked_fill_(~pick(extra, b, h), -math.inf)
            elif extra is not None:
                x += pick(extra, b, h)
            if s["mask"] is not None:
                x.masked_fill_(~pick(s["mask"], b, h), -math.inf)
            if case["causal"]:
                x.masked_fill_(torch.ones((Tq, Tk), dtype=torch.bool, device=dev).triu_(1), -math.inf)
            p = torch.softmax(x, dim=1)
            del x
            out[b, h] = p @ vh
            if train:
                doh = do[b, h].to(f64)
                dv[b, n] += p.T @ doh
                ds = doh @ vh.T
                ds -= (doh * out[b, h]).sum(1, keepdim=True)
                ds *= p
                ds *= scale
                dq[b, h] = ds @ kh
                dk[b, n] += ds.T @ qh

    def back(x):
        return x if case["layout"] == "bhsd" else x.transpose(1, 2)

    if not train:
        return {"out": back(out)}
    return {"out": back(out), "dq": back(dq), "dk": back(dk), "dv": back(dv)}
