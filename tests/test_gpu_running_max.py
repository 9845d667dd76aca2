"""Forwards whose first key tiles hold nothing but large negative scores (a float
mask of -1e9, of -1e30, or the like over left padding): the running maximum that
such a tile leaves behind must not show in the rows' results.

Bound per entry of O, against the eager oracle in float64: its rounding to 16 bits,
u |O| (u = 2^-8 bf16, 2^-11 fp16); P in two 16-bit parts, u^2 max|v| (in fp16 the
parts of a small p are subnormal: 2^-24 sum|v| more, as sum(p) >= 1/2 where the
maximum exceeds no row's by more than one step); 2^-18 max|v| for fp32 sums, exp2
and the merges; and the logits' own error e = D 2^-24 sum|q k| scale log2e (fp32 dot
products, and their sum with a score of at most 64), which moves every p by a
factor of at most 2^e and so O by 2 e max|v|.  LSE (base 2): e, and 2^-23 of its
size.
"""

import math

import pytest
import torch

import tilelang_fa2_4d_mask.ops  # noqa: F401  (registers the ops)
from oracle import eager as E

pytestmark = pytest.mark.gpu

CASES = [
    # D Tq Tk causal mask
    (128, 1, 700, False, False),     # few rows, one wave's tiles low then kept
    (64, 1, 5000, False, True),
    (256, 2, 700, False, False),
    (128, 200, 700, False, False),   # 256-row blocks, key axis split
    (64, 200, 700, False, True),
    (128, 600, 600, True, False),
    (256, 130, 500, False, False),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("low", [-1e9, -1e30, -70000.0])
@pytest.mark.parametrize("shift", [0.0, -40.0])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"D{c[0]}T{c[1]}-{c[2]}{'c' if c[3] else ''}{'m' if c[4] else ''}")
def test_low_tiles_first(cuda, case, dtype, low, shift):
    D, Tq, Tk, causal, masked = case
    print("case", case, dtype, low, shift, flush=True)
    scale = 1.0 if D == 64 else 0.5
    g = torch.Generator().manual_seed(D + Tq)
    q, k, v = (torch.randn((2, T, H, D), generator=g).to(dtype) for T, H in ((Tq, 4), (Tk, 2), (Tk, 2)))
    start = torch.tensor([Tk // 2, Tk // 5]).view(2, 1, 1, 1)
    if causal:       # every row keeps its own key: the low ones lie before row / 2
        start = torch.arange(Tq).view(1, 1, Tq, 1) // 2
    s = torch.where(torch.arange(Tk) >= start, shift, low).float().expand(2, 1, Tq, Tk).contiguous()
    m = None
    if masked:
        m = torch.rand((2, 1, Tq, Tk), generator=g) < 0.9
        m[..., Tk - 1] = True
    dv = [None if x is None else x.to(cuda) for x in (q, k, v, m, s)]
    with torch.no_grad():
        O, L, _, _ = torch.ops.tilelang_fa2_4d_mask.fwd(*dv, scale, causal, False, False)
    torch.cuda.synchronize()
    bhsd = [x.transpose(1, 2).double() for x in (q, k, v)]
    ref = E.eager_ref(*bhsd, m, s, scale=scale, is_causal=causal, compute_dtype=torch.float64).transpose(1, 2)
    logits = (bhsd[0] @ bhsd[1].repeat_interleave(2, dim=1).transpose(2, 3) + s.double()) * scale
    keep = torch.ones((Tq, Tk), dtype=torch.bool).tril() if causal else torch.ones((Tq, Tk), dtype=torch.bool)
    logits.masked_fill_(~(keep if m is None else keep & m), -math.inf)
    lse = torch.logsumexp(logits, dim=-1) * math.log2(math.e)
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    vmax = v.abs().max().item()
    dots = bhsd[0].abs() @ bhsd[1].abs().repeat_interleave(2, dim=1).transpose(2, 3)
    e = D * (dots.max().item() + 64) * 2.0 ** -24 * scale * math.log2(math.e)
    sub = 2.0 ** -24 * (1 + v.float().abs().sum(1).max().item()) if dtype == torch.float16 else 0.0
    bound = u * ref.abs() + (u * u + 2.0 ** -18 + 2 * e) * vmax + sub
    err = (O.double().cpu() - ref).abs()
    assert torch.isfinite(O).all()
    assert bool((err <= bound).all()), (err - bound).max().item()
    assert (L.double().cpu() - lse).abs().max().item() <= e + 2.0 ** -23 * lse.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("low", [-1e9, -1e30])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"D{c[0]}T{c[1]}-{c[2]}{'c' if c[3] else ''}{'m' if c[4] else ''}")
def test_nothing_but_low_keys(cuda, case, dtype, low):
    """Rows of which every key carries the same large negative score: fp32 sums
    take the small q k into it, all weights are equal, O is the mean of V."""
    D, Tq, Tk, causal, masked = case
    print("case", case, dtype, low, flush=True)
    g = torch.Generator().manual_seed(D + Tq)
    q, k, v = (torch.randn((2, T, H, D), generator=g).to(dtype) for T, H in ((Tq, 4), (Tk, 2), (Tk, 2)))
    q, k = q * 0.125, k * 0.125       # sum |q k| < 16, a fourth of fp32's step at 1e9
    s = torch.full((1, 1, Tq, Tk), low)
    keep = torch.ones((2, 1, Tq, Tk), dtype=torch.bool)
    if masked:
        keep = torch.rand((2, 1, Tq, Tk), generator=g) < 0.9
        keep[..., Tk - 1] = True
    dv = [x.to(cuda) for x in (q, k, v)] + [keep.to(cuda) if masked else None, s.to(cuda)]
    with torch.no_grad():
        O = torch.ops.tilelang_fa2_4d_mask.fwd(*dv, 0.5, causal, False, False)[0]
    w = keep.tril() if causal else keep
    ref = (w.double() / w.sum(-1, keepdim=True)) @ v.transpose(1, 2).double().repeat_interleave(2, dim=1)
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    sub = 2.0 ** -24 * (1 + v.float().abs().sum(1).max().item()) if dtype == torch.float16 else 0.0
    err = (O.double().cpu().transpose(1, 2) - ref).abs()
    assert bool((err <= u * ref.abs() + (u * u + 2.0 ** -18) * v.abs().max().item() + sub).all()), err.max().item()
