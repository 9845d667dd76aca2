"""Head dims that the kernels take in place (multiples of 16 below the kernels'
64 / 128 / 256): the columns past the operands' own are the next head's data in
a token-major layout.  With NaN in every other head, each of a head's results is
bit for bit what it is beside finite heads, and what the zero-padded problem at
the kernels' head dim gives (the kernels then do the same arithmetic).  Atomic dQ
adds the same products in no fixed order: it may differ from the deterministic one
by the rounding of its fp32 sums, Tk 2^-24 sum|dS K| scale, and a unit in the last
place of each of the two results (2^-7 bf16, 2^-10 fp16)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # D Tq Tk causal mask
    (16, 40, 70, False, False),      # few-rows forward
    (48, 300, 2049, False, False),   # key split
    (80, 200, 200, True, False),
    (96, 257, 300, False, True),
    (112, 130, 1500, False, True),   # masked key split
    (144, 150, 170, True, False),
    (208, 20, 90, False, True),
]


def _run(q, k, v, do, mask, causal, atomic, ds_limit):
    import tilelang_fa2_4d_mask as api
    import tilelang_fa2_4d_mask.fa2 as F

    F.DS_LIMIT_BYTES = ds_limit
    try:
        q, k, v = (x.detach().requires_grad_(True) for x in (q, k, v))
        out = api.tilelang_flash_attention(q, k, v, mask=mask, is_causal=causal, layout="bshd", scale=0.1,
                                           use_atomic_backward=atomic)
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), do))
    finally:
        F.DS_LIMIT_BYTES = 0


def _sum_bound(q, k, v, do, mask, causal, scale):
    """Tk 2^-24 sum_j |dS_ij K_jd| scale of each dQ entry, in 64 bits."""
    q, k, v, do = (x.cpu().double().transpose(1, 2) for x in (q, k, v, do))
    Tq, Tk = q.shape[2], k.shape[2]
    keep = torch.ones((Tq, Tk), dtype=torch.bool).tril() if causal else torch.ones((Tq, Tk), dtype=torch.bool)
    p = ((q @ k.transpose(2, 3)) * scale).masked_fill(~(keep if mask is None else keep & mask.cpu()), -math.inf).softmax(-1)
    dp = do @ v.transpose(2, 3)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    return (ds.abs() @ k.abs() * (scale * Tk * 2.0 ** -24)).transpose(1, 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"D{c[0]}T{c[1]}-{c[2]}")
def test_columns_in_place(cuda, case, dtype):
    from tilelang_fa2_4d_mask.fa2 import kernel_head_dim

    D, Tq, Tk, causal, masked = case
    g = torch.Generator().manual_seed(D)
    q, k, v, do = (torch.randn((2, T, 3, D), generator=g).to(dtype).to(cuda) for T in (Tq, Tk, Tk, Tq))
    mask = (torch.rand((2, 1, Tq, Tk), generator=g) < 0.7).to(cuda) if masked else None
    if masked:
        mask[..., 0] = True
    pad = [torch.nn.functional.pad(x, (0, kernel_head_dim(D) - D)) for x in (q, k, v, do)]
    dirty = []
    for x in (q, k, v, do):
        x = x.clone()
        x[:, :, 0::2] = float("nan")
        dirty.append(x)
    dq_det, dq_bound = None, None
    for atomic, limit in ((False, 0), (True, 0), (False, -1)):
        print("case", case, dtype, atomic, limit, flush=True)
        a = _run(q, k, v, do, mask, causal, atomic, limit)
        b = _run(*dirty, mask, causal, atomic, limit)
        c = _run(*pad, mask, causal, atomic, limit)
        for i, (x, y, z) in enumerate(zip(a, b, c)):
            assert torch.isfinite(x).all() and torch.isfinite(y[:, :, 1]).all(), i
            if atomic and i == 1:
                for got, ref in ((x, dq_det), (y[:, :, 1:2], dq_det[:, :, 1:2]), (z[..., :D], dq_det)):
                    assert ((got.cpu().double() - ref).abs() <= (dq_bound if got.shape[2] == 3 else dq_bound[:, :, 1:2])).all()
                continue
            assert torch.equal(x[:, :, 1], y[:, :, 1]), i
            assert torch.equal(x, z[..., :D]), i
        if not atomic and limit == 0:
            dq_det = a[1].cpu().double()
            dq_bound = _sum_bound(q, k, v, do, mask, causal, 0.1) + 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * dq_det.abs()
