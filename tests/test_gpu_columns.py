"""Head dims that the kernels take in place (multiples of 16 below the kernels'
64 / 128 / 256): the columns past the operands' own are the next head's data in
a token-major layout.  With NaN in every other head, each of a head's results is
bit for bit what it is beside finite heads, and what the zero-padded problem at
the kernels' head dim gives (the kernels then do the same arithmetic)."""

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
    # (atomic dQ over key ranges adds in no fixed order: its dQ is left out)
    for atomic, limit in ((False, 0), (True, 0), (False, -1)):
        print("case", case, dtype, atomic, limit, flush=True)
        a = _run(q, k, v, do, mask, causal, atomic, limit)
        b = _run(*dirty, mask, causal, atomic, limit)
        c = _run(*pad, mask, causal, atomic, limit)
        for i, (x, y, z) in enumerate(zip(a, b, c)):
            if atomic and i == 1:
                continue
            assert torch.isfinite(x).all()
            assert torch.equal(x[:, :, 1], y[:, :, 1]), i
            assert torch.equal(x, z[..., :D]), i
