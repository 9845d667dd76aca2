"""Forward of few query rows (fa_rows.hip) and of 256-row blocks with the key
axis split (fa_fwd.hip, SPLIT), against the eager oracle in float64.

Bound per entry of O: its own rounding to 16 bits, u |O| (half a unit in the
last place: u = 2^-8 bf16, of 8 significant bits, 2^-11 fp16, of 11); without a
mask or a score the rounding of P before P V, which moves O by at most
u sum(p |v|) / sum(p) <= u max|v|; with either P enters in two parts
(u^2 max|v|); 2^-18 max|v| for fp32 sums, exp2 and the merges' factors.  In fp16
the parts of a small p are subnormal (steps of 2^-24, so off by 2^-25 each, and
sum(p) >= 1/2 as the running maximum exceeds no row's by more than one step; for
large negative scores see test_gpu_running_max.py):
2^-24 sum|v| more.  LSE (base 2): fp32 dot products of D
16-bit values, |dlogit| <= D 2^-24 sum|q k| scale log2e < 2e-4 here.
"""

import ctypes
import math

import pytest
import torch

import tilelang_fa2_4d_mask.ops  # noqa: F401  (registers the ops)
from oracle import eager as E

pytestmark = pytest.mark.gpu


def _plan(B, Hq, Hk, D, Tq, Tk, causal, mask, score):
    from tilelang_fa2_4d_mask import _ext

    lib = _ext.load_library()
    p = _ext.FaFwdParams()
    p.batch, p.seqlen_q, p.seqlen_k, p.heads_q, p.heads_k, p.head_dim = B, Tq, Tk, Hq, Hk, D
    p.is_causal, p.scale = int(causal), 0.1
    p.mask, p.score = (256 if mask else None), (256 if score else None)
    plan = _ext.FaFwdPlan()
    _ext.check(lib.fa_fwd_plan(ctypes.byref(p), ctypes.byref(plan)), "fa_fwd_plan", lib)
    return plan


def _inputs(seed, B, Hq, Hk, D, Tq, Tk, dtype, mask, score):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((B, T, H, D), generator=g).to(dtype) for T, H in ((Tq, Hq), (Tk, Hk), (Tk, Hk)))
    m = s = None
    if mask == "bernoulli":      # odd row stride (a view): byte loads; one dead row
        m = (torch.rand((B, Hq, Tq, Tk + 1), generator=g) < 0.6)[..., :Tk]
        m[0, 0, 0] = False
    elif mask == "left":         # left padding, per batch entry, broadcast over heads
        start = torch.tensor([(Tk * (b + 1)) // (B + 1) for b in range(B)]).view(B, 1, 1, 1)
        m = (torch.arange(Tk) >= start).expand(B, 1, Tq, Tk).contiguous()
    elif mask == "chunk":
        m = (torch.arange(Tk) <= torch.arange(Tq)[:, None] + Tk - Tq).view(1, 1, Tq, Tk)
    if score == "normal":
        s = torch.randn((B, Hq, Tq, Tk), generator=g)
    elif score == "padding":     # -inf on the left, one row with nothing else
        s = torch.where(torch.arange(Tk) >= Tk // 2, 0.0, -math.inf).expand(B, 1, Tq, Tk).clone()
        s[0, 0, Tq - 1] = -math.inf
    return q, k, v, m, s


def _check(seed, B, Hq, Hk, D, Tq, Tk, dtype, causal, mask, score, scale, residual=False):
    dev = torch.device("cuda:0")
    q, k, v, m, s = _inputs(seed, B, Hq, Hk, D, Tq, Tk, dtype, mask, score)
    dv = [None if x is None else x.to(dev) for x in (q, k, v, m, s)]
    with torch.no_grad():
        O, L, ws, lo = torch.ops.tilelang_fa2_4d_mask.fwd(*dv, scale, causal, False, residual)
    torch.cuda.synchronize()
    _compare(O, L, lo if residual else None, q, k, v, m, s, scale, causal, dtype)


def _compare(O, L, lo, q, k, v, m, s, scale, causal, dtype):
    bhsd = [x.transpose(1, 2).double() for x in (q, k, v)]
    ref = E.eager_ref(*bhsd, m, s, scale=scale, is_causal=causal, compute_dtype=torch.float64).transpose(1, 2)
    O = O.double().cpu()
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    two = m is not None or s is not None
    vmax = v.abs().max().item()
    assert torch.equal(torch.isnan(O), torch.isnan(ref))
    fin = ~torch.isnan(ref)
    sub = 2.0 ** -24 * (1 + v.float().abs().sum(1).max().item()) if dtype == torch.float16 else 0.0
    bound = u * ref.abs() + ((u * u if two else u) + 2.0 ** -18) * vmax + sub
    assert bool(((O - ref).abs()[fin] <= bound[fin]).all()), (O - ref).abs()[fin].max().item()
    if lo is not None and two:
        both = (O + lo.double().cpu() - ref).abs()
        # O + residual: the rounding of O itself drops out
        assert bool((both[fin] <= (u * u * ref.abs() + (u * u + 2.0 ** -18) * vmax + sub)[fin]).all())
    lse = E.lse2_reference(*bhsd[:2], m, s, scale=scale, is_causal=causal)
    L = L.double().cpu()
    dead = ~torch.isfinite(lse)
    assert torch.equal(torch.isposinf(L), dead)
    assert (L - lse)[~dead].abs().max().item() < 2e-4


ROWS = [
    # B Hq Hk D Tq Tk dtype causal mask score scale
    (1, 4, 1, 128, 1, 1, torch.bfloat16, False, None, None, 0.09),
    (3, 8, 2, 128, 1, 31, torch.bfloat16, False, None, None, 0.09),
    (2, 8, 8, 64, 1, 4097, torch.float16, False, None, None, 0.125),      # ranges, last tile of one key
    (1, 32, 1, 128, 2, 2048, torch.bfloat16, False, None, None, -0.09),   # two row blocks
    (1, 6, 2, 64, 11, 33, torch.float16, True, None, None, 0.125),        # 33 packed rows, causal
    (2, 4, 2, 128, 64, 64, torch.bfloat16, True, "bernoulli", "normal", 0.09),
    (4, 8, 2, 128, 1, 3001, torch.bfloat16, False, "left", None, 0.09),
    (2, 4, 2, 64, 3, 4133, torch.bfloat16, False, "bernoulli", None, 0.125),   # byte loads
    (1, 4, 2, 128, 128, 1000, torch.float16, False, "chunk", None, 0.09),
    (2, 4, 4, 128, 1, 2048, torch.bfloat16, False, None, "padding", 0.09),
    (1, 4, 2, 128, 5, 700, torch.bfloat16, False, "bernoulli", "normal", 0.0),
    (1, 4, 2, 128, 5, 700, torch.bfloat16, False, None, "normal", -0.09),
    (1, 4, 1, 256, 1, 2500, torch.bfloat16, False, None, None, 0.06),
    (2, 4, 2, 256, 17, 300, torch.float16, False, "bernoulli", "normal", 0.06),
]


@pytest.mark.parametrize("case", ROWS, ids=lambda c: f"B{c[0]}H{c[1]}-{c[2]}D{c[3]}T{c[4]}-{c[5]}{c[8] or ''}{c[9] or ''}")
@pytest.mark.parametrize("residual", [False, True])
def test_few_rows(cuda, case, residual):
    B, Hq, Hk, D, Tq, Tk, dtype, causal, mask, score, scale = case
    plan = _plan(B, Hq, Hk, D, Tq, Tk, causal, mask, score)
    assert plan.needs_mask_ws == 0
    print("case", case, "ranges", plan.key_split, flush=True)
    _check(1, *case, residual=residual)


# All keys in one range, as large batches run: no workspace, so no split.  Then a wave
# has over 32 tiles, what it looks at together: dead ones between live ones, a window
# wholly dead before one that is live, and the next tile's loads beside the last
# tile's work throughout.
ONE_RANGE = [
    # D mask score
    (128, None, None),
    (64, "bernoulli", None),
    (128, "late", None),
    (64, "late", "normal"),
    (128, "gaps", None),
    (256, "gaps", "normal"),
    (128, None, "padding"),
    (256, None, None),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", ONE_RANGE, ids=lambda c: f"D{c[0]}{c[1] or ''}{c[2] or ''}")
def test_many_tiles_per_wave(cuda, case, dtype):
    from tilelang_fa2_4d_mask import _ext

    D, mask, score = case
    B, Hq, Hk, Tq, Tk, scale = 2, 4, 2, 3, 4300, 0.1
    tiles = -(-Tk // 32)
    assert tiles > 4 * 32            # four waves take every fourth tile each
    print("case", case, dtype, flush=True)
    q, k, v, m, s = _inputs(6, B, Hq, Hk, D, Tq, Tk, dtype, mask, score)
    if mask == "late":               # all of each wave's first window dead, for one batch entry
        m = torch.ones((B, 1, Tq, Tk), dtype=torch.bool)
        m[0, ..., : 4 * 32 * 32] = False
    elif mask == "gaps":             # two of three tiles dead, and a window with one live tile
        t = torch.arange(Tk) // 32
        m = ((t % 3 == 1) & ((t < 64) | (t >= 128) | (t == 100))).expand(B, 1, Tq, Tk).contiguous()
    dv = [None if x is None else x.to(cuda) for x in (q, k, v, m, s)]
    O = torch.full((B, Tq, Hq, D), float("nan"), dtype=dtype, device=cuda)
    L = torch.empty((B, Hq, Tq), device=cuda)
    p = _ext.FaFwdParams()
    p.q, p.k, p.v, p.mask, p.score = (_ext.ptr(x) for x in dv)
    p.o, p.lse = O.data_ptr(), L.data_ptr()
    for n, x in (("q", dv[0]), ("k", dv[1]), ("v", dv[2]), ("o", O)):
        for a, st in zip("bth", x.stride()):
            setattr(p, f"{n}_stride_{a}", st)
    for n, x in (("mask", dv[3]), ("score", dv[4])):
        if x is not None:
            st = [0 if x.shape[i] == 1 else x.stride(i) for i in range(3)]
            for a, v_ in zip("bhq", st):
                setattr(p, f"{n}_stride_{a}", v_)
    p.batch, p.seqlen_q, p.seqlen_k, p.heads_q, p.heads_k, p.head_dim = B, Tq, Tk, Hq, Hk, D
    p.scale, p.dtype = scale, _ext.dtype_code(dtype)
    p.stream = torch.cuda.current_stream().cuda_stream
    lib = _ext.load_library()
    plan = _ext.FaFwdPlan()
    _ext.check(lib.fa_fwd_plan(ctypes.byref(p), ctypes.byref(plan)), "fa_fwd_plan", lib)
    assert plan.needs_mask_ws == 0 and plan.key_split > 1
    _ext.check(lib.fa_fwd(ctypes.byref(p)), "fa_fwd", lib)
    torch.cuda.synchronize()
    _compare(O, L, None, q, k, v, m, s, scale, False, dtype)


SPLIT = [
    (1, 4, 2, 128, 300, 2049, torch.bfloat16, False, None, None, 0.09),     # last range: a tile of one key
    (2, 4, 2, 64, 257, 1111, torch.float16, False, None, None, 0.125),
    (1, 2, 1, 128, 1100, 1100, torch.bfloat16, True, None, None, 0.09),     # causal: empty ranges of short blocks
    (1, 2, 2, 64, 1024, 1024, torch.bfloat16, True, None, "normal", 0.125),
    (1, 4, 2, 128, 200, 2000, torch.bfloat16, False, "bernoulli", None, 0.09),
    (1, 4, 2, 128, 200, 2000, torch.float16, False, "chunk", "normal", -0.09),
    (1, 4, 1, 64, 300, 1500, torch.bfloat16, False, "left", None, 0.125),   # dead leading tiles: short lists
    (1, 2, 1, 128, 700, 700, torch.bfloat16, True, "bernoulli", None, 0.09),
]


@pytest.mark.parametrize("case", SPLIT, ids=lambda c: f"B{c[0]}H{c[1]}-{c[2]}D{c[3]}T{c[4]}-{c[5]}{c[8] or ''}{c[9] or ''}")
def test_key_split(cuda, case):
    B, Hq, Hk, D, Tq, Tk, dtype, causal, mask, score, scale = case
    plan = _plan(B, Hq, Hk, D, Tq, Tk, causal, mask, score)
    assert plan.key_split > 1 and plan.needs_mask_ws == 1
    print("case", case, "ranges", plan.key_split, flush=True)
    _check(2, *case, residual=True)


# Causal at head dim 64: blocks of 128 rows (four waves) without a mask or score
CAUSAL64 = [
    (1, 4, 2, 64, 129, 129, torch.bfloat16, True, None, None, 0.125),     # second block of one row
    (2, 12, 4, 64, 1999, 1999, torch.float16, True, None, None, 0.125),
    (2, 64, 64, 64, 300, 70, torch.bfloat16, True, None, None, 0.125),    # rows past the keys, not split
    (1, 2, 1, 64, 130, 1000, torch.bfloat16, True, None, None, -0.125),   # keys past the rows
    (1, 2, 1, 64, 1100, 1100, torch.float16, True, None, None, 0.0),      # scale 0, split
]


@pytest.mark.parametrize("case", CAUSAL64, ids=lambda c: f"B{c[0]}H{c[1]}-{c[2]}D{c[3]}T{c[4]}-{c[5]}")
def test_causal_head_dim_64(cuda, case):
    B, Hq, Hk, D, Tq, Tk, dtype, causal, mask, score, scale = case
    plan = _plan(B, Hq, Hk, D, Tq, Tk, causal, mask, score)
    print("case", case, "ranges", plan.key_split, flush=True)
    _check(4, *case)


def test_backward_after_a_forward_that_read_the_mask_itself(cuda):
    """The fwd op without ``residual`` leaves no prepared mask where its kernels
    read the bytes; the bwd op then prepares it: same gradients as with it."""
    q, k, v, m, _ = _inputs(3, 2, 4, 2, 64, 40, 500, torch.bfloat16, "bernoulli", None)
    q, k, v, m = (x.to(cuda) for x in (q, k, v, m))
    ops = torch.ops.tilelang_fa2_4d_mask
    O, L, ws, lo = ops.fwd(q, k, v, m, None, 0.125, False, False, False)
    _, _, ws1, _ = ops.fwd(q, k, v, m, None, 0.125, False, False, True)
    assert ws.numel() == 0 and ws1.numel() > 0
    do = torch.randn_like(O)
    a = ops.bwd(do, q, k, v, O, L, m, None, ws, lo, 0.125, False, False)
    b = ops.bwd(do, q, k, v, O, L, m, None, ws1, lo, 0.125, False, False)
    for x, y in zip(a, b):
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(), y.nan_to_num())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Tq", [1, 40, 200])
@pytest.mark.parametrize("where", ["k", "v", "v_inf"])
def test_non_finite_keys_under_infinite_scores(cuda, D, Tq, where):
    """A score of -inf keeps its key: NaN in its K row, NaN or Inf in its V row
    reach O (0 times them is NaN), whether or not other keys of its tile have
    finite scores."""
    q, k, v, _, _ = _inputs(5, 2, 4, 2, D, Tq, 300, torch.bfloat16, None, None)
    s = torch.zeros((2, 1, Tq, 300))
    s[0, ..., :200] = -math.inf         # whole tiles
    s[1, ..., 100:105] = -math.inf
    x = k if where == "k" else v
    for b, h, j in ((0, 0, 70), (1, 1, 102)):
        x[b, j, h] = math.inf if where == "v_inf" else math.nan
    dv = [t.to(cuda) for t in (q, k, v)]
    with torch.no_grad():
        O = torch.ops.tilelang_fa2_4d_mask.fwd(*dv, None, s.to(cuda), 0.1, False, False, False)[0].cpu()
    ref = E.eager_ref(*(t.transpose(1, 2).double() for t in (q, k, v)), None, s, scale=0.1, is_causal=False,
                      compute_dtype=torch.float64).transpose(1, 2)
    bad = torch.isnan(ref)
    assert bad[0, :, :2].all() and bad[1, :, 2:].all() and not bad[0, :, 2:].any() and not bad[1, :, :2].any()
    assert torch.equal(torch.isnan(O), bad)
