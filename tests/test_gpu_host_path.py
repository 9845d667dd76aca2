"""The native eager host path (csrc/fa_host.cpp) against the general one (the
registered custom ops): the same launches, so the same bits, over the forms of
operands it takes and those it hands back; and what autograd expects of its
node."""

import pytest
import torch

import tilelang_fa2_4d_mask as api
import tilelang_fa2_4d_mask.fa2 as F

pytestmark = pytest.mark.gpu


def _qkv(dev, layout, D=64, B=2, Hq=4, Hk=2, Tq=70, Tk=90, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    out = []
    for T, H in ((Tq, Hq), (Tk, Hk), (Tk, Hk), (Tq, Hq)):
        x = torch.randn((B, T, H, D), generator=g).to(dtype).to(dev)
        if layout != "bshd":
            x = x.transpose(1, 2)
        if layout == "bhsd_contiguous":
            x = x.contiguous()
        out.append(x)
    return out


def _step(q, k, v, do, layout, **kw):
    q, k, v = (x.detach().requires_grad_(True) for x in (q, k, v))
    out = api.tilelang_flash_attention(q, k, v, layout=layout[:4], use_atomic_backward=False, **kw)
    return (out, *torch.autograd.grad(out, (q, k, v), do))


def _both(monkeypatch, fn):
    a = fn()
    with monkeypatch.context() as m:
        m.setattr(F, "_plain_eager", lambda *t: False)
        b = fn()
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype
        assert torch.equal(x, y)
    return a


@pytest.mark.parametrize("layout", ["bhsd", "bhsd_contiguous", "bshd"])
@pytest.mark.parametrize("side", ["none", "mask", "mask_b1", "score", "both", "mask_strided"])
@pytest.mark.parametrize("D", [64, 96, 256, 40])
def test_same_bits(cuda, monkeypatch, layout, side, D):
    q, k, v, do = _qkv(cuda, layout, D)
    g = torch.Generator().manual_seed(1)
    m = (torch.rand((2, 4, 70, 90), generator=g) < 0.8).to(cuda)
    m[..., 0] = True
    kw = dict(is_causal=side in ("none", "score"))
    if side == "mask_b1":
        kw["mask"] = m[:1, :1]
    elif side in ("mask", "both"):
        kw["mask"] = m[:, :1]
    elif side == "mask_strided":
        kw["mask"] = m.transpose(2, 3).contiguous().transpose(2, 3)
    if side in ("score", "both"):
        kw["score"] = torch.randn((1, 4, 70, 90), generator=g).to(cuda)
    _both(monkeypatch, lambda: _step(q, k, v, do, layout, **kw))
    with torch.no_grad():
        _both(monkeypatch, lambda: (api.tilelang_flash_attention(q, k, v, layout=layout[:4], **kw),))


def test_output_gradients_to_copy(cuda, monkeypatch):
    q, k, v, _ = _qkv(cuda, "bhsd")

    def total():      # dO: stride 0 everywhere
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        return torch.autograd.grad(api.tilelang_flash_attention(*x, use_atomic_backward=False).sum(), x)

    def rows():       # dO: zeros but one row; only k asks for a gradient
        kk = k.detach().requires_grad_(True)
        return torch.autograd.grad(api.tilelang_flash_attention(q, kk, v, use_atomic_backward=False)[:, :, 3].float().sum(), kk)

    _both(monkeypatch, total)
    _both(monkeypatch, rows)


def test_native_path_runs(cuda, monkeypatch):
    """The plain call does not reach the custom ops."""
    from tilelang_fa2_4d_mask import ops

    def refuse(*a, **k):
        raise AssertionError("general path")

    monkeypatch.setattr(ops, "attention", refuse)
    monkeypatch.setattr(F, "_general_backward", refuse)
    q, k, v, do = _qkv(cuda, "bhsd", 96)
    _step(q, k, v, do, "bhsd", is_causal=True)


def test_autograd_contract(cuda):
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]

    out = api.tilelang_flash_attention(*leaf)
    out.mul_(2)                                      # the saved output changes
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        out.backward(do)
    out = api.tilelang_flash_attention(*leaf)
    with torch.no_grad():
        leaf[0].add_(1)                              # a saved input changes
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        out.backward(do)

    out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    a = torch.autograd.grad(out, leaf, do, retain_graph=True)
    b = torch.autograd.grad(out, leaf, do)           # again, then never more
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, leaf, do)

    moved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (moved.append(t.shape), t.cpu())[1], lambda t: t.to(cuda)):
        out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    assert len(moved) >= 5
    c = torch.autograd.grad(out, leaf, do)
    assert all(torch.equal(x, y) for x, y in zip(a, c))

    out = api.tilelang_flash_attention(*leaf)
    g = torch.autograd.grad(out, leaf, do, create_graph=True)
    with pytest.raises(RuntimeError):                # no second derivative
        g[0].sum().backward()


def test_only_the_score_wants_a_gradient(cuda):
    """It gets none, but the output takes part in autograd as through the custom op."""
    q, k, v, do = _qkv(cuda, "bhsd")
    score = torch.zeros((1, 1, 70, 90), device=cuda, requires_grad=True)
    out = api.tilelang_flash_attention(q, k, v, score=score)
    assert out.requires_grad
    out.backward(do)
    assert score.grad is None


def test_settings_between_forward_and_backward(cuda, monkeypatch):
    """A dS limit or the event log set after the forward still rules its backward."""
    q, k, v, do = _qkv(cuda, "bhsd", Tq=300, Tk=300)
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    ref = torch.autograd.grad(api.tilelang_flash_attention(*leaf, use_atomic_backward=False), leaf, do)
    out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    with F.record_kernel_events() as log:
        got = torch.autograd.grad(out, leaf, do)
    assert {"fa_bwd_preprocess", "fa_bwd", "fa_bwd_finalize"} == set(log.elapsed_ms())
    assert all(torch.equal(x, y) for x, y in zip(ref, got))
    calls = []
    real = F._backward_impl
    monkeypatch.setattr(F, "_backward_impl", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    monkeypatch.setattr(F, "DS_LIMIT_BYTES", -1)
    torch.autograd.grad(out, leaf, do)
    assert calls == [1]


def test_transforms_and_streams(cuda, monkeypatch):
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]

    def loss(*x):
        return (api.tilelang_flash_attention(*x, use_atomic_backward=False) * do).float().sum()

    ref = torch.autograd.grad(loss(*leaf), leaf)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = torch.autograd.grad(loss(*leaf), leaf)
    torch.cuda.current_stream().wait_stream(s)
    assert all(torch.equal(x, y) for x, y in zip(ref, got))
    with torch.inference_mode():
        x = [t.clone() for t in (q, k, v)]
        assert torch.equal(api.tilelang_flash_attention(*x), api.tilelang_flash_attention(q, k, v))


@pytest.mark.parametrize("bad", ["mask_shape", "mask_device", "heads", "dtype", "head_dim"])
def test_refusals(cuda, monkeypatch, bad):
    """What the general path refuses, with its error, is refused the same way."""
    q, k, v, _ = _qkv(cuda, "bhsd")
    mask = None
    if bad == "mask_shape":
        mask = torch.ones((2, 3, 70, 90), dtype=torch.bool, device=cuda)
    elif bad == "mask_device":
        mask = torch.ones((2, 1, 70, 90), dtype=torch.bool)
    elif bad == "heads":
        k, v = k[:, :1].expand(2, 3, 90, 64), v[:, :1].expand(2, 3, 90, 64)
    elif bad == "dtype":
        q, k, v = q.float(), k.float(), v.float()
    elif bad == "head_dim":
        q, k, v = (torch.zeros((1, 2, 4, 320), dtype=torch.bfloat16, device=cuda) for _ in range(3))
    errors = []
    for general in (False, True):
        with monkeypatch.context() as m:
            if general:
                m.setattr(F, "_plain_eager", lambda *t: False)
            with pytest.raises(Exception) as e:
                F.flash_attention_with_4d_mask(q, k, v, mask)
            errors.append((type(e.value), str(e.value)))
    assert errors[0] == errors[1]


def test_batched_output_gradients(cuda):
    """A batch of output gradients in one backward (what a vectorised jacobian
    does) is the loop over single ones."""
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    G = torch.stack([do, 2 * do, torch.roll(do, 1, 2)])
    out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    got = torch.autograd.grad(out, leaf, G, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        ref = torch.autograd.grad(out, leaf, G[i], retain_graph=True)
        assert all(torch.equal(x[i], y) for x, y in zip(got, ref))


def test_dispatch_mode_around_the_backward_sees_it(cuda):
    """A dispatch mode entered after the forward sees the backward op, as it would
    one from the general path."""
    from torch.utils._python_dispatch import TorchDispatchMode

    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    ref = torch.autograd.grad(api.tilelang_flash_attention(*leaf, use_atomic_backward=False), leaf, do)
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
    with Mode():
        got = torch.autograd.grad(out, leaf, do)
    assert any("tilelang_fa2_4d_mask.bwd" in s for s in seen), seen
    assert all(torch.equal(x, y) for x, y in zip(ref, got))


def test_operands_that_are_not_their_memory(cuda, monkeypatch):
    """Negated and all-zero tensors (what complex views and autograd make of them)."""
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    _both(monkeypatch, lambda: _step(torch._neg_view(q), k, v, do, "bhsd"))
    _both(monkeypatch, lambda: (api.tilelang_flash_attention(q, k, v, score=torch._neg_view(torch.ones((1, 1, 70, 90), device=cuda))),))
    for g in (torch._neg_view(do), torch._efficientzerotensor(do.shape, dtype=do.dtype, device=cuda)):
        out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False)
        got = torch.autograd.grad(out, leaf, g, retain_graph=True)
        ref = torch.autograd.grad(out, leaf, (g + 0 * do).contiguous())
        assert all(torch.equal(x, y) for x, y in zip(got, ref))


def test_profiles_name_both_directions(cuda):
    q, k, v, do = _qkv(cuda, "bhsd")
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        _step(q, k, v, do, "bhsd")
    names = {e.key for e in prof.key_averages()}
    assert {"tilelang_fa2_4d_mask::fwd", "tilelang_fa2_4d_mask::bwd"} <= names


@pytest.mark.parametrize("general", [False, True])
def test_a_broadcast_mask_saved_on_the_host(cuda, monkeypatch, general):
    """save_on_cpu gives back a copy with a plane per head of a mask that the
    forward saw broadcast over them (and prepared as one plane)."""
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    m = (torch.rand((2, 1, 70, 90), generator=torch.Generator().manual_seed(1)) < 0.8).to(cuda)
    m[..., 0] = True
    if general:
        monkeypatch.setattr(F, "_plain_eager", lambda *t: False)
    ref = torch.autograd.grad(api.tilelang_flash_attention(*leaf, mask=m, use_atomic_backward=False), leaf, do)
    with torch.autograd.graph.save_on_cpu():
        out = api.tilelang_flash_attention(*leaf, mask=m, use_atomic_backward=False)
    got = torch.autograd.grad(out, leaf, do)
    assert all(torch.equal(x, y) for x, y in zip(ref, got))


@pytest.mark.parametrize("side", [False, True])
def test_saved_tensors_changed_by_hooks(cuda, side):
    """Hooks that give saved tensors back laid out otherwise change nothing; those
    that leave them in another type or on another device are refused."""
    q, k, v, do = _qkv(cuda, "bhsd")
    leaf = [x.detach().requires_grad_(True) for x in (q, k, v)]
    kw = {}
    if side:
        g = torch.Generator().manual_seed(1)
        m = torch.rand((2, 1, 70, 90), generator=g) < 0.8
        m[..., 0] = True
        kw = {"mask": m.to(cuda), "score": torch.randn((1, 4, 70, 90), generator=g).to(cuda)}

    def grads(unpack):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = api.tilelang_flash_attention(*leaf, use_atomic_backward=False, **kw)
        return torch.autograd.grad(out, leaf, do)

    ref = grads(lambda t: t)
    for a, b in ((-1, -2), (0, 1)):
        got = grads(lambda t: t.transpose(a, b).contiguous().transpose(a, b) if t.dim() > 1 else t)
        assert all(torch.equal(x, y) for x, y in zip(ref, got))
    for unpack in (lambda t: t.float(), lambda t: t.cpu(), lambda t: t.to(torch.float16) if t.is_floating_point() else t,
                   lambda t: t.cpu() if t.dtype == torch.float32 else t):
        with pytest.raises(ValueError):
            grads(unpack)
