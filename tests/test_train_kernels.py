"""Kernel form of the fine-tuning path (ops/train.py, runtime/autograd_stage.py) against 64-bit references, and which calls
take it."""
import dataclasses
import math

import pytest
import torch

from src.models.config import resolve_model
from src.models.weights import random_stage_weights
from src.runtime.autograd_stage import AutogradStage, _plain

# bf16 has 7 stored bits: a value in [1, 2) is rounded by at most half a unit of 2^-7, so by 2^-8 of itself
BF16 = 2.0 ** -8
EDGES = [1, 15, 16, 17, 63, 64, 65, 130]  # 16 rows a wave, 32 queries and 64 keys a tile


def _rel(x, y):
    return float((x.double().cpu() - y).norm() / y.norm().clamp_min(1e-30))


def _turn(x, T, D, sign=1.0):
    f = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    a = torch.arange(T, dtype=torch.float64)[:, None] * f
    c, s = torch.cos(a)[None, :, None], sign * torch.sin(a)[None, :, None]
    u, v = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _attend(q, k, v):
    B, T, nh, D = q.shape
    k, v = (t.repeat_interleave(nh // t.shape[2], 2).transpose(1, 2) for t in (k, v))
    s = q.transpose(1, 2) @ k.transpose(-1, -2) / math.sqrt(D)
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    return (torch.softmax(s, -1) @ v).transpose(1, 2), torch.logsumexp(s, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("T,D", [(1, 64), (2, 128), (777, 128), (100003, 64)])
def test_angles(T, D):
    """64-bit cosines and sines rounded once: the host's, but for values on the edge of a rounding."""
    from src import ops
    from src.ops import train
    from src.ops.reference import rope_cos_sin, rope_inv

    ops.require_native()
    scaling = {"rope_type": "llama3", "factor": 8.0, "original_max_position_embeddings": 8192} if T == 2 else None
    got = train.angles(rope_inv(D, 500000.0, scaling).cuda(), T).cpu()
    want = torch.cat(rope_cos_sin(D, T, 500000.0, None, scaling), 1)
    assert float((got != want).float().mean()) < 1e-4 and float((got - want).abs().max()) <= 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,D", [(4, 4, 128), (4, 1, 128), (6, 3, 64)])
@pytest.mark.parametrize("T", EDGES)
def test_attention_and_its_gradient(T, nh, nkv, D):
    """Results are bf16, rounded once: that rounding is the whole tolerance; everything in between is 32 bits or two bf16
    terms."""
    from src import ops
    from src.ops import train

    ops.require_native()
    B, gen = 2, torch.Generator().manual_seed(T + nh + D)
    x = torch.randn(B * T, (nh + 2 * nkv) * D, generator=gen).to(torch.bfloat16)
    do = torch.randn(B * T, nh * D, generator=gen).to(torch.bfloat16)
    f = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    a = torch.arange(T, dtype=torch.float64)[:, None] * f
    table = torch.cat([a.cos(), a.sin()], 1).float().cuda()
    qkv = train.rope_(x.cuda(), table, nh + nkv, D)
    w = x.double().view(B, T, -1, D)
    turned = torch.cat([_turn(w[:, :, :nh + nkv], T, D), w[:, :, nh + nkv:]], 2).reshape(B * T, -1)
    assert _rel(qkv, turned) < BF16
    # the attention from the same rounded rows, its gradient through the turn
    y = qkv.double().cpu().view(B, T, -1, D).requires_grad_(True)
    ref, lse = _attend(y[:, :, :nh], y[:, :, nh:nh + nkv], y[:, :, nh + nkv:])
    g, = torch.autograd.grad(ref, y, do.double().view(B, T, nh, D))
    g = torch.cat([_turn(g[:, :, :nh + nkv], T, D, -1.0), g[:, :, nh + nkv:]], 2).reshape(B * T, -1)
    out, out32, den = train.attention(qkv, B, nh, nkv, D, True)
    assert _rel(out, ref.detach().reshape(B * T, -1)) < BF16
    assert _rel(out32, ref.detach().reshape(B * T, -1)) < 1e-5  # hi + lo weights: 2^-17 a term
    assert torch.allclose(den.cpu().double().view(B, nh, T) * math.log(2.0), lse.detach(), atol=2e-5)
    again, _, _ = train.attention(qkv, B, nh, nkv, D, False)
    assert torch.equal(out, again)
    dq = train.attention_grad(qkv, B, nh, nkv, D, out32, den, do.cuda(), table)
    for lo, hi in ((0, nh), (nh, nh + nkv), (nh + nkv, nh + 2 * nkv)):
        r = g[:, lo * D:hi * D]
        if float(r.norm()) > 1e-9:  # (one token: its score has no gradient)
            assert _rel(dq[:, lo * D:hi * D], r) < BF16
        else:
            assert float(dq[:, lo * D:hi * D].abs().max()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("T,nh,D", [(64, 4, 128), (200, 4, 64), (700, 2, 128)])
def test_attention_is_no_less_exact_than_32_bits(T, nh, D):
    """What the kernels hold in 32 bits against 64 bits: no further off than softmax and products in 32 bits are, a quarter
    allowed for sums in another order.  (With probabilities and score gradients in 16 bits the output was 7 to 11 times as
    far off.)"""
    from src import ops
    from src.ops import train

    ops.require_native()
    gen = torch.Generator().manual_seed(T + D)
    x = torch.randn(T, 3 * nh * D, generator=gen).to(torch.bfloat16)
    do = torch.randn(T, nh * D, generator=gen).to(torch.bfloat16)

    def plain(dtype):
        y = x.to("cuda", dtype).view(1, T, 3 * nh, D).requires_grad_(True)
        out, _ = _attend(y[:, :, :nh], y[:, :, nh:2 * nh], y[:, :, 2 * nh:])
        g, = torch.autograd.grad(out, y, do.to("cuda", dtype).view(1, T, nh, D))
        return out.detach().reshape(T, nh * D), g[0, :, nh:2 * nh].reshape(T, -1), g[0, :, 2 * nh:].reshape(T, -1)

    _, out32, lse = train.attention(x.cuda(), 1, nh, nh, D, True)
    f32 = dict(dtype=torch.float32, device="cuda")
    part, table = torch.empty(2, T, nh * D, **f32), torch.cat([torch.ones(T, D // 2), torch.zeros(T, D // 2)], 1)
    torch.ops.mpamd.train_attn_grad(x.cuda(), 1, nh, nh, D ** -0.5, out32.view(-1), lse, do.cuda(), torch.empty(nh * T, **f32),
                                    table.cuda().view(-1), part.view(-1), torch.empty_like(x, device="cuda"))
    for name, got, ref, want in zip(("out", "dk", "dv"), (out32, part[0], part[1]), plain(torch.float32), plain(torch.float64)):
        assert _rel(got, want.cpu()) <= 1.25 * _rel(ref, want.cpu()), (name, _rel(got, want.cpu()), _rel(ref, want.cpu()))


@pytest.mark.gpu
def test_attention_passes_what_is_not_a_number():
    """A value or key that is not finite shows in every token from its own on, and in the gradients through those."""
    from src import ops
    from src.ops import train

    ops.require_native()
    T, nh, D, at = 130, 2, 64, 70
    gen = torch.Generator().manual_seed(1)
    x = torch.randn(T, 3 * nh * D, generator=gen).to(torch.bfloat16)
    do = torch.randn(T, nh * D, generator=gen).to(torch.bfloat16).cuda()
    table = torch.cat([torch.ones(T, D // 2), torch.zeros(T, D // 2)], 1).cuda()
    for col in (nh * D, 2 * nh * D):  # the first key, the first value
        for bad in (float("nan"), float("inf")):
            y = x.clone()
            y[at, col:col + D] = bad
            out, out32, lse = train.attention(y.cuda(), 1, nh, nh, D, True)
            dq = train.attention_grad(y.cuda(), 1, nh, nh, D, out32, lse, do, table)[:, :D]
            o = out[:, :D]
            assert not o[at:].isfinite().any() and o[:64].isfinite().all() and out[:, D:].isfinite().all()
            assert not dq[at:].isfinite().any() and dq[:64].isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("H", [8, 512, 2056, 4096, 4104, 16384])
def test_norm_and_its_gradient(H):
    from src import ops
    from src.ops import train

    ops.require_native()
    gen = torch.Generator().manual_seed(H)
    x, y, dy, res = (torch.randn(3, H, generator=gen).to(torch.bfloat16) for _ in range(4))
    w = (torch.rand(H, generator=gen) + 0.5).to(torch.bfloat16)
    total, out = train.norm(x.cuda(), w.cuda(), 1e-5, y.cuda())
    assert torch.equal(total.cpu(), x + y)
    t = (x + y).double().requires_grad_(True)
    ref = t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert _rel(out, ref.detach()) < BF16
    g, = torch.autograd.grad(ref, t, dy.double())
    dx = train.norm_grad(total, dy.cuda(), w.cuda(), 1e-5, res.cuda())
    assert _rel(dx, g + res.double()) < BF16
    same, out = train.norm(total, w.cuda(), 1e-5)
    assert same is total and _rel(out, ref.detach()) < BF16


@pytest.mark.gpu
@pytest.mark.parametrize("F", [16, 48, 1040])
def test_gate_gradient(F):
    from src import ops
    from src.models.weights import interleave_gate_up
    from src.ops import train

    ops.require_native()
    gen = torch.Generator().manual_seed(F)
    g, u, d = (2 * torch.randn(5, F, generator=gen).to(torch.bfloat16) for _ in range(3))
    gu = interleave_gate_up(g.t().contiguous(), u.t().contiguous()).t().contiguous().cuda()
    gd, ud = g.double().requires_grad_(True), u.double().requires_grad_(True)
    dg, du = torch.autograd.grad(torch.nn.functional.silu(gd) * ud, (gd, ud), d.double())
    ref = interleave_gate_up(dg.t().contiguous(), du.t().contiguous()).t()
    assert _rel(train.glu_grad_(gu, d.cuda()), ref) < BF16


@pytest.mark.gpu
@pytest.mark.parametrize("prompt", [None, (1, 3), (2, 5), (2, 0)])
@pytest.mark.parametrize("nkv", [4, 1])
def test_stage_on_kernels_against_the_plain_form(prompt, nkv, monkeypatch):
    """Both forms against the same blocks in 64 bits: the kernels are at least as close."""
    cfg = dataclasses.replace(resolve_model("small-llama"), num_key_value_heads=nkv)
    w = random_stage_weights(cfg, 1, 4, has_embed=False, has_head=False, device="cuda", seed=3)
    B, T, gen = 2, 70, torch.Generator().manual_seed(8)
    h, go = (torch.randn(B, T, cfg.hidden_size, generator=gen).to(torch.bfloat16) for _ in range(2))
    p = None if prompt is None else torch.randn(3, *prompt, cfg.hidden_size, generator=gen).to(torch.bfloat16)
    w64 = random_stage_weights(cfg, 1, 4, has_embed=False, has_head=False, device="cuda", seed=3)
    for lay in w64.layers:
        for n in ("input_norm", "qkv", "o", "post_norm", "gate_up", "down"):
            setattr(lay, n, getattr(lay, n).double().cpu())
    ex = AutogradStage(cfg, w64, "cpu", torch.float64)
    want = [ex.forward(h.double(), None if p is None else p.double())] + \
        list(ex.backward(h.double(), go.double(), None if p is None else p.double()))
    ag = AutogradStage(cfg, w, "cuda")
    hid = torch.empty(h.numel() + 1, dtype=h.dtype, device="cuda")[1:].view(h.shape).copy_(h)  # (not 16-byte aligned)

    def both():
        with torch.no_grad():
            out = ag.forward(hid, p)
        return [out] + list(ag.backward(hid, go, p))

    assert ag._kernels(hid, p)
    fast = both()
    monkeypatch.setattr(AutogradStage, "_kernels", lambda *a: False)
    slow = both()
    for f, s, r in zip(fast, slow, want):
        assert (f is None) == (s is None) == (r is None)
        if r is not None:
            assert f.shape == s.shape and f.dtype == s.dtype
        if r is not None and r.numel():
            assert _rel(f, r) <= 1.05 * _rel(s, r)


def test_which_calls_take_the_kernels(monkeypatch):
    """Everything but ordinary bf16 rows of a dense block keeps the plain form (route only: no GPU needed)."""
    from src import ops
    from src.ops import train

    monkeypatch.setattr(ops, "require_native", lambda: None)
    assert train.shape_ok(resolve_model("llama2-7b")) and train.shape_ok(resolve_model("mistral-7b"))
    assert not train.shape_ok(resolve_model("mixtral-8x7b")) and not train.shape_ok(resolve_model("gpt2"))
    cfg = resolve_model("tiny-llama")
    assert not train.shape_ok(dataclasses.replace(cfg, head_dim=96))
    assert train.rows_ok(1, 1) and train.rows_ok(65535, 7) and not train.rows_ok(65536, 1) and not train.rows_ok(0, 5)
    assert not train.rows_ok(1, 0) and not train.rows_ok(1, (1 << 24) + 1)
    w = random_stage_weights(cfg, 0, 2, has_embed=False, has_head=False, device="cpu")
    ag = AutogradStage(cfg, w, "cpu")
    h = torch.randn(1, 4, cfg.hidden_size, dtype=torch.bfloat16)
    assert not ag._kernels(h, None)  # the CPU
    assert _plain(h) and _plain(torch.nn.Parameter(h)) and not _plain(torch.nn.Buffer(h).as_subclass(_Sub))
    with torch.autograd.forward_ad.dual_level():
        assert not _plain(h)
    seen = []
    torch.func.vmap(lambda t: (seen.append(_plain(t)), t)[1])(h)
    assert seen == [False]

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, f, t, a=(), k=None):
            return f(*a, **(k or {}))

    with Mode():
        assert not _plain(h)


def test_forward_stays_differentiable():
    """A caller that differentiates ``forward`` itself, twice if it likes."""
    cfg = resolve_model("tiny-llama")
    w = random_stage_weights(cfg, 0, 1, has_embed=False, has_head=False, device="cpu", dtype=torch.float32)
    ag = AutogradStage(cfg, w, "cpu", torch.float32)
    h = torch.randn(1, 3, cfg.hidden_size, requires_grad=True)
    g, = torch.autograd.grad(ag.forward(h).square().sum(), h, create_graph=True)
    g2, = torch.autograd.grad(g.square().sum(), h)
    assert g2.abs().sum() > 0


class _Sub(torch.Tensor):
    pass
