"""GQA decode attention (csrc/attention_mfma.hip) at the edges of its steps, waves and slices, and the sum of a prompt's
slices (csrc/attention.hip), against fp64.

The references start from the queries and keys that the kernels multiply, bit for bit, so all that is left between the two
is bf16: weights p are rounded to 8 bits, in the sum of values and in its denominator, and so is the result.  A unit of that
rounding is 2^-8 of the number, which makes |error| <= 2^-8 (sum p |v| + 2 |out|); 32-bit sums take a hundredth of it.

``marked`` values stand for the slice they are in: one column is theirs (the last one is the new token's), so a slice's
weight is a result of its own and not a small part of one.
"""
import math

import pytest
import torch

from src import ops

PAGE = 64
SHAPES = [(128, 8, 2), (128, 8, 1), (128, 16, 1), (128, 4, 2), (64, 8, 2), (64, 2, 2)]


def _turn(x, cos, sin):
    """The kernels' rotation: entry d with d + D / 2, the second product rounded to 32 bits first, then to bf16."""
    a, b = x.double().chunk(2, -1)
    c, s = cos.double(), sin.double()
    rounded = lambda t: t.float().double()  # noqa: E731
    return torch.cat([(a * c - rounded(b * s)).float(), (a * s + rounded(b * c)).float()], -1).to(torch.bfloat16)


def _values(n, nkv, D, part, marked, g, new=True):
    """Values of a context of n tokens in slices of ``part``."""
    if not marked:
        return torch.randn(n, nkv, D, generator=g).to(torch.bfloat16)
    v = torch.zeros(n, nkv, D)
    v.scatter_(2, (torch.arange(n) // part % (D - 1))[:, None, None].expand(n, nkv, 1), 1.0)
    if new:
        v[n - 1] = 0.0
        v[n - 1, :, D - 1] = 1.0
    return (v * (0.5 + torch.rand(n, nkv, 1, generator=g))).to(torch.bfloat16)


def _attend(q, k, v, weight=None):
    """(output, bound) [heads, D] of queries [heads, D] over k and v [context, kv heads, D]; ``weight`` [context]: how often
    each token counts."""
    rep = q.shape[0] // k.shape[1]
    kd, vd = (x.double().repeat_interleave(rep, 1) for x in (k, v))
    s = torch.einsum("hd,chd->hc", q.double(), kd) / math.sqrt(q.shape[1])
    e = torch.exp(s - s.amax(-1, keepdim=True)) * (1.0 if weight is None else weight)
    p = e / e.sum(-1, keepdim=True)
    out = torch.einsum("hc,chd->hd", p, vd)
    return out, 1.01 * 2 ** -8 * (torch.einsum("hc,chd->hd", p, vd.abs()) + 2 * out.abs())


@pytest.mark.gpu
@pytest.mark.parametrize("T,nkv", [(4, 2), (8, 8), (12, 1), (16, 2), (24, 3)])
def test_every_session_and_slice_is_met(T, nkv):
    """Grids whose columns (sessions) are turned over the XCDs, with slices that shorter sessions do not have."""
    test_edges(64, 4 * nkv, nkv, [1 + 37 * t * t % 401 for t in range(T)], 128, True)


@pytest.mark.gpu
@pytest.mark.parametrize("marked", [False, True])
@pytest.mark.parametrize("D,nh,nkv", SHAPES)
@pytest.mark.parametrize("ctxs,part", [([1, 31, 32, 33, 64, 65], 128), ([127, 128, 129, 159, 160, 161], 256),
                                       ([1, 96, 511, 640, 900], 128), ([1, 2300], 256), ([40, 8197], 128),
                                       ([1, 97, 511, 512, 513, 640, 1153, 2300], 512)])
def test_edges(D, nh, nkv, ctxs, part, marked):
    """Slices past a context, waves without a step, tails of a step, 1 to 65 slices; the cache past each context is NaN."""
    ops.require_native()
    g = torch.Generator().manual_seed(D + nh + sum(ctxs))
    T, parts = len(ctxs), math.ceil(max(ctxs) / part)
    pages = [-(-c // PAGE) for c in ctxs]
    tables, at = torch.zeros(T, max(pages), dtype=torch.int32), torch.randperm(sum(pages), generator=g).to(torch.int32)
    kc = torch.full((sum(pages), nkv, PAGE, D), float("nan")).to(torch.bfloat16)
    vc = kc.clone()
    qkv = torch.randn(T, (nh + 2 * nkv) * D, generator=g).to(torch.bfloat16)
    ang = torch.arange(max(ctxs))[:, None] / 1e4 ** (torch.arange(D // 2)[None] * 2 / D)
    cos, sin = ang.cos().float(), ang.sin().float()
    want, bound, news, slots = [], [], [], []
    for t, c in enumerate(ctxs):
        own, at = at[:pages[t]], at[pages[t]:]
        tables[t, :pages[t]] = own
        k, v = torch.randn(c, nkv, D, generator=g).to(torch.bfloat16), _values(c, nkv, D, part, marked, g)
        for i in range(c - 1):
            kc[own[i // PAGE], :, i % PAGE], vc[own[i // PAGE], :, i % PAGE] = k[i], v[i]
        qkv[t, (nh + nkv) * D:] = v[c - 1].flatten()
        q, kn, _ = (x.view(-1, D) for x in qkv[t].split([nh * D, nkv * D, nkv * D]))
        k[c - 1] = _turn(kn, cos[c - 1], sin[c - 1])
        news.append((k[c - 1], v[c - 1]))
        slots.append(int(own[(c - 1) // PAGE]) * PAGE + (c - 1) % PAGE)
        for x, y in zip((want, bound), _attend(_turn(q, cos[c - 1], sin[c - 1]), k, v)):
            x.append(y)
    dev = [x.cuda() for x in (qkv, kc, vc, tables, torch.arange(T, dtype=torch.int32), torch.tensor(ctxs, dtype=torch.int32))]
    blocks = torch.stack([torch.arange(T), torch.ones(T, dtype=torch.long)]).to(torch.int32).cuda()
    got = ops.attention_mfma_rope(*dev, blocks, torch.tensor(ctxs).cuda() - 1, cos.cuda(), sin.cuda(),
                                  torch.tensor(slots).cuda(), nh, nkv, D ** -0.5, part_size=part, num_parts=parts)
    err = (got.cpu().double().view(T, nh, D) - torch.stack(want)).abs()
    assert (err <= torch.stack(bound) + 1e-9).all(), (err / torch.stack(bound)).max()
    for t, (k, v) in enumerate(news):  # the new token's row is in the cache
        p, i = divmod(slots[t], PAGE)
        assert torch.equal(dev[2][p, :, i].cpu(), v) and torch.equal(dev[1][p, :, i].cpu(), k)


@pytest.mark.parametrize("D,nh,nkv", [(128, 8, 2), (64, 8, 2)])
@pytest.mark.parametrize("ctx,part", [(8197, 128), (2300, 256), (900, 128)])
def test_bound_sees_every_slice(D, nh, nkv, ctx, part):
    """A slice left out or counted twice, or the new token lost, is past the bound of the marked values (oracle only)."""
    g = torch.Generator().manual_seed(D + ctx)
    q, k = torch.randn(nh, D, generator=g).to(torch.bfloat16), torch.randn(ctx, nkv, D, generator=g).to(torch.bfloat16)
    v = _values(ctx, nkv, D, part, True, g)
    want, bound = _attend(q, k, v)
    wrong = [(s, n) for s in range(-(-ctx // part)) for n in (0.0, 2.0)] + [(None, 0.0)]
    for s, n in wrong:
        w = torch.ones(ctx, dtype=torch.float64)
        w[ctx - 1 if s is None else slice(s * part, (s + 1) * part)] = n
        assert ((_attend(q, k, v, w)[0] - want).abs() > 2 * bound).any(), (s, n)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv", [(4, 1), (4, 4)])
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 7, 8, 9, 17])
def test_slices_of_a_prompt_are_added(parts, nh, nkv):
    """Every form of the sum (2, 4, 8 at once, any number) over many rows, of which early ones have empty slices."""
    ops.require_native()
    D, T = 128, 64 * parts - 5
    g = torch.Generator().manual_seed(parts + nkv)
    q, k = torch.randn(T, nh, D, generator=g).to(torch.bfloat16), torch.randn(T, nkv, D, generator=g).to(torch.bfloat16)
    v = _values(T, nkv, D, 64, True, g, new=False)
    kc, vc = (torch.zeros(parts, PAGE, nkv, D, dtype=x.dtype).view(-1, nkv, D).index_copy(0, torch.arange(T), x)
              .view(parts, PAGE, nkv, D).transpose(1, 2).contiguous().cuda() for x in (k, v))
    bt = torch.arange(parts, dtype=torch.int32)[None].cuda()
    ctx = torch.arange(1, T + 1, dtype=torch.int32)
    blocks = torch.from_numpy(ops.fa_blocks([T], nh // nkv, 4)).cuda()
    got = ops.attention_fa(q.view(T, -1).cuda(), kc, vc, bt, torch.zeros(T, dtype=torch.int32).cuda(), ctx.cuda(), blocks, nh,
                           nkv, D ** -0.5, max_ctx=T, waves=4, num_parts=parts)
    for t in sorted({0, 1, 62, 63, 64, T // 2, T - 65, T - 2, T - 1} & set(range(T))):
        want, bound = _attend(q[t], k[:t + 1], v[:t + 1])
        err = (got[t].cpu().double().view(nh, D) - want).abs()
        assert (err <= bound + 1e-9).all(), (t, (err / bound).nan_to_num().max())
