"""GQA decode attention (csrc/attention_mfma.hip) at the edges of its steps, waves and slices, against fp64."""
import math

import pytest
import torch

from src import ops

pytestmark = pytest.mark.gpu
PAGE = 64


@pytest.mark.parametrize("D,nh,nkv", [(128, 8, 2), (128, 8, 1), (128, 16, 1), (128, 4, 2), (64, 8, 2), (64, 2, 2)])
@pytest.mark.parametrize("ctxs,part", [([1, 31, 32, 33, 64, 65], 128), ([127, 128, 129, 159, 160, 161], 256),
                                       ([1, 96, 511, 640, 900], 128), ([1, 2300], 256), ([40, 8197], 128)])
def test_edges(D, nh, nkv, ctxs, part):
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

    def turned(x, pos):  # in 32 bits, rounded to bf16 as the cache holds it
        a, b = x.float().chunk(2, -1)
        c, s = cos[pos], sin[pos]
        return torch.cat([a * c - b * s, b * c + a * s], -1).to(torch.bfloat16)

    want, bound, news, slots = [], [], [], []
    for t, c in enumerate(ctxs):
        own, at = at[:pages[t]], at[pages[t]:]
        tables[t, :pages[t]] = own
        k, v = (torch.randn(c, nkv, D, generator=g).to(torch.bfloat16) for _ in range(2))
        for i in range(c - 1):
            kc[own[i // PAGE], :, i % PAGE], vc[own[i // PAGE], :, i % PAGE] = k[i], v[i]
        q, kn, vn = (x.view(-1, D) for x in qkv[t].split([nh * D, nkv * D, nkv * D]))
        q, k[c - 1], v[c - 1] = turned(q, c - 1), turned(kn, c - 1), vn
        news.append((k[c - 1], v[c - 1]))
        slots.append(int(own[(c - 1) // PAGE]) * PAGE + (c - 1) % PAGE)
        kd, vd = (x.double().repeat_interleave(nh // nkv, 1) for x in (k, v))
        s = torch.einsum("hd,chd->hc", q.double(), kd) / math.sqrt(D)
        p = s.softmax(-1)
        want.append(torch.einsum("hc,chd->hd", p, vd))
        # p rounded to bf16 (2^-8 of each, the sum's included) and the result (2^-8); an element of q or k may round the
        # other way where the 32-bit rotation is fused: 2^-8 of one product in a score
        e = 2 ** -8 * (2 + 4 * (q.double().abs().max() * kd.abs().max() / math.sqrt(D)).item())
        bound.append(e * torch.einsum("hc,chd->hd", p, vd.abs()))
    dev = [x.cuda() for x in (qkv, kc, vc, tables, torch.arange(T, dtype=torch.int32), torch.tensor(ctxs, dtype=torch.int32))]
    blocks = torch.stack([torch.arange(T), torch.ones(T, dtype=torch.long)]).to(torch.int32).cuda()
    got = ops.attention_mfma_rope(*dev, blocks, torch.tensor(ctxs).cuda() - 1, cos.cuda(), sin.cuda(),
                                  torch.tensor(slots).cuda(), nh, nkv, D ** -0.5, part_size=part, num_parts=parts)
    err = (got.cpu().double().view(T, nh, D) - torch.stack(want)).abs()
    assert (err <= torch.stack(bound) + 1e-9).all(), (err / torch.stack(bound)).max()
    for t, (k, v) in enumerate(news):  # the new token's row is in the cache (k: last bit as above)
        p, i = divmod(slots[t], PAGE)
        assert torch.equal(dev[2][p, :, i].cpu(), v)
        assert ((dev[1][p, :, i].cpu().float() - k.float()).abs() <= 2 ** -7 * k.float().abs() + 1e-6).all()
