"""Tiled expert products (csrc/moe.hip) at the edges of their tiles against 64-bit products."""
import pytest
import torch

from src import ops
from src.models.config import MoESpec
from src.ops import moe
from tests.test_prompt_gemm import gates_far_below_zero

pytestmark = pytest.mark.gpu

# rows of the experts: none, one, ends of a wave's 64 rows, of half a tile, of a tile, of a band of 8 tiles
COUNTS = {"small": [0, 1, 63, 64, 65], "tile": [127, 128, 129, 0, 255], "whole": [256, 257, 511], "band": [2049]}


def _lists(counts):
    E = len(counts)
    off = [sum(counts[:i]) for i in range(E + 1)]
    act = [e for e in range(E) if counts[e]]
    return torch.tensor(counts + off + act + [0] * (E - len(act)) + [len(act)], dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("rows", COUNTS)
@pytest.mark.parametrize("N,K", [(32, 64), (256, 128), (288, 192), (544, 320), (96, 96)])
@pytest.mark.parametrize("form", [2, 3])
def test_products(rows, N, K, form):
    """Every output is one sum of K exact products in 32 bits, rounded to bf16: half a unit of 2^-7 at most; gated forms
    round the gate's exponential too, far below that."""
    ops.require_native()
    counts = COUNTS[rows]
    E, R = len(counts), sum(counts)
    g = torch.Generator().manual_seed(N + K + R)
    T = R + 3
    x = torch.randn(T, K, generator=g).to(torch.bfloat16)
    tok = torch.randint(0, T, (R,), generator=g, dtype=torch.int32)
    w = torch.randn(E, N, K, generator=g).div(K ** 0.5).to(torch.bfloat16)
    wp = torch.stack([ops.pack_weight(m) for m in w.cuda()])
    lists, owner = _lists(counts), torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    z = torch.einsum("rk,rnk->rn", x.double()[tok.long()], w.double()[owner]) if R < 400 else \
        torch.cat([x.double()[tok[owner == e].long()] @ w[e].double().t() for e in range(E)])
    for glu, limit in ((0, 0.0), (1, 0.0), (1, 1.5)):
        out = torch.full((R, N // 2 if glu else N), float("nan"), dtype=torch.bfloat16, device="cuda")
        torch.ops.mpamd.moe_gemm(form, x.cuda(), tok.cuda(), lists, wp, out, R, T, glu, 16, limit, 0)
        want = z
        if glu:
            v = z.view(R, N // 32, 2, 16)
            a, b = v[:, :, 0].reshape(R, -1), v[:, :, 1].reshape(R, -1)
            want = torch.nn.functional.silu(a) * b if not limit else moe._glu(z, 16, limit)
        assert float((out.double().cpu() - want).norm() / want.norm()) < 2.0 ** -8
        again = torch.empty_like(out)
        torch.ops.mpamd.moe_gemm(form, x.cuda(), tok.cuda(), lists, wp, again, R, T, glu, 16, limit, 0)
        assert torch.equal(out, again)
    rows_in = x.cuda()[tok.long().cuda()].contiguous()  # sorted rows, fp32 out
    out = torch.full((R, N), float("nan"), device="cuda")
    torch.ops.mpamd.moe_gemm(form, rows_in, None, lists, wp, out, R, T, 0, 1, 0.0, 0)
    assert float((out.double().cpu() - z).norm() / z.norm()) < 1e-5


@pytest.mark.parametrize("E,N,K,each", [(70, 64, 64, 130), (3, 256, 128, 22400)])
def test_many_experts_and_many_tiles(E, N, K, each):
    """Experts past a wave's 64 lanes, and more than 64 tiles to a workgroup (which takes them 64 at a time); rows that begin
    at 8 bytes.  The tolerance as above."""
    ops.require_native()
    if E == 3:
        N = 16640  # 65 weight tiles of 264 row tiles: 17160 tiles on 256 workgroups
    counts = [each + e % 2 for e in range(E)]
    R = sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, K, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(E, N, K, generator=g, device="cuda").div(K ** 0.5).to(torch.bfloat16)
    wp, lists = torch.stack([ops.pack_weight(m) for m in w]), _lists(counts)
    room = torch.full((R * N + 4,), float("nan"), dtype=torch.bfloat16, device="cuda")
    for out in (room[:R * N].view(R, N), room[4:].view(R, N)):
        out.fill_(float("nan"))
        torch.ops.mpamd.moe_gemm(3, x, None, lists, wp, out, R, R, 0, 1, 0.0, 0)
        at = 0
        for e, n in enumerate(counts):
            want = x[at:at + n].float() @ w[e].float().t()
            assert float((out[at:at + n].float() - want).norm() / want.norm()) < 2.0 ** -8
            at += n


@pytest.mark.parametrize("form", [2, 3])
def test_not_a_number_stays_in_its_rows(form):
    """A row that holds something that is no number: its own outputs show it (with a limit the gate takes the limit for it, as
    the pass over a product's rows does), no other row does."""
    ops.require_native()
    E, N, K, R = 2, 64, 128, 300
    g = torch.Generator().manual_seed(form)
    x = torch.randn(R, K, generator=g).to(torch.bfloat16)
    x[70, 5], x[260, 9] = float("nan"), float("inf")
    w = torch.randn(E, N, K, generator=g).div(K ** 0.5).to(torch.bfloat16)
    wp, lists = torch.stack([ops.pack_weight(m) for m in w.cuda()]), _lists([180, 120])
    tok, bad = torch.arange(R, dtype=torch.int32).cuda(), torch.zeros(R, dtype=torch.bool)
    bad[70] = bad[260] = True
    for glu, limit in ((0, 0.0), (1, 0.0), (1, 1.5)):
        out = torch.empty(R, N // 2 if glu else N, dtype=torch.bfloat16, device="cuda")
        torch.ops.mpamd.moe_gemm(form, x.cuda(), tok, lists, wp, out, R, R, glu, 16, limit, 0)
        assert out[~bad].isfinite().all()
        if limit:
            z, want = torch.empty(R, N, dtype=torch.bfloat16, device="cuda"), torch.empty_like(out)
            torch.ops.mpamd.moe_gemm(form, x.cuda(), tok, lists, wp, z, R, R, 0, 16, 0.0, 0)
            ops.mixers.clamped_glu(z, want, 16, limit)
            assert torch.equal(out.isfinite(), want.isfinite())
        else:
            assert out[70].isnan().all() and not (out[260].isfinite() & (out[260] != 0)).any()


@pytest.mark.parametrize("counts,N,K", [([300, 0, 129, 100], 800, 4096), ([1062, 898, 793, 730, 607, 544, 435, 331], 4096, 4160),
                                        ([257] * 70, 304, 4096), ([2049], 768, 4160), ([40, 20], 512, 4096)])
def test_tiles_of_the_last_round_in_halves(counts, N, K):
    """With a workspace, whole tiles that some workgroups would make alone are cut at the middle of K (also of an odd number of
    stages), half-full ones go round; every output is written, none of the workspace is read that was not.  Two sums of half
    the products each, added in 32 bits: the tolerance as above."""
    ops.require_native()
    E, R = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, K, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(E, N, K, generator=g, device="cuda").div(K ** 0.5).to(torch.bfloat16)
    wp, lists = torch.stack([ops.pack_weight(m) for m in w]), _lists(counts)
    need = torch.ops.mpamd.moe_gemm_ws(3, K)
    assert need > 0 == torch.ops.mpamd.moe_gemm_ws(3, 4032)
    ws = torch.full((need,), float("nan"), device="cuda")
    out = torch.full((R, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    torch.ops.mpamd.moe_gemm(3, x, None, lists, wp, out, R, R, 0, 1, 0.0, 0, ws)
    at = 0
    for e, n in enumerate(counts):
        want = x[at:at + n].float() @ w[e].float().t()
        assert n == 0 or float((out[at:at + n].float() - want).norm() / want.norm()) < 2.0 ** -8
        at += n


@pytest.mark.parametrize("T,W,ff", [(2700, 4096, 4096), (600, 256, 2048)])
def test_the_same_prompt_has_the_same_bits(T, W, ff):
    """Tiles that are cut in K hold the same rows in each pass: an expert's rows lie in the order of their tokens."""
    ops.require_native()
    E, g = 8, torch.Generator(device="cuda").manual_seed(T)
    draw = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, router = draw(T, W).to(torch.bfloat16), draw(E, W).div(W ** 0.5).to(torch.bfloat16)
    up, down = (torch.stack([ops.pack_weight(m) for m in draw(E, *s).div(s[1] ** 0.5).to(torch.bfloat16)])
                for s in ((2 * ff, W), (W, ff)))
    spec, ctx = MoESpec(E, 2, ff, 0.0), torch.ones(T, dtype=torch.int32, device="cuda")
    assert moe.expert_form(2 * T, E, False) == 3

    def mlp():
        e = lambda name, shape, dtype=torch.bfloat16: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
        return moe.mixtral_mlp(x, ctx, router, up, down, spec, torch.empty_like(x), e)

    out = mlp()
    for _ in range(5):
        assert torch.equal(mlp(), out)


@pytest.mark.parametrize("T,E,top", [(17, 5, 2), (300, 64, 64), (511, 8, 2), (512, 8, 2), (1024, 65, 8), (4100, 512, 4), (9000, 3, 1)])
@pytest.mark.parametrize("ordered", [False, True])
def test_places_of_rows(T, E, top, ordered, monkeypatch):
    """Choices up to the ends of a wave's 64, of its share that stays in registers (512) and past it; tokens without a choice.
    Every row has its token and its expert; in the order of the tokens where the down product is cut."""
    ops.require_native()
    monkeypatch.setattr(moe, "_parts", lambda *a: int(ordered))
    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(T, 64, generator=g).to(torch.bfloat16), torch.randn(E, 64, generator=g).to(torch.bfloat16)
    ctx = (torch.rand(T, generator=g) < 0.9).to(torch.int32)
    e = lambda name, shape, dtype=torch.bfloat16: torch.full(shape, -7, dtype=dtype, device="cuda")  # noqa: E731
    spec = MoESpec(E, top, 64, 1.0)
    c = moe.choose(x.cuda(), w.cuda(), ctx.cuda(), spec, e)
    lists, slot, tok = c.lists.tolist(), c.slot.cpu(), c.tok.tolist()
    counts, off = lists[:E], lists[E:2 * E + 1]
    assert off == [sum(counts[:i]) for i in range(E + 1)] and off[E] == int(ctx.sum()) * top
    assert lists[3 * E + 1] == sum(n > 0 for n in counts)
    assert [tok[r] for r in slot[ctx > 0].flatten().tolist()] == [t for t in range(T) if ctx[t] for _ in range(top)]
    assert bool((slot[ctx == 0] == -1).all())
    for a, b in zip(off, off[1:]):
        assert len(set(tok[a:b])) == b - a and (not ordered or T <= 16 or tok[a:b] == sorted(tok[a:b]))


def test_which_rows_are_ordered():
    """Where the tiles of the last round are cut: wide experts with many rows each."""
    ops.require_native()
    for ff, tokens, packed, want in ((14336, 2700, False, True), (4096, 512, False, True), (4096, 511, False, False),
                                     (4032, 2700, False, False), (1408, 4298, False, False), (14336, 2700, True, False)):
        assert (moe._parts(MoESpec(8, 2, ff, 1.0), tokens, packed) > 0) == want


@pytest.mark.parametrize("counts", [[1, 0], [16, 17], [33, 64], [65, 3]])
def test_few_rows_of_large_experts(counts):
    """64 MB of experts and more come past the caches where an expert's rows are one pass (64), else from them; an odd number of
    weight tiles.  One sum of K exact products in 32 bits: 1e-5, gated ones rounded to bf16."""
    ops.require_native()
    E, N, K, R = 2, 4128, 4096, sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randn(R, K, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(E, N, K, generator=g, device="cuda").div(K ** 0.5).to(torch.bfloat16)
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).tolist()
    tok = torch.arange(R, dtype=torch.int32, device="cuda")
    for rows in (N, N - 16):  # the second: 257 tiles, 67 MB
        v = w[:, :rows].contiguous()
        assert v.numel() * 2 >= 64 << 20
        wp, lists = torch.stack([ops.pack_weight(m) for m in v]), _lists(counts)
        z = torch.stack([v[e].double() @ x[i].double() for i, e in enumerate(owner)])
        out = torch.full((R, rows), float("nan"), device="cuda")
        torch.ops.mpamd.moe_gemm(1, x, tok, lists, wp, out, R, R, 0, 1, 0.0, 0)
        assert float((out.double() - z).norm() / z.norm()) < 1e-5
        if rows % 32 == 0:
            u = z.view(R, rows // 32, 2, 16)
            want = torch.nn.functional.silu(u[:, :, 0].reshape(R, -1)) * u[:, :, 1].reshape(R, -1)
            act = torch.full((R, rows // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
            torch.ops.mpamd.moe_gemm(1, x, tok, lists, wp, act, R, R, 1, 16, 0.0, 0)
            assert float((act.double() - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.parametrize("K", [32, 96, 128, 672, 768, 800, 1408, 1568])
@pytest.mark.parametrize("n", [1, 17, 40])
def test_few_rows_of_any_depth(n, K):
    """Waves without a 32-column step, with fewer than are in flight at once (6, or 4 from 17 rows on), as many, one more and
    one less.  One sum of K exact products in 32 bits."""
    ops.require_native()
    counts = [n, 0, 3]
    E, N, R = len(counts), 48, sum(counts)
    g = torch.Generator().manual_seed(K + n)
    x = torch.randn(R, K, generator=g).to(torch.bfloat16)
    w = torch.randn(E, N, K, generator=g).div(K ** 0.5).to(torch.bfloat16)
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).tolist()
    z = torch.stack([w[e].double() @ x[i].double() for i, e in enumerate(owner)])
    out = torch.full((R, N), float("nan"), device="cuda")
    torch.ops.mpamd.moe_gemm(1, x.cuda(), torch.arange(R, dtype=torch.int32, device="cuda"), _lists(counts),
                             torch.stack([ops.pack_weight(m) for m in w.cuda()]), out, R, R, 0, 1, 0.0, 0)
    assert float((out.double().cpu() - z).norm() / z.norm()) < 1e-5


@pytest.mark.parametrize("form", [1, 2, 3])
def test_gates_far_below_zero(form):
    """g / (1 + exp(-g)) u, rounded to bf16 once; the exponential of 88 is 1e-5 of itself off."""
    ops.require_native()
    x, w, z = gates_far_below_zero("cuda")
    want = torch.nn.functional.silu(z[:, :16]) * z[:, 16:]
    out = torch.full((3, 16), float("nan"), dtype=torch.bfloat16, device="cuda")
    torch.ops.mpamd.moe_gemm(form, x, torch.arange(3, dtype=torch.int32, device="cuda"), _lists([3]), ops.pack_weight(w)[None].contiguous(),
                             out, 3, 3, 1, 16, 0.0, 0)
    assert float(((out.double() - want) / want).abs().max()) < 2.0 ** -8 + 2e-5


@pytest.mark.parametrize("counts", [[1, 0, 16], [300, 130, 20], [128, 257, 100]])
@pytest.mark.parametrize("N", [32, 160])
def test_nothing_behind_the_output(counts, N):
    """What lies behind the last expert's rows, up to where a whole tile would end, stays as it was."""
    ops.require_native()
    K, R = 128, sum(counts)
    g = torch.Generator().manual_seed(N + R)
    x = torch.randn(R, K, generator=g).to(torch.bfloat16)
    w = torch.randn(len(counts), N, K, generator=g).div(K ** 0.5).to(torch.bfloat16)
    wp, tok = torch.stack([ops.pack_weight(m) for m in w.cuda()]), torch.arange(R, dtype=torch.int32, device="cuda")
    z = torch.cat([r.double() @ w[e].double().t() for e, r in enumerate(x.split(counts))])
    for glu in (0, 1):
        room = torch.full((R + 512, N // (1 + glu)), -3.0, dtype=torch.bfloat16, device="cuda")
        torch.ops.mpamd.moe_gemm(3, x.cuda(), tok, _lists(counts), wp, room[:R], R, R, glu, 16, 0.0, 0)
        v = z.view(R, N // 32, 2, 16)
        want = torch.nn.functional.silu(v[:, :, 0].reshape(R, -1)) * v[:, :, 1].reshape(R, -1) if glu else z
        assert bool((room[R:] == -3.0).all())
        assert float((room[:R].double().cpu() - want).norm() / want.norm()) < 2.0 ** -8
