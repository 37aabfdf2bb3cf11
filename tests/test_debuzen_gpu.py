"""Debuzen on the GPU: every HIP kernel against the plain oracle (tests/debuzen_oracle.py), then the executor, its graphs
and the scheduler end to end, in bf16 and in 32-bit."""
import json
import os
import subprocess

import numpy as np
import pytest
import torch

from src import ops
from src.ops import mixers as mops
from src.ops import window as wops
from tests import debuzen_oracle as O
from tests import debuzen_utils as U
from tests.test_debuzen import edge_keys, leave_garbage

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
TOL = {"bf16": dict(atol=3e-2, rtol=2e-2), "fp32": dict(atol=2e-4, rtol=2e-4)}


def close(got, want, tol):
    torch.testing.assert_close(got.float().cpu(), want.float().cpu(), **tol)


def near(got, want, dt="bf16"):
    """bf16 operands are rounded, so an error has a size on the whole and a few outliers among a million."""
    if dt == "fp32":
        return close(got, want, TOL[dt])
    d, want = got.double().cpu() - want.double(), want.double()
    assert d.pow(2).mean().sqrt() < 6e-3 * want.pow(2).mean().sqrt()
    assert (d.abs() < 0.1 + 0.03 * want.abs()).all()


def unpack(x, n, W, packed):
    return ops.unpack_act(x, n, W) if packed else x


# ------------------------------------------------------------------ residual stream
@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("n,W,groups", [(1, 64, 1), (37, 70, 5), (5, 4096, 8), (300, 96, 3), (9, 33, 33), (70, 2048, 2), (3, 6144, 1)])
@pytest.mark.parametrize("form", ["norm", "replace", "copy"])
def test_stream_norms_in_parts(dt, n, W, groups, form):
    y, res, w = torch.randn(n, W).to(DTYPES[dt]), torch.randn(n, W), torch.randn(W)
    for packed in {False, dt == "bf16" and W % 32 == 0}:
        for part in {False, dt == "bf16" and W % 4 == 0}:  # split-K slabs of a decode product
            add = torch.randn(3, n, W) if part else y
            want = 0.5 * (add.double().sum(0) if part else add.double()) + (0 if form == "replace" else res.double())
            cols = 2 * W if form == "copy" else W
            r = res.to(DEV)
            x = torch.zeros((ops.packed_numel(n, cols),) if packed else (n, cols), dtype=DTYPES[dt], device=DEV)
            mops.add_norm(add.to(DEV), r, 0.5, None if form == "copy" else w.to(DEV), 1e-5, x, packed=packed, groups=groups,
                          keep=form != "replace", copy=cols if form == "copy" else 0)
            close(r, want, dict(atol=3e-5, rtol=3e-5))
            x = unpack(x, n, cols, packed)
            close(x[:, :W], want if form == "copy" else O.group_norm(want, w.double(), 1e-5, groups), TOL[dt])
            if form == "copy":
                assert (x[:, W:] == 0).all()


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("W,groups", [(64, 2), (70, 5), (4096, 8), (33, 1), (2048, 2)])
@pytest.mark.parametrize("decode", [False, True])
def test_token_shift(dt, W, groups, decode):
    """Steps of a few sequences at unlike places; a first token has nothing ahead of it, whatever the row holds."""
    g = torch.Generator().manual_seed(3)
    lens = [9, 70, 3, 20]
    res = [torch.randn(n, W, generator=g) for n in lens]
    w, mu = torch.randn(W, generator=g), torch.rand(W, generator=g)
    want = [O.shifted(O.group_norm(r.double(), w.double(), 1e-5, groups), mu.double()) for r in res]
    rows = torch.full((5, 2, W), 1e4, device=DEV)
    at = [0] * 4
    steps = [[1, 1, 1, 1]] * 3 if decode else [[2, 33, 1, 0], [1, 1, 2, 17], [6, 36, 0, 3]]
    for st in steps:
        parts = list(zip(at, st))
        seq, ctx = U._meta(parts)
        r = torch.cat([x[s:s + n] for x, (s, n) in zip(res, parts)]).to(DEV)
        n = r.shape[0]
        scratch = None if decode else (torch.empty(5, W, device=DEV), torch.empty(n, groups, device=DEV))
        packed = decode and dt == "bf16" and W % 32 == 0
        x = torch.zeros((ops.packed_numel(n, W),) if packed else (n, W), dtype=DTYPES[dt], device=DEV)
        mops.add_norm(None, r, 0.0, w.to(DEV), 1e-5, x, packed=packed, groups=groups,
                      shift=(mu.to(DEV), rows, seq.to(DEV), ctx.to(DEV), scratch))
        close(unpack(x, n, W, packed), torch.cat([x[s:s + n] for x, (s, n) in zip(want, parts)]), TOL[dt])
        at = [a + n for a, n in zip(at, st)]


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("W,groups", [(96, 3), (70, 1), (4096, 8), (33, 11)])
def test_normed_embedding_rows_and_soft_cap(dt, W, groups):
    table, i, w = torch.randn(50, W).to(DTYPES[dt]), torch.randint(0, 50, (9,)), torch.randn(W)
    want = O.group_norm(table[i].double(), w.double(), 1e-3, groups)
    for packed in {False, dt == "bf16" and W % 32 == 0}:
        res = torch.zeros(9, W, device=DEV)
        cat = torch.zeros((ops.packed_numel(9, 2 * W),) if packed else (9, 2 * W), dtype=DTYPES[dt], device=DEV)
        mops.embed_rows_norm(i.to(DEV), table.to(DEV), res, w.to(DEV), 1e-3, groups, cat, W, 2 * W, packed)
        close(res, want, dict(atol=2e-5, rtol=2e-5))
        cat = unpack(cat, 9, 2 * W, packed)
        close(cat[:, W:], want, TOL[dt])
        assert (cat[:, :W] == 0).all()
        out = torch.zeros((ops.packed_numel(3, W),) if packed else (3, W), dtype=DTYPES[dt], device=DEV)
        mops.rows_norm(res, torch.tensor([7, 0, 3], dtype=torch.int32, device=DEV), w.to(DEV), 1e-3, out, packed=packed, groups=groups)
        close(unpack(out, 3, W, packed), O.group_norm(want[[7, 0, 3]], w.double(), 1e-3, groups), TOL[dt])
    z = (30 * torch.randn(5, 157)).to(DTYPES[dt])
    close(mops.softcap(z.to(DEV), 12.5), O.soft_cap(z.double(), 12.5), TOL[dt])


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("F,block", [(24, 8), (20, 20), (7, 1), (512, 16)])
def test_silu_glu(dt, F, block):
    z = (3 * torch.randn(33, 2 * F)).to(DTYPES[dt])
    v = z.double().view(33, F // block, 2, block)
    want = (O.silu(v[:, :, 0]) * v[:, :, 1]).reshape(33, F)
    close(mops.clamped_glu(z.to(DEV), torch.empty(33, F, dtype=DTYPES[dt], device=DEV), block, 0.0), want, TOL[dt])


# ------------------------------------------------------------------ window attention
def run_window(a, form, splits=1, packed=False, rows=None):
    """form: any / blocks / rows; ``splits``: of the visible keys; ``rows``: of a query block."""
    T, H, V = a.q.shape[0], a.H, a.V
    kw = {}
    if form != "any":
        most = wops.mfma_ok(H, a.G, a.D, V, a.page)
        assert most
        rep = H // a.G
        if form == "blocks":
            rows = min(rows or most, most)
            kw = dict(form=1, blocks=torch.from_numpy(wops.window_blocks(a.ntoks, a.starts, rep, rows, a.size + a.keep)).to(DEV),
                      parts=(rows, 1))
        else:
            span = min(int(a.q_ctx.max()), a.size + a.keep) + 2 * (wops.KEYS - 1)
            ps = wops.KEYS * -(-span // (wops.KEYS * splits))
            kw = dict(form=2, parts=(ps, -(-span // ps)))
            if kw["parts"][1] > 1:
                kw["ws"] = torch.full((kw["parts"][1] * T * H * (V + 2),), 3.0, device=DEV)
    out = torch.zeros(ops.packed_numel(T, a.K) if packed else T * a.K, dtype=a.dt, device=DEV)
    out = out if packed else out.view(T, a.K)
    y = unpack(a.run(out, packed, **kw), T, a.K, packed)
    assert (y[:, :a.col] == 0).all() and (y[:, a.col + H * V:] == 0).all()
    return y[:, a.col:a.col + H * V]


PROMPT = ([70, 2, 1, 130, 33, 300], [0, 30, 63, 64, 100, 5])
MASKS = [(1, 0), (33, 0), (64, 3), (65, 64), (31, 1), (1000, 0), (20, 90)]
SHAPES = [(4, 2, 64, 64), (32, 8, 128, 128), (8, 8, 64, 48), (12, 4, 48, 16), (20, 5, 128, 80), (8, 1, 64, 128), (1, 1, 16, 16),
          (18, 6, 80, 32), (24, 12, 96, 112), (7, 7, 16, 32), (10, 2, 80, 96)]


def fit(H, G, D, V, page=64):
    return wops.mfma_ok(H, G, D, V, page)


@pytest.mark.parametrize("H,G,D,V", SHAPES)
@pytest.mark.parametrize("size,keep", MASKS)
@pytest.mark.parametrize("sigmoid", [False, True])
def test_window_prompts(H, G, D, V, size, keep, sigmoid):
    a = U.Window(*PROMPT, H, G, D, V, size, keep, sigmoid, dt=torch.bfloat16, device=DEV, page=64, col=16, pad=4, mult=1.3)
    want = a.want()
    most = fit(H, G, D, V)
    for rows in {64, most} - {0} if most else ():
        if rows >= H // G:
            near(run_window(a, "blocks", rows=rows), want)
    near(run_window(a, "any"), want)


@pytest.mark.parametrize("H,G,D,V", SHAPES)
@pytest.mark.parametrize("size,keep", MASKS)
@pytest.mark.parametrize("sigmoid", [False, True])
def test_window_decode(H, G, D, V, size, keep, sigmoid):
    starts = [0, 30, 31, 32, 33, 49, 63, 64, 65, 96, 200, 299, 511]
    for page in (32, 128):
        if not fit(H, G, D, V, page):
            continue
        a = U.Window([1] * len(starts), starts, H, G, D, V, size, keep, sigmoid, dt=torch.bfloat16, device=DEV, page=page,
                     col=32, pad=(-H * V) % 32)
        want = a.want()
        for splits in (1, 3):
            near(run_window(a, "rows", splits), want)
            near(run_window(a, "rows", splits, packed=True), want)


def test_the_usual_shapes_have_their_mfma_form():
    for s in ((32, 8, 128, 128), (4, 2, 64, 64), (24, 12, 96, 112), (8, 1, 64, 128)):
        assert fit(*s) >= 64


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("H,G,D,V", [(4, 2, 64, 64), (1, 1, 2, 1), (3, 1, 20, 6), (36, 6, 24, 10), (2, 2, 300, 200), (9, 3, 15, 14)])
@pytest.mark.parametrize("size,keep", [(1, 0), (17, 0), (16, 16), (40, 3), (200, 0)])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_window_any_shape(dt, H, G, D, V, size, keep, sigmoid):
    a = U.Window([20, 1, 2, 90], [0, 30, 15, 64], H, G, D, V, size, keep, sigmoid, dt=DTYPES[dt], device=DEV, page=16, col=5, pad=3,
                 mult=0.6)
    near(run_window(a, "any"), a.want(), dt)


@pytest.mark.parametrize("form", ["any", "blocks", "rows"])
@pytest.mark.parametrize("H,G,D,V", [(8, 2, 64, 64), (8, 8, 64, 32)])
@pytest.mark.parametrize("size,keep", [(72, 0), (64, 4), (128, 65), (1, 1), (33, 32)])
@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("i", [299, 192, 128, 63])
def test_a_key_that_stands_out(form, H, G, D, V, size, keep, sigmoid, i):
    """One key is what the query asks for: found just inside the window and among the kept first tokens, in a prompt and
    decoded, wherever its page is; just outside it leaves no trace."""
    ntoks, starts = ([1], [i]) if form == "rows" else ([i + 1], [0])
    for j in edge_keys(i, size, keep):
        res = []
        for sign in (1, -1):
            a = U.Window(ntoks, starts, H, G, D, V, size, keep, sigmoid, 32, dt=torch.bfloat16, device=DEV, page=64, spike=(i, j),
                         scale=0.25, head=None)
            a.z[0][j, (H + G) * D:] *= sign
            a.fill()
            got = run_window(a, form, 2)[-1]
            close(got, a.want()[-1], TOL["bf16"])
            res.append(got.float())
        d = (res[0] - res[1]).abs().max()
        assert (d > 0.5) if i - j < size or j < keep else (d == 0), (j, d)


@pytest.mark.parametrize("form", ["any", "blocks", "rows"])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_what_a_page_held_before_is_not_read(form, sigmoid):
    starts = [0, 40, 65, 130]
    ntoks, starts = ([1] * 4, starts) if form == "rows" else ([s + 1 for s in starts], [0] * 4)
    a = U.Window(ntoks, starts, 8, 2, 64, 64, 50, 3, sigmoid, dt=torch.bfloat16, device=DEV, page=64)
    a.cache.fill_(float("nan"))
    a.fill()
    near(run_window(a, form, 2), a.want())


@pytest.mark.parametrize("form", ["any", "blocks", "rows"])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_scores_far_from_zero(form, sigmoid):
    """Scores in the hundreds, both ways, and the first tokens, where sink or bias decide."""
    ntoks, starts = ([1] * 4, [0, 1, 2, 130]) if form == "rows" else ([1, 3, 140], [0, 0, 0])
    for head in (-60.0, 60.0):
        a = U.Window(ntoks, starts, 8, 2, 64, 64, 90, 2, sigmoid, dt=torch.bfloat16, device=DEV, page=64, scale=3.0, head=head)
        # (a score's rounding counts as it is)
        close(run_window(a, form, 2), a.want(), dict(atol=0.35, rtol=0.1))


def test_blocks_cover_every_token_once():
    for ntoks, starts, rep, rows in (([70, 0, 1, 130, 33], [0, 5, 63, 64, 100], 4, 64), ([1], [9], 8, 256), ([1024] * 8, [0] * 8, 1, 128),
                                     ([5000], [0], 12, 64), ([3] * 50, [7] * 50, 3, 64)):
        b = wops.window_blocks(ntoks, starts, rep, rows, 500)
        seen = np.concatenate([np.arange(t, t + n) for t, n in b.T])
        assert sorted(seen.tolist()) == list(range(sum(ntoks))) and b[1].max() * rep <= rows
        edges = np.cumsum([0] + ntoks)
        assert all(np.searchsorted(edges, t, "right") == np.searchsorted(edges, t + n - 1, "right") for t, n in b.T if n)


# ------------------------------------------------------------------ recurrences
GATED = [("gla", 2, 2, 32, 16), ("gla", 3, 3, 64, 40), ("gla", 2, 2, 128, 128), ("gla", 1, 1, 256, 64), ("gla", 2, 2, 20, 9),
         ("gla", 1, 1, 1, 1), ("gla", 1, 1, 300, 30), ("gated_delta", 4, 4, 64, 32), ("gated_delta", 4, 2, 128, 128),
         ("gated_delta", 2, 1, 24, 18), ("gated_delta", 2, 2, 256, 48), ("gated_delta", 6, 3, 16, 16), ("gated_delta", 1, 1, 1, 1),
         ("gated_delta", 2, 1, 272, 16), ("mamba2", 4, 2, 48, 48), ("mamba2", 6, 2, 128, 64), ("mamba2", 3, 3, 20, 10),
         ("mamba2", 2, 1, 200, 32), ("mamba2", 1, 1, 1, 1), ("mamba2", 8, 1, 16, 128), ("mamba2", 2, 2, 260, 8)]


def check_gated(a, got, dt):
    want, states = a.want()
    n = a.H * a.V
    g = torch.cat([torch.cat(x) for x in got])
    w = torch.cat([x[:sum(len(r) for r in y)] for x, y in zip(want, got)]).float()
    assert (g[:, :a.col] == 0).all() and (g[:, a.col + n:] == 0).all()
    d = g[:, a.col:a.col + n] - w
    err = d.pow(2).mean(1).sqrt() / w.pow(2).mean().sqrt()
    # (a sequence's first output is its value times one number, which may be near zero ahead of the norm)
    lim = (1.2e-2, 6e-3) if dt == "bf16" else (1e-4, 2e-5)
    if a.V > 1:  # (heads of one number: their norm is a sign, which any rounding near zero turns)
        assert err.quantile(0.9) < lim[0] and err.median() < lim[1], err
    assert torch.isfinite(d).all()
    s = states.float()
    d = a.state[1:].cpu() - s
    assert d.pow(2).mean().sqrt() < (1e-2 if dt == "bf16" else 1e-5) * s.pow(2).mean().sqrt()


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("kind,H,G,D,V", GATED)
@pytest.mark.parametrize("taps", [4, 1, 7])
def test_recurrences(dt, kind, H, G, D, V, taps):
    """Portions of many sizes beside decoded tokens, states carried from step to step."""
    if kind == "gla" and taps != 4:
        pytest.skip("no convolution")
    lens = [107, 1, 24, 200, 35]
    groups = 2 if kind == "mamba2" and H * V % 2 == 0 and H > 2 else 1
    A, R = (24, 40) if D % 16 == 0 else (5, 7)
    a = U.Gated(kind, lens, H, G, D, V, DTYPES[dt], DEV, taps, groups, ranks=(A, R), col=8, pad=8)
    got = [[] for _ in lens]
    for ntoks, decode in (([17, 1, 2, 130, 16], False), ([1, 0, 1, 1, 1], True), ([2, 0, 20, 33, 0], False), ([1, 0, 1, 1, 1], True),
                          ([1, 0, 0, 1, 1], True), ([70, 0, 0, 2, 16], False), ([15, 0, 0, 32, 0], False)):
        for i, r in enumerate(U.split(a.step(ntoks, decode), ntoks)):
            if r.numel():
                got[i].append(r)
    assert a.at == lens
    check_gated(a, got, dt)


@pytest.mark.parametrize("kind,D,V", [("mamba2", 16, 300), ("mamba2", 16, 301), ("gated_delta", 16, 320), ("gated_delta", 17, 258),
                                      ("mamba2", 16, 129), ("mamba2", 200, 32)])
@pytest.mark.parametrize("taps", [4, 16])
def test_convolutions_of_wide_heads(kind, D, V, taps):
    """Heads whose channels are four or eight to a lane, neighbours and not, and so two or four rows on their way: ends of rows and
    of blocks, from nothing and from a ring."""
    lens = [53, 1, 18]
    a = U.Gated(kind, lens, 2, 1, D, V, torch.bfloat16, DEV, taps, ranks=(24, 40) if D % 16 == 0 else (5, 7), col=8, pad=8)
    got = [[] for _ in lens]
    for ntoks in ([33, 1, 3], [17, 0, 15], [3, 0, 0]):
        for i, r in enumerate(U.split(a.step(ntoks), ntoks)):
            if r.numel():
                got[i].append(r)
    assert a.at == lens
    check_gated(a, got, "bf16")


@pytest.mark.parametrize("kind,H,G,D,V", [g for g in GATED if g[0] != "gated_delta" and g[3] <= 256])
def test_long_prompts_in_parts(kind, H, G, D, V):
    """Sequences cut into parts that run at once: from nothing, from an earlier state, beside short ones."""
    from src.ops.gated import chunk_plan

    lens, steps = [900, 1, 400, 140], ([17, 0, 400, 2], [700, 1, 0, 130], [183, 0, 0, 8])
    assert [len(set(chunk_plan(s, 16)["parts"][4])) > 2 for s in steps[:2]] == [True, True]
    A, R = (24, 40) if D % 16 == 0 else (5, 7)
    a = U.Gated(kind, lens, H, G, D, V, torch.bfloat16, DEV, ranks=(A, R), col=8, pad=8, tau=40.0, decay=-3.0)
    got = [[] for _ in lens]
    for ntoks in steps:
        for i, r in enumerate(U.split(a.step(ntoks, waves=16), ntoks)):
            if r.numel():
                got[i].append(r)
    assert a.at == lens
    check_gated(a, got, "bf16")


@pytest.mark.parametrize("kind,H,G,D,V", [("gla", 4, 4, 64, 64), ("gated_delta", 4, 2, 128, 64), ("mamba2", 4, 2, 64, 96),
                                          ("gated_delta", 8, 8, 32, 32)])
@pytest.mark.parametrize("packed", [False, True])
def test_recurrences_token_by_token(kind, H, G, D, V, packed):
    """Decode batches with padding rows, packed outputs."""
    lens = [40] * 5
    a = U.Gated(kind, lens, H, G, D, V, torch.bfloat16, DEV, ranks=(32, 16), col=64, pad=32)
    got = [[] for _ in lens]
    for _ in range(40):
        for i, r in enumerate(U.split(a.step([1] * 5, True, packed=packed, pads=3), [1] * 5)):
            got[i].append(r)
    check_gated(a, got, "bf16")
    b = U.Gated(kind, lens, H, G, D, V, torch.bfloat16, DEV, ranks=(32, 16), col=64, pad=32)
    b.step([40] * 5, packed=packed)
    d = (a.state[1:] - b.state[1:]).pow(2).mean().sqrt() / b.state[1:].pow(2).mean().sqrt()
    assert d < 8e-3  # prompt and decode leave the same state


@pytest.mark.parametrize("kind,H,G,D,V", [("gla", 2, 2, 64, 32), ("gated_delta", 2, 2, 64, 32), ("mamba2", 2, 2, 64, 32)])
@pytest.mark.parametrize("decay", [-8.0, 4.0])
def test_long_memory_and_sudden_loss(kind, H, G, D, V, decay):
    """Decays next to one over a thousand tokens, and decays that wipe the state in one."""
    a = U.Gated(kind, [1000, 33], H, G, D, V, torch.bfloat16, DEV, decay=decay, tau=1e4 if decay < 0 else 0.05, col=8, pad=8)
    got = [[], []]
    for ntoks in ([1, 16], [700, 2], [298, 15], [1, 0]):
        for i, r in enumerate(U.split(a.step(ntoks), ntoks)):
            got[i].append(r)
    check_gated(a, got, "bf16")


def test_steps_of_recurrences_cover_every_token_once():
    from src.ops.gated import CHUNK, chunk_plan

    for ntoks in ([70, 0, 1, 130, 33], [1], [16, 32, 0], [5000], [3] * 50):
        p = chunk_plan(ntoks)
        tok, n = p["chunks"]
        assert n.max() <= CHUNK and np.concatenate([np.arange(t, t + k) for t, k in zip(tok, n)]).tolist() == list(range(sum(ntoks)))
        off, cnt, first, k = p["seqs"]
        assert cnt.tolist() == [x for x in ntoks if x] and (tok[first] == off).all()
        assert (first + k == np.append(first[1:], len(tok))).all()
        cut = chunk_plan(ntoks, 100).get("parts")
        if cut is not None:
            o, n, f, b, part = cut
            assert (np.diff(f) == b[:-1]).all() and (tok[f] == o).all() and n.sum() == sum(ntoks) and (part == 0).sum() == len(off)
            assert (np.diff(part)[part[1:] > 0] == 1).all() and ((n == CHUNK * b) | (np.append(part[1:], 0) == 0)).all()


# ------------------------------------------------------------------ executor
@pytest.fixture(scope="module", params=sorted(U.MODELS) + ["packed"])
def model(request, tmp_path_factory):
    ranks = (5, 7)
    if request.param == "packed":  # every GEMM has a decode form, every mixer its MFMA forms
        cfg = U.config([U.par2(U.win(8, 2, 64, 64, 70, 32), U.ssd(4, 32, 64, 2, 4), 64),
                        U.par(U.win(4, 4, 32, 48, 90, 16, keep=3), U.delta(8, 4, 32, 16), 96), U.gla(4, 32, 64, 16.0, 128),
                        U.par2(U.win(6, 2, 48, 32, 33, 48), U.ssd(2, 64, 32, 1, 2, 3), 0)], vocab=333, width=256, groups=2,
                       loop=(1, 3, 2))
        ranks = (16, 32)
    else:
        cfg = U.MODELS[request.param]
    w = U.tensors(cfg, seed=3, ranks=ranks)
    return cfg, w, U.write(tmp_path_factory.mktemp(request.param), cfg, w), request.param


def check(got, want, dt, scale, name):
    got = got.float().cpu()
    assert torch.isfinite(got).all()
    err = (got - want).pow(2).mean(-1).sqrt() / scale
    if dt == "fp32":
        # (heads of one number: their norm magnifies a sum near zero)
        assert err.max() < (2e-2 if name == "ones" else 2e-3) and err.median() < 2e-4, err
    elif name != "ones":
        assert err.quantile(0.85) < 0.08 and err.max() < 1.5, err


@pytest.mark.parametrize("dt", sorted(DTYPES))
def test_prompts_decoding_portions_and_batches(model, dt):
    cfg, w, d, name = model
    n = 230
    toks = {k: U.ids(n, cfg["vocab"], s) for s, k in enumerate("abc")}
    want = {k: O.forward(cfg, w, t).float() for k, t in toks.items()}
    scale = want["a"].std()
    ex = U.executor(d, DEV, dt, max_sessions=4)
    check(ex.forward([("w", n)], toks["a"].to(DEV), logit_rows=range(n)), want["a"], dt, scale, name)
    ex.sessions.close("w")
    # one token at a time (graph replays), three sessions of different lengths together
    got = {k: [] for k in toks}
    at = {"a": 5, "b": 2, "c": 64}
    ex.forward(list(at.items()), torch.cat([toks[k][:m] for k, m in at.items()]).to(DEV))
    for _ in range(70):
        x = torch.cat([toks[k][at[k]:at[k] + 1] for k in toks]).to(DEV)
        y = ex.forward([(k, 1) for k in toks], x)
        assert ex.last_graphed
        for r, k in enumerate(toks):
            got[k].append(y[r].float().cpu())
            at[k] += 1
    for k, lo in (("a", 5), ("b", 2), ("c", 64)):
        check(torch.stack(got[k]), want[k][lo:lo + 70], dt, scale, name)
    # portions, short and long, beside decoded tokens
    pieces, wants = [], []
    for step in ({"a": 2, "b": 1}, {"b": 30, "c": 1, "a": 1}, {"a": 17, "b": 3}, {"c": 2, "a": 70, "b": 1},
                 {"b": 64, "a": 2, "c": 65}):
        x = torch.cat([toks[k][at[k]:at[k] + m] for k, m in step.items()]).to(DEV)
        pieces.append(ex.forward(list(step.items()), x, logit_rows=range(x.numel())).float().cpu())
        for k, m in step.items():
            wants.append(want[k][at[k]:at[k] + m])
            at[k] += m
    check(torch.cat(pieces), torch.cat(wants), dt, scale, name)
    # everything given back and used again, whatever it holds
    for k in toks:
        ex.sessions.close(k)
    leave_garbage(ex, 1e4)
    check(ex.forward([("z", n)], toks["b"].to(DEV), logit_rows=range(n)), want["b"], dt, scale, name)
    ex.sessions.close("z")
    leave_garbage(ex, float("nan"))
    y = [ex.forward([("d", 1)], toks["c"][i:i + 1].to(DEV)).float().cpu() for i in range(20)]
    check(torch.cat(y), want["c"][:20], dt, scale, name)


def test_graph_replays_equal_the_eager_step(model):
    """Decode graphs, replayed with other work between the replays."""
    cfg, w, d, _ = model
    t = [U.ids(60, cfg["vocab"], s) for s in range(3)]
    outs = []
    for graphs in (True, False):
        ex = U.executor(d, DEV, "bf16", use_graphs=graphs)
        ex.forward([(f"s{i}", 9 + i) for i in range(3)], torch.cat([x[:9 + i] for i, x in enumerate(t)]).to(DEV))
        got = []
        for k in range(20):
            got.append(ex.forward([(f"s{i}", 1) for i in range(3)], torch.stack([x[9 + i + k] for i, x in enumerate(t)]).to(DEV)).cpu())
            assert ex.last_graphed == graphs
            if k % 5 == 2:  # another shape and an eager step in between
                ex.forward([("o", 7 + k)], t[0][:7 + k].to(DEV), reset=[True])
                ex.forward([("o", 1)], t[0][:1].to(DEV))
                torch.cuda.synchronize()
        outs.append(torch.stack(got))
    assert torch.equal(outs[0], outs[1])


def test_long_contexts_of_whole_and_cut_prompts(model):
    """1100 tokens, then decoding: far behind every window, kept first tokens still there."""
    cfg, w, d, name = model
    if name != "packed":
        pytest.skip("one model is enough")
    n = 1100
    t = U.ids(n, cfg["vocab"], 7)
    want = O.forward(cfg, w, t, torch.float32).float()
    for dt in sorted(DTYPES):
        ex = U.executor(d, DEV, dt, max_seq_len=1280, max_tokens_per_step=2048)
        check(ex.forward([("w", n)], t.to(DEV), logit_rows=range(n)), want, dt, want.std(), name)
        at, got = 0, []
        for m in (700, 2, 63, 64, 1, 200, 3, 33, 1, 3) + (1,) * 30:
            got.append(ex.forward([("c", m)], t[at:at + m].to(DEV), logit_rows=range(m)).cpu())
            at += m
        assert at == n
        check(torch.cat(got), want, dt, want.std(), name)


def test_cuts_change_only_rounding(model):
    """The same tokens whole, in pairs and one by one differ by no more than the product's rounding."""
    cfg, w, d, name = model
    n = 64
    t = U.ids(n, cfg["vocab"], 11)
    ex = U.executor(d, DEV, "fp32")
    res = []
    for key, sizes in (("w", [n]), ("p", [2] * (n // 2)), ("d", [1] * n)):
        at, got = 0, []
        for m in sizes:
            got.append(ex.forward([(key, m)], t[at:at + m].to(DEV), logit_rows=range(m)).float().cpu())
            at += m
        res.append(torch.cat(got))
    for r in res[1:]:
        check(r, res[0], "fp32", res[0].std(), name)


def test_wide_decode_batches(model):
    """65 and more rows take other GEMM forms."""
    cfg, w, d, name = model
    ex = U.executor(d, DEV, "bf16", max_sessions=80, max_seq_len=64, kv_cache_bytes=512 << 20)
    t = U.ids(80 * 6, cfg["vocab"], 5).view(80, 6)
    ex.forward([(f"s{i}", 5) for i in range(80)], t[:, :5].reshape(-1).to(DEV))
    y = ex.forward([(f"s{i}", 1) for i in range(80)], t[:, 5].to(DEV)).float().cpu()
    want = torch.stack([O.forward(cfg, w, t[i])[-1].float() for i in range(80)])
    check(y, want, "bf16", want.std(), name)


def test_stage_split_equals_full(model):
    """The cut is inside the loop where the model has one: the embedding travels along."""
    cfg, w, d, _ = model
    n = len(O.runs(cfg))
    s0 = U.executor(d, DEV, "bf16", role="stage0", end=2)
    s1 = U.executor(d, DEV, "bf16", role="last", start=2, end=n)
    full = U.executor(d, DEV, "bf16")
    t = U.ids(50, cfg["vocab"]).to(DEV)
    for a, b in ((0, 40), (40, 41), (41, 42), (42, 50)):
        h = s0.forward([("a", b - a)], t[a:b])
        assert h.dtype == torch.float32 and h.shape[-1] == s0.cfg.hidden_width
        assert torch.equal(s1.forward([("a", b - a)], h), full.forward([("a", b - a)], t[a:b]))


def test_greedy_generation_through_the_scheduler(model):
    from tests.test_kafunex import serve

    cfg, w, d, name = model
    reqs = [(U.ids(n, cfg["vocab"], n).tolist(), 6 + n % 3) for n in (1, 2, 9, 40, 71)]
    want = [O.greedy(cfg, w, torch.tensor(p), n) for p, n in reqs]
    ex = U.executor(d, DEV, "fp32")
    assert serve(ex, reqs, batch=3, n_slots=2) == want
    assert serve(ex, reqs, batch=5, prefill_chunk=4, max_step_tokens=11) == want
    out = serve(U.executor(d, DEV, "bf16"), reqs, batch=4)  # bf16 may part from it at a near tie
    assert all(len(a) == len(b) for a, b in zip(out, want))


def test_trace_run_program(model, tmp_path):
    cfg, w, d, name = model
    if name != "packed":
        pytest.skip("one model is enough")
    a, b = U.ids(120, cfg["vocab"], 1), U.ids(90, cfg["vocab"], 2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:101].tolist(), "want": [5, 100]}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": b[:80].tolist(), "want": []},
                                     {"id": "a", "tokens": a[101:102].tolist(), "want": [0]}], "end": []},
             {"step": 2, "entries": [{"id": "b", "tokens": b[80:].tolist(), "want": []}], "end": ["b"]},
             {"step": 3, "entries": [{"id": "a", "tokens": a[102:].tolist(), "want": [7, 2]},
                                     {"id": "c", "tokens": b.tolist(), "want": [89]}], "end": ["a", "c"]}]
    A, B = O.forward(cfg, w, a).float(), O.forward(cfg, w, b).float()
    want = {0: A[[5, 100]], 1: A[[101]], 3: torch.stack([A[109], A[104], B[89]])}
    for dt, flag in (("fp32", "float32"), ("bf16", "bfloat16")):
        out = tmp_path / dt
        out.mkdir()
        r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", d, "--dtype", flag, "--out", str(out),
                            "--max-tokens", "256"], text=True, capture_output=True,
                           input="".join(json.dumps(s) + "\n" for s in steps), timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        for k, y in want.items():
            got = torch.from_numpy(np.fromfile(out / f"{k}.f32", "<f4").reshape(-1, cfg["vocab"]))
            check(got, y, dt, A.std(), name)
