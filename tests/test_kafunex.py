"""Kafunex on the CPU data path: configuration, loading, every mechanism alone, the executor, the scheduler and the
command line, against the plain oracle (tests/kafunex_oracle.py)."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from src.models.config import resolve_model
from src.ops import hybrid as hops
from tests import kafunex_oracle as O
from tests import kafunex_utils as U

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = dict(atol=2e-4, rtol=2e-4)


@pytest.fixture(scope="module", params=sorted(U.MODELS))
def model(request, tmp_path_factory):
    cfg = U.MODELS[request.param]
    w = U.tensors(cfg, seed=3, gain=1.5)
    return cfg, w, U.write(tmp_path_factory.mktemp(request.param), cfg, w)


def ref(cfg, w, ids):
    return O.forward(cfg, w, ids).float()


# ------------------------------------------------------------------ configuration and weights
def test_registry_reads_every_size(tmp_path):
    cfg = U.MODELS["mixed"]
    c = resolve_model(U.write(tmp_path, cfg, U.tensors(cfg)))
    assert (c.model_type, c.hybrid, c.num_hidden_layers) == ("kafunex", True, 5)
    assert (c.vocab_size, c.hidden_size, c.rms_norm_eps) == (157, 72, 1e-5)
    for sp, e in zip(c.layers, cfg["layers"]):
        m = e["mixer"]
        assert (sp.mixer, sp.heads, sp.dim, sp.vdim, sp.ff) == (e["type"], m["heads"], m["dim"], m["vdim"],
                                                                e["mlp"]["ff"])
        if e["type"] == "attention":
            assert (sp.kv_heads, sp.chunk, sp.scale) == (m["kv_heads"], m["mask"]["size"], m["scale"])
    assert c.layer_param_bytes(1.0) * 5 > 0 and c.kv_bytes_per_token_per_layer() > 0
    assert type(c).from_hf_dict(json.loads(json.dumps(cfg))).layers == c.layers


@pytest.mark.parametrize("change,match", [
    (lambda c: c.update(architecture="Nobody"), "unknown architecture"),
    (lambda c: c["layers"][0].update(type="other"), "unsupported mixer"),
    (lambda c: c["layers"][1]["mixer"].update(kv_heads=3), "multiple of kv_heads"),
    (lambda c: c["layers"][1]["mixer"].update(vdim=8), "vdim must equal dim"),
    (lambda c: c["layers"][0]["mlp"].update(kind="moe"), "feed-forward kind")])
def test_bad_configurations_are_refused(tmp_path, change, match):
    cfg = json.loads(json.dumps(U.MODELS["mixed"]))
    change(cfg)
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    with pytest.raises(ValueError, match=match):
        resolve_model(str(tmp_path))


def test_wrong_tensor_shape_is_refused(tmp_path):
    cfg = U.MODELS["no_mlp"]
    w = U.tensors(cfg)
    w["l0.mix.k"] = w["l0.mix.k"][:-1].contiguous()
    with pytest.raises(ValueError, match="mix.k"):
        U.executor(U.write(tmp_path, cfg, w), "cpu", "fp32")


def test_offload_and_tensor_split_are_refused(model):
    from src.parallel.tensor_parallel import check_tp

    with pytest.raises(ValueError, match="resident"):
        U.executor(model[2], "cpu", "fp32", offload=True)
    with pytest.raises(ValueError, match="tensor parallelism"):
        check_tp(resolve_model(model[2]), 2)


def test_block_sizes_count_the_recurrent_state():
    from src.block_utils import auto_num_blocks
    from src.partition import balanced_splits, stage_cost_model

    c = resolve_model("kafunex-7b")
    state = c.state_bytes_per_session_per_layer()
    assert state == 32 * 128 * 128 * 4 * 3 // 4
    lots, none = (auto_num_blocks(c, 20 << 30, max_sessions=n) for n in (2048, 0))
    assert lots < none
    assert stage_cost_model(c, batch=64)[0] > stage_cost_model(c, batch=1)[0]
    assert len(balanced_splits(c, 4)) == 3


def test_preset_runs_with_random_weights():
    ex = U.executor("tiny-kafunex", "cpu", "fp32")
    assert torch.isfinite(ex.forward([("a", 50)], U.ids(50, 640))).all()


# ------------------------------------------------------------------ mechanisms
def test_embedding_and_positions():
    W, T = 30, 5
    table = torch.randn(9, W)
    pos = torch.tensor([0, 1, 2, 40000, 7])
    res, xb = torch.empty(T, W), torch.empty(T, W)
    ids = torch.tensor([0, 8, 3, 3, 1])
    hops.embed_pos(ids, table, pos, hops.position_frequencies(W, "cpu"), res, xb)
    want = torch.cat([O.sinusoid(1, W, start=int(p)) for p in pos]).float() + table[ids]
    torch.testing.assert_close(res, want, atol=1e-6, rtol=1e-6)
    assert torch.equal(res, xb)
    assert float(res[0, 1] - table[0, 1]) == pytest.approx(1.0, abs=1e-6) and float(res[0, 0] - table[0, 0]) == 0.0


def test_norms_and_activation():
    y, res, w = torch.randn(4, 20), torch.randn(4, 20), torch.randn(20)
    want = res.double() + O.rms(y.double(), 1e-2) * w.double()
    got = res.clone()
    hops.residual_norm(y, got, w, 1e-2, torch.empty(4, 20))
    torch.testing.assert_close(got, want.float(), **TOL)
    out = hops.rows_norm(res, torch.tensor([2, 0], dtype=torch.int32), w, 1e-2, torch.empty(2, 20))
    torch.testing.assert_close(out, (O.rms(res.double(), 1e-2) * w.double())[[2, 0]].float(), **TOL)
    torch.testing.assert_close(hops.relu2(y, torch.empty(4, 20)), y.clamp(min=0) ** 2)


def test_recurrence_alone_and_its_state():
    H, D, V, L = 3, 5, 7, 19
    g = torch.Generator().manual_seed(0)
    z = torch.randn(L, H * (2 * D + V), generator=g)
    b, lo, nw = torch.randn(H * D, generator=g), torch.rand(H * D, generator=g), torch.randn(V, generator=g)
    zq, zf, v = z.double().split([H * D, H * D, H * V], 1)
    q = (zq * torch.sigmoid(zq)).view(L, H, D)
    f = O.forget_gate(zf, b.double(), lo.double()).view(L, H, D)
    o, S = O.hgrn2_scan(q, f, v.view(L, H, V))
    want = (O.rms(o, 1e-3) * nw.double()).reshape(L, -1)
    state = torch.full((2, H, D, V), 1e9)  # what a slot's last user left
    ctx = torch.arange(1, L + 1, dtype=torch.int32)
    got = hops.hgrn2(z, b, lo, nw, state, torch.ones(L, dtype=torch.int32), ctx, torch.empty(L, H * V), 1e-3)
    torch.testing.assert_close(got, want.float(), **TOL)
    torch.testing.assert_close(state[1], S.float(), **TOL)
    assert (state[0] == 1e9).all()


def attention_case(L, H, G, D, chunk, scale, seed=0, spikes=()):
    """Projected rows, weights and the oracle's core output; ``spikes``: (query, key) pairs made to stand out."""
    g = torch.Generator().manual_seed(seed)
    q, k = torch.randn(L, H * D, generator=g), torch.randn(L, G * D, generator=g)
    for i, j in spikes:  # one query and one key share a direction no other token has much of
        d = torch.sign(torch.randn(D, generator=g))
        q[i] = q[i] * 0.1 + 3 * d.repeat(H)
        k[j] = k[j] * 0.1 + 3 * d.repeat(G)
    gate = torch.randn(L, H * D, generator=g)
    wq, wk = 1 + 0.3 * torch.randn(H * D, generator=g), 1 + 0.3 * torch.randn(G * D, generator=g)
    talk = (torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)).bfloat16().float()
    return q, k, gate, wq, wk, talk


def attention_oracle(q, k, gate, wq, wk, talk, H, G, D, chunk, scale, eps):
    dd = torch.float64
    L = q.shape[0]
    qn = O.rms(q.to(dd), eps) * wq.to(dd)
    kn = O.rms(k.to(dd), eps) * wk.to(dd)
    o = O.attention_core(qn.view(L, H, D), kn.view(L, G, D), k.to(dd).view(L, G, D), scale, talk.to(dd), chunk)
    return (o.reshape(L, H * D) * torch.sigmoid(gate.to(dd))).float()


def attention_product(q, k, gate, wq, wk, talk, H, G, D, chunk, scale, eps, page=8, rows=None, order=None):
    """The ops on a paged cache: ``order`` permutes the page ids, ``rows`` limits the queries that are asked for."""
    L = q.shape[0]
    n = (L + page - 1) // page
    pages = torch.arange(n) if order is None else order
    cache, rk = torch.full((n + 2, G, page, D), 7.0), torch.full((n + 2, page), 9.0)
    table = torch.full((2, n), -1, dtype=torch.int32)
    table[1] = pages.int()
    pos = torch.arange(L)
    slots = pages[pos // page] * page + pos % page
    z = torch.cat([q, k, gate], 1)
    wqk = wq * wk.view(G, 1, D).expand(G, H // G, D).reshape(-1)
    qn = torch.empty(L, H * D)
    hops.talk_prep(z, wqk, qn, cache, rk, slots, eps)
    r = torch.arange(L) if rows is None else torch.tensor(rows)
    return hops.talk_attention(z[r], qn[r], talk, cache, rk, table, torch.ones(len(r), dtype=torch.int32),
                               (r + 1).int(), torch.empty(len(r), H * D), chunk, scale)


@pytest.mark.parametrize("L,H,G,D,chunk,scale", [(40, 4, 2, 8, 13, 0.3), (9, 1, 1, 4, 1, 1.0), (33, 6, 3, 5, 8, 0.2),
                                                 (33, 3, 1, 8, 64, 0.5), (17, 4, 4, 8, 16, 0.25)])
def test_attention_alone(L, H, G, D, chunk, scale):
    a = attention_case(L, H, G, D, chunk, scale)
    want = attention_oracle(*a, H, G, D, chunk, scale, 1e-4)
    order = torch.randperm((L + 7) // 8 + 2, generator=torch.Generator().manual_seed(1))[: (L + 7) // 8]
    torch.testing.assert_close(attention_product(*a, H, G, D, chunk, scale, 1e-4, order=order), want, **TOL)


@pytest.mark.parametrize("i,j,seen", [(12, 0, True), (13, 13, True), (13, 12, False), (25, 13, True), (26, 25, False),
                                      (26, 0, False), (38, 26, True), (39, 38, False), (15, 15, True), (16, 13, True)])
def test_a_standing_out_key_at_a_chunk_edge(i, j, seen):
    """Chunks of 13, pages of 8: the key is found exactly when it lies in the query's chunk."""
    H, G, D, chunk, scale = 4, 2, 8, 13, 1.0
    a = list(attention_case(40, H, G, D, chunk, scale, spikes=[(i, j)]))
    a[5] = torch.eye(H)
    want = attention_oracle(*a, H, G, D, chunk, scale, 1e-6)
    got = attention_product(*a, H, G, D, chunk, scale, 1e-6, rows=[i])
    torch.testing.assert_close(got[0], want[i], **TOL)
    b = list(a)
    b[1] = a[1].clone()
    b[1][j] = -b[1][j]
    moved = (attention_product(*b, H, G, D, chunk, scale, 1e-6, rows=[i])[0] - got[0]).abs().max()
    assert (moved > 0.3) == seen
    off = attention_oracle(*a, H, G, D, chunk + 1, scale, 1e-6)  # an oracle one token off must show
    if not seen and j == i - i % chunk - 1 and j // (chunk + 1) == i // (chunk + 1):
        assert (off[i] - want[i]).abs().max() > 0.3


def test_mixed_slopes():
    talk = torch.randn(6, 6)
    torch.testing.assert_close(hops.talk_sigma(talk), (talk.double() @ O.slopes(6)).float(), **TOL)


def test_recurrent_plan_covers_every_token():
    for ntoks in ([1], [5, 0, 1000, 1, 17], [128] * 9, [4000], [129, 191, 193, 300]):
        for heads in (1, 4, 32):
            p = hops.hgrn2_plan(ntoks, heads, seg_tokens=128)
            seg = p["seg"].T.tolist()
            got = sorted(t for o, n, _, _ in seg for t in range(o, o + n))
            assert got == list(range(sum(ntoks)))
            slots = sorted(s for *_, s, _ in seg if s >= 0)
            assert slots == list(range(p["slots"])) and all(n > 0 for _, n, _, _ in seg)
            for first, k, tok0, _ in p["multi"].T.tolist():
                chain = sorted(s for s in seg if first <= s[2] < first + k)
                assert chain[0][0] == tok0 and chain[-1][3] == -1
                assert [c[3] for c in chain[:-1]] == [c[2] for c in chain[1:]]
                assert all(c[1] % 16 == 0 for c in chain[:-1])


def _round_cost(plan, room):
    """Tokens that the rounds of a plan's segments last for, each with its start."""
    n = [n for _, n, _, _ in plan["seg"].T.tolist()]
    return -(-len(n) // room) * (max(n) + hops.SEG_START) if n else 0


@pytest.mark.parametrize("ntoks", [[1], [5, 0, 1000, 1, 17], [128] * 9, [4000], [1801, 750, 1400, 349], [0, 0], [8192], [40] * 100,
                                   [300, 2000], [700] * 5, [129, 4100, 900], [64] * 30 + [2000]])
def test_recurrent_plan_fits_its_rounds(ntoks):
    """Without a length given: every token once, whole blocks, and rounds within a tenth of what the best of all lengths gives."""
    for heads, per_cu in ((1, 2), (16, 1), (16, 2), (32, 2), (600, 1)):
        p, room = hops.hgrn2_plan(ntoks, heads, per_cu=per_cu), max(1, per_cu * 256 // heads)
        seg = p["seg"].T.tolist()
        assert sorted(t for o, n, _, _ in seg for t in range(o, o + n)) == list(range(sum(ntoks)))
        assert all(n % 16 == 0 for _, n, _, d in seg if d >= 0)
        if room > 1 and seg:  # (more heads than workgroups at once: no round is shared)
            every = [hops.hgrn2_plan(ntoks, heads, seg_tokens=T) for T in range(128, max(ntoks) + 144, 16)]
            assert _round_cost(p, room) <= 1.1 * min(_round_cost(q, room) for q in every)


def test_recurrent_plan_of_a_ragged_step():
    """Where 16 segments run at once, 18 or 35 of them would take a round more."""
    for heads, per_cu in ((16, 1), (32, 2)):
        assert hops.hgrn2_plan([1801, 750, 1400, 349], heads, per_cu=per_cu)["seg"].shape[1] <= 16


# ------------------------------------------------------------------ executor
def test_whole_prompts(model):
    cfg, w, d = model
    ex = U.executor(d, "cpu", "fp32")
    for n in (1, 2, 3, 64, 65, 130):
        t = U.ids(n, cfg["vocab"], n)
        got = ex.forward([("a", n)], t, reset=[True], logit_rows=range(n))
        torch.testing.assert_close(got, ref(cfg, w, t), **TOL)


def test_prefill_equals_decoding_and_portions(model):
    cfg, w, d = model
    n = 90
    t = U.ids(n, cfg["vocab"])
    want = ref(cfg, w, t)
    ex = U.executor(d, "cpu", "fp32")
    for name, sizes in (("decode", [1] * n), ("pairs", [2] * (n // 2)), ("odd", [2, 3, 5, 7, 11, 13, 17, 19, 2, 11]),
                        ("head", [67, 1, 1, 2, 19])):
        assert sum(sizes) == n
        at, got = 0, []
        for k in sizes:
            got.append(ex.forward([(name, k)], t[at:at + k], logit_rows=range(k)))
            at += k
        torch.testing.assert_close(torch.cat(got), want, **TOL)
        ex.sessions.close(name)


def test_unequal_batches_equal_each_alone(model):
    cfg, w, d = model
    ex = U.executor(d, "cpu", "fp32")
    lens = {"a": 70, "b": 3, "c": 41, "d": 1}
    toks = {k: U.ids(n + 12, cfg["vocab"], n) for k, n in lens.items()}
    at = {k: 0 for k in lens}
    steps = [{"a": 30, "b": 2}, {"a": 1, "c": 20, "b": 1}, {"d": 1, "c": 21, "a": 39}, {"a": 1, "b": 1, "c": 1, "d": 1},
             {"d": 1, "b": 1}, {"c": 2, "a": 1}, {"b": 1, "d": 5}]
    for s in steps:
        x = torch.cat([toks[k][at[k]:at[k] + n] for k, n in s.items()])
        got = ex.forward(list(s.items()), x)
        for r, (k, n) in enumerate(s.items()):
            at[k] += n
            torch.testing.assert_close(got[r], ref(cfg, w, toks[k][:at[k]])[-1], **TOL)


def test_pages_and_slots_are_used_again(model):
    cfg, w, d = model
    ex = U.executor(d, "cpu", "fp32", max_sessions=2, num_pages=3, page_size=64)
    for k in range(5):
        t = U.ids(100 + k, cfg["vocab"], k)
        got = ex.forward([(f"s{k}", t.numel())], t)
        torch.testing.assert_close(got[0], ref(cfg, w, t)[-1], **TOL)
        u = U.ids(30, cfg["vocab"], 50 + k)
        torch.testing.assert_close(ex.forward([(f"u{k}", 30)], u)[0], ref(cfg, w, u)[-1], **TOL)
        with pytest.raises(Exception):
            ex.forward([(f"x{k}", 1)], t[:1])  # no third slot
        ex.sessions.close(f"s{k}")
        ex.sessions.close(f"u{k}")
        for s in ([] if ex.state is None else ex.state.states) + ex.cache.rows + ex.cache.rk:
            s.fill_(1e6)  # whatever is left there must not be read
    assert ex.sessions.free_pages == 3


def test_long_decoding(model):
    cfg, w, d = model
    n = 260
    t = U.ids(n, cfg["vocab"], 9)
    ex = U.executor(d, "cpu", "fp32")
    ex.forward([("a", 10)], t[:10])
    got = torch.cat([ex.forward([("a", 1)], t[i:i + 1]) for i in range(10, n)])
    torch.testing.assert_close(got, ref(cfg, w, t)[10:], **TOL)


def test_chunked_prefill_of_a_long_step(model):
    cfg, w, d = model
    t = U.ids(150, cfg["vocab"], 4)
    ex = U.executor(d, "cpu", "fp32", max_tokens_per_step=37)
    got = ex.forward([("a", 120), ("b", 30)], t)
    torch.testing.assert_close(got[0], ref(cfg, w, t[:120])[-1], **TOL)
    torch.testing.assert_close(got[1], ref(cfg, w, t[120:])[-1], **TOL)


def test_stage_split_equals_full(model):
    cfg, w, d = model
    L = len(cfg["layers"])
    s0 = U.executor(d, "cpu", "bf16", role="stage0", end=1)
    s1 = U.executor(d, "cpu", "bf16", role="segment", start=1, end=2)
    s2 = U.executor(d, "cpu", "bf16", role="last", start=2, end=L)
    full = U.executor(d, "cpu", "bf16")
    t = U.ids(40, cfg["vocab"])
    h = s0.forward([("a", 40)], t)
    assert h.dtype == torch.float32 == s0.hidden_dtype  # the stream between stages stays 32-bit
    torch.testing.assert_close(s2.forward([("a", 40)], s1.forward([("a", 40)], h)), full.forward([("a", 40)], t))


def test_fork_and_rewind(model):
    cfg, w, d = model
    ex = U.executor(d, "cpu", "fp32")
    t = U.ids(30, cfg["vocab"])
    ex.forward([("a", 25)], t[:25])
    ex.sessions.fork("a", "b")
    ex.forward([("a", 3)], t[:3])
    torch.testing.assert_close(ex.forward([("b", 5)], t[25:])[0], ref(cfg, w, t)[-1], **TOL)
    if ex.state is not None:
        with pytest.raises(ValueError, match="rewound"):
            ex.forward([("b", 1)], t[:1], starts=[10])
    got = ex.forward([("b", 30)], t, starts=[0])  # from the first token it can always start over
    torch.testing.assert_close(got[0], ref(cfg, w, t)[-1], **TOL)


def test_bf16_path_is_close(model):
    cfg, w, d = model
    t = U.ids(120, cfg["vocab"], 2)
    want = ref(cfg, w, t)
    got = U.executor(d, "cpu", "bf16").forward([("a", 120)], t, logit_rows=range(120)).float()
    err = (got - want).pow(2).mean(-1).sqrt() / want.std()
    # (a head of one value is normed to its sign, which rounding can flip: not every position can be close)
    assert err.quantile(0.95) < 0.1


# ------------------------------------------------------------------ scheduler, sampling, command line
def serve(ex, reqs, **kw):
    from src.parallel.engine import PipelineServingEngine, Request
    from src.runtime.sampler import SamplingParams

    eng = PipelineServingEngine(ex, None, **kw)
    rs = [eng.submit(Request(prompt=p, max_new_tokens=n, params=SamplingParams(0.0, 1.0, 0, 1.0), seed=i, rid=f"r{i}",
                             eos_token_id=None, stop_on_repeat=0)) for i, (p, n) in enumerate(reqs)]
    eng.run_until_idle(max_rounds=800)
    return [list(r.generated) for r in rs]


def test_greedy_generation_through_the_scheduler(model):
    cfg, w, d = model
    reqs = [(U.ids(n, cfg["vocab"], n).tolist(), 7 + n % 3) for n in (1, 2, 9, 40, 71, 5, 18)]
    want = [O.greedy(cfg, w, torch.tensor(p), n) for p, n in reqs]
    ex = U.executor(d, "cpu", "fp32")
    assert serve(ex, reqs, batch=3, n_slots=2) == want
    assert serve(ex, reqs, batch=6, prefill_chunk=4, max_step_tokens=11) == want
    assert not ex.sessions.sessions


def test_trace_run_program(model, tmp_path):
    cfg, w, d = model
    a, b = U.ids(20, cfg["vocab"], 1), U.ids(9, cfg["vocab"], 2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:11].tolist(), "want": [0, 10]}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": b[:8].tolist(), "want": []},
                                     {"id": "a", "tokens": a[11:12].tolist(), "want": [0]}], "end": []},
             {"step": 2, "entries": [{"id": "b", "tokens": b[8:].tolist(), "want": []}], "end": ["b"]},
             {"step": 3, "entries": [{"id": "a", "tokens": a[12:].tolist(), "want": [7, 2]},
                                     {"id": "c", "tokens": b.tolist(), "want": [8]}], "end": ["a", "c"]}]
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", d, "--dtype", "float32", "--out",
                        str(tmp_path), "--max-tokens", "128", "--device", "cpu"], text=True, capture_output=True,
                       input="".join(json.dumps(s) + "\n" for s in steps), timeout=240)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [ln for ln in r.stdout.splitlines() if ln.startswith("done")] == [f"done {k}" for k in range(4)]
    A, B = ref(cfg, w, a), ref(cfg, w, b)
    want = {0: A[[0, 10]], 1: A[[11]], 3: torch.stack([A[19], A[14], B[8]])}
    assert sorted(os.listdir(tmp_path)) == [f"{k}.f32" for k in sorted(want)]
    for k, y in want.items():
        got = torch.from_numpy(np.fromfile(tmp_path / f"{k}.f32", "<f4").reshape(-1, cfg["vocab"]))
        torch.testing.assert_close(got, y, **TOL)


def test_cli_generates(tmp_path):
    """Client (stage 0) and tail server from ``python -m src.main`` over TCP, greedy, against the oracle."""
    from tests.test_engine_gloo import _free_port

    cfg = U.config([U.rec(), U.att(), U.rec(2, 8, 8)], vocab=300)
    w = U.tensors(cfg, seed=8)
    d = U.write(tmp_path / "m", cfg, w)
    reg, p1, p0, pr = (_free_port() for _ in range(4))
    env = dict(os.environ, OMP_NUM_THREADS="1")
    common = [sys.executable, "-m", "src.main", "--model", d, "--splits", "2", "--dtype", "fp32", "--device", "cpu",
              "--host", "127.0.0.1", "--device_channel", "off", "--max_seq_len", "128", "--max_sessions", "4",
              "--temperature", "0", "--kv_cache_gb", "0.05"]
    srv = subprocess.Popen(common + ["--stage", "1", "--dht_port", str(reg), "--rpc_port", str(p1)], cwd=ROOT, env=env,
                           stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    try:
        r = subprocess.run(common + ["--stage", "0", "--dht_port", str(p0), "--rpc_port", str(pr),
                                     "--dht_initial_peers", f"127.0.0.1:{reg}", "--max_new_tokens", "6", "--prompt",
                                     "hello there"], cwd=ROOT, env=env, capture_output=True, text=True, timeout=150)
        assert r.returncode == 0, r.stderr[-3000:]
    finally:
        srv.kill()
        srv.wait()
    from src.models.tokenizer import load_tokenizer

    tok = load_tokenizer(d, resolve_model(d))
    want = O.greedy(cfg, w, torch.tensor(tok(("hello there")).input_ids[0]), 6)
    if tok.eos_token_id in want:
        want = want[:want.index(tok.eos_token_id)]
    assert f"GENERATED: {tok.decode(want, skip_special_tokens=True)}" in r.stdout
