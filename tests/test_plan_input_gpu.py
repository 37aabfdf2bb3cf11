"""Staging of a ragged step's plan (``executor._PlanInput``): steps in flight, buffers that are too small, the block table."""
import numpy as np
import pytest
import torch

from src import native, ops
from src.models.config import resolve_model
from src.models.weights import random_stage_weights
from src.runtime import executor

pytestmark = pytest.mark.gpu


def _stage(name, **kw):
    cfg = resolve_model(name)
    w = random_stage_weights(cfg, 0, cfg.num_hidden_layers, has_embed=True, has_head=True, device="cuda:0", seed=3)
    return executor.StageExecutor(cfg, w, "cuda:0", max_sessions=12, max_seq_len=512, kv_cache_bytes=256 << 20, warmup=False, **kw)


def _steps(ex, wait):
    g, outs = torch.Generator().manual_seed(1), []
    for i in range(14):  # (more than a ring's turns; every second step goes on with sessions that are there)
        n = [1 + int(x) for x in torch.randint(0, 90, (1 + i % 5,), generator=g)]
        ids = torch.randint(0, 500, (sum(n),), generator=g).cuda()
        outs.append(ex.forward([(f"s{j}", k) for j, k in enumerate(n)], ids, reset=[i % 2 == 0] * len(n)).clone())
        if wait:
            torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("name", ["small-llama", "tiny-kafunex", "tiny-fubapel", "tiny-nuvorax", "tiny-debuzen"])
def test_steps_in_flight(name, monkeypatch):
    """The same logits, to the last bit, of steps that follow each other at once, of steps that are waited for, and where most arrays
    do not fit the step's buffer."""
    ops.require_native()
    want = _steps(_stage(name), True)
    for a, b in zip(_steps(_stage(name), False), want):
        assert torch.equal(a, b)
    real = executor._PlanInput.room
    monkeypatch.setattr(executor._PlanInput, "room", lambda self, shape, dtype:
                        None if self._at and len(shape) > 1 and shape[1] % 2 == 0 else real(self, shape, dtype))
    for a, b in zip(_steps(_stage(name), False), want):
        assert torch.equal(a, b)


def test_a_full_buffer_grows():
    ops.require_native()
    inp = executor._PlanInput(torch.device("cuda:0"), 4096)
    ex = _stage("small-llama")
    big = np.arange(3000, dtype=np.int32)
    inp.open(4096)
    a, b = inp.put(np.arange(5, dtype=np.int64)), inp.put(big)
    inp.close(ex.sessions)
    assert torch.equal(a.cpu(), torch.arange(5)) and torch.equal(b.cpu(), torch.from_numpy(big))
    inp.open(4096)
    c, d = inp.put(np.arange(7, dtype=np.int64)), inp.put(big[::2])
    inp.close(ex.sessions)
    assert inp.size > 4096 and d.data_ptr() == c.data_ptr() + 64  # (fits now, at the next 16 bytes)
    assert torch.equal(c.cpu(), torch.arange(7)) and torch.equal(d.cpu(), torch.from_numpy(big[::2].copy()))


def test_plan_on_the_device():
    """What the step's kernels read: positions, slots and sequences as the host made them, and the block table that they use."""
    ops.require_native()
    ex = _stage("small-llama")
    for n in ([5, 300, 64], [40, 1]):
        seqs = [(f"s{j}", k) for j, k in enumerate(n)]
        p = ex.plan(seqs)
        T, S = sum(n), len(n)
        n64, n32 = np.empty((2, T), np.int64), np.empty(2 * T + S, np.int32)
        rows = np.array([s.row for s in p.sessions], np.int32)
        native.build_meta(rows, p.starts, p.ntoks, ex.sessions.table, ex.cache.page_size, n64[0], n64[1], n32[:T], n32[T:2 * T], n32[2 * T:])
        assert np.array_equal(p.meta_i64.cpu().numpy(), n64) and np.array_equal(p.meta_i32.cpu().numpy(), n32)
        assert np.array_equal(ex.sessions.table_dev.cpu().numpy(), ex.sessions.table) and not ex.sessions._dirty
        fb, waves = ops.fa_plan(p.ntoks, ex.nh, ex.nkv, ex._n_cu)
        assert np.array_equal(p.fablocks.cpu().numpy(), fb) and p.fa_waves == waves
        assert (p.qblocks is None) == (T > ops.wide_rows())
        ex.commit(p)


def test_tables_of_an_odd_number_of_words(monkeypatch):
    """5 sessions of 5 pages: the table arrives with the plan, in a buffer that stays as it is."""
    ops.require_native()
    cfg = resolve_model("small-llama")
    w = random_stage_weights(cfg, 0, 1, has_embed=True, has_head=False, device="cuda:0", seed=3)
    ex = executor.StageExecutor(cfg, w, "cuda:0", max_sessions=5, max_seq_len=320, kv_cache_bytes=16 << 20, warmup=False)
    assert ex.sessions.table.size == 25
    copies, sync = [], ex.sessions.sync_table
    monkeypatch.setattr(ex.sessions, "sync_table", lambda: copies.append(1) or sync())
    size, at = ex._input.size, ex._input._host.data_ptr()
    for i in range(200):
        sid = f"s{i % 5}"
        ex.forward([(sid, 2 + i)], torch.zeros(2 + i, dtype=torch.long, device="cuda"), reset=[True])
        if i % 40 == 39:
            assert np.array_equal(ex.sessions.table_dev.cpu().numpy(), ex.sessions.table)
    assert ex._input.size == size and ex._input._host.data_ptr() == at and not copies
