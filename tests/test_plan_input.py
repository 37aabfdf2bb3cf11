"""The buffer that a ragged step's plan arrives in (``executor._PlanInput``), its launch played by the host."""
import types

import numpy as np
import pytest
import torch

from src.runtime import executor
from src.runtime.kv_cache import PageAllocator
from src.runtime.session import SessionManager


def _sessions(rows, pages, page=4):
    cache = types.SimpleNamespace(device=torch.device("cpu"), page_size=page, allocator=PageAllocator(rows * pages))
    return SessionManager(cache, max_sessions=rows, max_seq_len=pages * page)


@pytest.fixture
def launches(monkeypatch):
    seen = []

    def plan_input(host, meta, table):
        seen.append(host.numel())
        assert host.numel() % 8 == 0 and host.numel() == meta.numel() + (0 if table is None else 4 * table.numel())
        meta.copy_(host[:meta.numel()])
        if table is not None:
            table.view(-1).copy_(host[meta.numel():].view(torch.int32))

    monkeypatch.setattr(executor, "torch", types.SimpleNamespace(
        empty=lambda *a, pin_memory=False, **kw: torch.empty(*a, **kw), uint8=torch.uint8, from_numpy=torch.from_numpy,
        ops=types.SimpleNamespace(mpamd=types.SimpleNamespace(plan_input=plan_input)),
        cuda=types.SimpleNamespace(Event=lambda: types.SimpleNamespace(record=lambda: None, synchronize=lambda: None))))
    return seen


def _step(inp, sessions, sid, tokens):
    """A prompt: its session anew, two arrays of ``tokens``."""
    s = sessions.open(sid)
    sessions.reset(sid)
    sessions.reserve(s, min(tokens, s.max_length))
    inp.open(24 * tokens + 4 + sessions.table.nbytes + 256)
    a, b = np.arange(2 * tokens, dtype=np.int64), np.arange(2 * tokens + 1, dtype=np.int32)
    got = inp.put(a), inp.put(b)
    inp.close(sessions)
    assert np.array_equal(got[0].numpy(), a) and np.array_equal(got[1].numpy(), b)
    assert np.array_equal(sessions.table_dev.numpy(), sessions.table) and not sessions._dirty


# tables of an odd number of words and of an even one
@pytest.mark.parametrize("rows,pages", [(5, 5), (1, 125), (255, 65), (256, 65), (5, 6)])
def test_a_buffer_of_any_table_keeps_its_size(rows, pages, launches):
    sessions = _sessions(rows, pages)
    inp = executor._PlanInput(torch.device("cpu"), 24 * 40 + 4 + sessions.table.nbytes + 256)
    size, host = inp.size, inp._host.data_ptr()
    for i in range(200):
        _step(inp, sessions, f"s{i % rows}", 1 + i % 40)
    assert len(launches) == 200 and inp.size == size and inp._host.data_ptr() == host


def test_a_buffer_grows_to_the_largest_step(launches):
    """What did not fit once fits from then on, and steps that come after it ask for no more."""
    sessions = _sessions(5, 5)
    inp = executor._PlanInput(torch.device("cpu"), 4096)
    sizes = []
    for i in range(60):
        inp.open(4096)
        arrays = [np.arange(n, dtype=np.int32) for n in (100, 1500 + i % 7, 300)]
        got = [inp.put(a) for a in arrays]
        inp.close(sessions)
        assert all(np.array_equal(g.numpy(), a) for g, a in zip(got, arrays))
        sizes.append(inp.size)
    assert sizes[0] == 4096 and sizes[-1] == sizes[8] <= 12288


def test_a_table_that_was_not_sent_is_sent_later(launches, monkeypatch):
    """A launch that raises leaves the device's table old: the next step brings it."""
    sessions = _sessions(5, 6)
    inp = executor._PlanInput(torch.device("cpu"), 4096)
    real = executor.torch.ops.mpamd.plan_input

    def fails(*a):
        raise RuntimeError("no launch")

    monkeypatch.setattr(executor.torch.ops.mpamd, "plan_input", fails)
    with pytest.raises(RuntimeError, match="no launch"):
        _step(inp, sessions, "a", 9)
    assert not np.array_equal(sessions.table_dev.numpy(), sessions.table)
    monkeypatch.setattr(executor.torch.ops.mpamd, "plan_input", real)
    inp.open(4096)
    inp.put(np.arange(3, dtype=np.int64))
    inp.close(sessions)
    assert np.array_equal(sessions.table_dev.numpy(), sessions.table) and not sessions._dirty
