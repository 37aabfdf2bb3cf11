"""Sampler semantics (reference src/rpc_handler.py:327-403) on the CPU path."""
import pytest
import torch

from src import ops
from src.ops import reference as ref
from src.runtime.sampler import BatchSampler, SamplingParams, session_seed


def test_greedy_and_penalty():
    lg = torch.zeros(10)
    lg[3], lg[4] = 5.0, 4.9
    assert ref.sample_row(lg, 0.0, 0.9, 0) == 3
    # token 3 repeated 3x: rp**3 then last-3 strong penalty rp**3 -> token 4 wins under top_k=1
    assert ref.sample_row(lg, 1.0, 1.0, 1, 1.5, [3, 3, 3]) == 4
    # negative logits are multiplied by the penalty
    lg2 = torch.full((5,), -1.0)
    lg2[0] = -0.5
    assert ref.sample_row(lg2, 1.0, 1.0, 1, 2.0, [0]) != 0


def test_top_p_keeps_first_and_cum_le_p():
    lg = torch.log(torch.tensor([0.5, 0.3, 0.15, 0.05]))
    g = torch.Generator().manual_seed(0)
    seen = {ref.sample_row(lg, 1.0, 0.6, 0, 1.0, [], generator=g) for _ in range(200)}
    assert seen == {0}  # cum: 0.5 <= 0.6 kept, 0.8 > 0.6 dropped
    seen = {ref.sample_row(lg, 1.0, 0.85, 0, 1.0, [], generator=g) for _ in range(400)}
    assert seen == {0, 1}
    seen = {ref.sample_row(lg, 1.0, 0.1, 0, 1.0, [], generator=g) for _ in range(50)}
    assert seen == {0}  # first token always kept


def test_batch_sampler_cpu():
    s = BatchSampler("cpu")
    lg = torch.randn(3, 50)
    out = s(lg, [SamplingParams(0.0, 0.9, 0, 1.0)] * 3, [[], [], []], [1, 2, 3])
    assert torch.equal(out, torch.argmax(lg, -1))
    out = s(lg, [SamplingParams(1.0, 0.9, 5, 1.5)] * 3, [[1], [2, 2], []], [session_seed("a", 1)] * 3)
    assert out.shape == (3,) and int(out.max()) < 50


def _batch(n, V, seed):
    g = torch.Generator().manual_seed(seed)
    hist = [torch.randint(0, V, (k % 70,), generator=g).tolist() for k in range(n)]
    par = [SamplingParams(0.5 + 0.1 * (k % 9), 0.8 + 0.01 * (k % 20), (0, 50, 7)[k % 3], 1.0 + 0.1 * (k % 5)) for k in range(n)]
    return (3 * torch.randn(n, V, generator=g)).bfloat16(), par, hist, torch.randint(0, 1 << 62, (n,), generator=g).tolist()


def _one_by_one(lg, par, hist, seeds):
    """What a row gets when its parameters come as tensors of their own."""
    from src import ops

    rec = torch.zeros(len(par), 50, dtype=torch.int32)
    for r, h in enumerate(hist):
        h = h[-50:]
        rec[r, :len(h)] = torch.tensor(h, dtype=torch.int32)
    t = lambda v, dt: torch.tensor(v, dtype=dt, device=lg.device)  # noqa: E731
    return ops.sample(lg, t([p.temperature for p in par], torch.float32), t([p.top_p for p in par], torch.float32),
                      t([p.top_k for p in par], torch.int32), t([p.repetition_penalty for p in par], torch.float32),
                      rec.to(lg.device), t([min(len(h), 50) for h in hist], torch.int32), t(seeds, torch.int64))


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_batch_sampler_calls_in_flight(dev):
    """Calls that are not waited for keep their own rows' parameters, histories and seeds, of any number of rows."""
    s = BatchSampler(dev, max_rows=24)
    steps = [_batch(n, 700, k) for k, n in enumerate((24, 1, 7, 24, 60, 3, 24, 2))]
    lgs = [lg.to(dev) for lg, *_ in steps]
    if dev == "cuda":  # (the device has not begun with the first call when the second buffer is filled)
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
    got = [s(lg, *rest) for lg, (_, *rest) in zip(lgs, steps)]
    for lg, g, (_, *rest) in zip(lgs, got, steps):
        assert torch.equal(g.cpu(), torch.cat([_one_by_one(lg[i:i + 24], *[r[i:i + 24] for r in rest])
                                               for i in range(0, len(g), 24)]).cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("V", [32000, 50000, 70000])
def test_batch_sampler_on_several_streams(V, monkeypatch):
    """Rows in LDS, in the workspace and in its records: the workspace is one for all streams, so that a call waits for the one
    before it.  Each call has its own logits, parameters, histories and seeds."""
    s = BatchSampler("cuda", max_rows=48)
    steps = [_batch(n, V, k) for k, n in enumerate((48, 31, 48, 48, 7, 48))]
    lgs = [lg.cuda() for lg, *_ in steps]
    want = [_one_by_one(lg, *rest) for lg, (_, *rest) in zip(lgs, steps)]
    torch.cuda.synchronize()
    waited, wait = [], torch.cuda.Stream.wait_event
    monkeypatch.setattr(torch.cuda.Stream, "wait_event", lambda st, ev: (waited.append(not ev.query()), wait(st, ev))[1])
    got = []
    for st, lg, (_, *rest) in zip([torch.cuda.Stream() for _ in range(3)] * 2, lgs, steps):
        with torch.cuda.stream(st):
            torch.cuda._sleep(5_000_000)  # (two calls' streams are busy at once)
            got.append(s(lg, *rest))
    torch.cuda.synchronize()
    assert len(waited) == 5 and any(waited)
    assert all(torch.equal(g, w) for g, w in zip(got, want))
