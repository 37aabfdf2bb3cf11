"""End-to-end stage executor on the GPU (HIP kernels + hipGraph decode) vs the fp32 dense oracle."""
import pytest
import torch

from src.models.config import resolve_model
from src.models.reference_model import reference_forward
from src.models.weights import random_stage_weights
from src.runtime.executor import StageExecutor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", ["small-llama", "tiny-llama"])
@pytest.mark.parametrize("graphs", [False, True])
def test_executor_matches_fp32_reference(model, graphs):
    cfg = resolve_model(model)
    w = random_stage_weights(cfg, 0, cfg.num_hidden_layers, has_embed=True, has_head=True, device="cuda",
                             dtype=torch.bfloat16, seed=3)
    ex = StageExecutor(cfg, w, "cuda", kv_cache_bytes=256 << 20, max_sessions=8, max_seq_len=512,
                       use_graphs=graphs)
    g = torch.Generator().manual_seed(0)
    prompts = [torch.randint(0, cfg.vocab_size, (n,), generator=g) for n in (37, 5)]
    ids = torch.cat(prompts).cuda()
    logits = ex.forward([("a", 37), ("b", 5)], ids)
    seqs = [p.clone() for p in prompts]
    wf = [w]
    for step in range(6):
        for i, p in enumerate(seqs):
            r = reference_forward(wf, p.cuda())[-1]
            torch.testing.assert_close(logits[i].float(), r, atol=0.06, rtol=0.05)
        nxt = torch.argmax(logits.float(), -1)
        seqs = [torch.cat([s, nxt[i:i + 1].cpu()]) for i, s in enumerate(seqs)]
        logits = ex.forward([("a", 1), ("b", 1)], nxt)


def test_graph_and_eager_agree():
    cfg = resolve_model("small-llama")
    w = random_stage_weights(cfg, 0, cfg.num_hidden_layers, has_embed=True, has_head=True, device="cuda", seed=5)
    outs = []
    for graphs in (False, True):
        ex = StageExecutor(cfg, w, "cuda", kv_cache_bytes=128 << 20, max_sessions=4, max_seq_len=512,
                           use_graphs=graphs)
        ids = torch.arange(3 * 20, device="cuda").view(3, 20) % cfg.vocab_size
        ex.forward([(f"s{i}", 20) for i in range(3)], ids.view(-1))
        tok = torch.tensor([1, 2, 3], device="cuda")
        res = []
        for _ in range(4):
            lg = ex.forward([(f"s{i}", 1) for i in range(3)], tok)
            res.append(lg.float())
            tok = torch.argmax(lg.float(), -1)
        outs.append(torch.stack(res))
    torch.testing.assert_close(outs[0], outs[1], atol=2e-2, rtol=2e-2)


def test_pipeline_split_equals_single_stage_on_gpu():
    """Two stages chained in one process == one stage (same weights by construction)."""
    cfg = resolve_model("small-llama")
    L = cfg.num_hidden_layers
    full = random_stage_weights(cfg, 0, L, has_embed=True, has_head=True, device="cuda", seed=9)
    s0 = random_stage_weights(cfg, 0, 3, has_embed=True, has_head=False, device="cuda", seed=9)
    s1 = random_stage_weights(cfg, 3, L, has_embed=False, has_head=True, device="cuda", seed=9)
    kw = dict(kv_cache_bytes=64 << 20, max_sessions=4, max_seq_len=256)
    e_full = StageExecutor(cfg, full, "cuda", **kw)
    e0, e1 = StageExecutor(cfg, s0, "cuda", **kw), StageExecutor(cfg, s1, "cuda", **kw)
    ids = (torch.arange(30, device="cuda") * 7) % cfg.vocab_size
    a = e_full.forward([("x", 30)], ids)
    b = e1.forward([("x", 30)], e0.forward([("x", 30)], ids))
    assert torch.equal(a, b)
    t = torch.argmax(a.float(), -1)
    for _ in range(3):
        a = e_full.forward([("x", 1)], t)
        b = e1.forward([("x", 1)], e0.forward([("x", 1)], t))
        assert torch.equal(a, b)
        t = torch.argmax(a.float(), -1)


@pytest.mark.parametrize("rows,width,dtype", [(1, 1, torch.long), (5, 1, torch.long), (256, 1, torch.long), (3, 4, torch.bfloat16),
                                              (64, 4096, torch.bfloat16), (70, 4100, torch.float32), (3, 5, torch.bfloat16)])
def test_step_input(rows, width, dtype):
    """Metadata and rows arrive whole, and rows past the step's own stay; an odd width goes by a copy."""
    from src import ops

    ops.require_native()
    n = -(-28 * rows // 8) * 8
    host = torch.randint(0, 256, (n,), dtype=torch.uint8).pin_memory()
    meta = torch.zeros(n, dtype=torch.uint8, device="cuda")
    x = torch.randint(-99, 99, (rows, width), device="cuda").to(dtype)
    dst = torch.full((rows + 3, width), 7, dtype=dtype, device="cuda")
    ops.step_input(host, meta, x, dst[:rows])
    assert torch.equal(meta.cpu(), host) and torch.equal(dst[:rows], x) and bool((dst[rows:] == 7).all())
    with pytest.raises(RuntimeError, match="pinned"):
        ops.step_input(host.clone(), meta, None, dst)


def test_step_input_keeps_its_memory():
    """Pinned memory that is let go of while a queued step has still to read it is not handed out before the step has."""
    from src import ops

    ops.require_native()
    n = 16 * 28 * 64
    meta, dst = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.zeros(1, dtype=torch.long, device="cuda")
    ring = torch.randint(0, 200, (2, n), dtype=torch.uint8).pin_memory()
    want, at = ring[1].clone(), ring.data_ptr()
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)
    ops.step_input(ring[1], meta, None, dst)
    read = torch.cuda.Event()
    read.record()
    del ring
    other = [torch.full((2, n), 255, dtype=torch.uint8).pin_memory() for _ in range(3)]
    assert not read.query()  # (10 ms and more of queued work)
    assert all(t.data_ptr() != at for t in other)
    torch.cuda.synchronize()
    assert torch.equal(meta.cpu(), want)


class _Waited:
    """An event that notes whether it was waited for while it was still to come."""

    def __init__(self, event, seen):
        self.event, self.seen = event, seen

    def synchronize(self):
        self.seen.append(not self.event.query())
        self.event.synchronize()


def test_steps_ahead_of_the_device():
    """Many more steps than staging blobs, queued behind other work and none waited for, each of other sessions in another order:
    the logits of steps that were.  A blob is filled again only when the half of the ring that it is in has been read."""
    cfg = resolve_model("small-llama")
    w = random_stage_weights(cfg, 0, cfg.num_hidden_layers, has_embed=True, has_head=True, device="cuda", seed=5)
    steps, lens = 240, [20, 3, 47, 31, 8]
    who = [[(k * m + i) % 5 for i in range(3)] for k in range(steps) for m in (1 + k % 4,)]
    toks = torch.randint(0, cfg.vocab_size, (steps, 3), device="cuda")
    ids = torch.randint(0, cfg.vocab_size, (sum(lens),), device="cuda")
    outs, seen = [], []
    for wait in (True, False):
        ex = StageExecutor(cfg, w, "cuda", kv_cache_bytes=128 << 20, max_sessions=8, max_seq_len=512, warmup=False)
        ex.forward([(f"s{i}", n) for i, n in enumerate(lens)], ids)
        res = torch.empty(steps, 3, cfg.vocab_size, dtype=torch.bfloat16, device="cuda")
        torch.cuda.synchronize()
        for k in range(steps):
            if not wait and k % 40 == 1:
                torch.cuda._sleep(10_000_000)
            res[k].copy_(ex.forward([(f"s{i}", 1) for i in who[k]], toks[k]))
            if wait:
                torch.cuda.synchronize()
                continue
            for g in ex._graphs.values():
                g._half_ev = [_Waited(e, seen) if isinstance(e, torch.cuda.Event) else e for e in g._half_ev]
        outs.append(res)
    assert torch.equal(*outs)
    assert len(ex._graphs) == 1 and len(seen) == steps // 8 - 2 and sum(seen) >= 6
