"""Prompts of dense uniform decoders: which products they run on, beside the same step on the library's."""
import pytest
import torch

from src import ops
from src.models.config import resolve_model
from src.models.weights import random_stage_weights
from src.ops import prompt
from src.runtime.executor import StageExecutor

pytestmark = pytest.mark.gpu


# row tiles that the table gives to the gate / up product alone, to the down product too, and to all four
# (a stage with a head: none, and the same bits)
@pytest.mark.parametrize("T,head", [(300, False), (1000, False), (4330, False), (1000, True)])
def test_products_of_a_prompt(T, head, monkeypatch):
    ops.require_native()
    cfg = resolve_model("llama2-7b")
    w = random_stage_weights(cfg, 0, 1, has_embed=False, has_head=head, device="cuda:0", seed=T)
    x = torch.randn(T, cfg.hidden_size, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).cuda()
    want = 0 if head else sum(prompt.chosen(T, *s) for s in prompt.shapes(cfg))
    outs, calls, run = [], [], prompt._run
    monkeypatch.setattr(prompt, "_run", lambda *a: calls.append(a) or run(*a))
    for table in (prompt.table(), {}):
        monkeypatch.setitem(prompt._STATE, "table", table)
        ex = StageExecutor(cfg, w, "cuda:0", max_sessions=4, max_seq_len=T + 8, kv_cache_bytes=1 << 30, warmup=False)
        outs.append(ex.forward([("a", T - 100), ("b", 100)], x).double())
    assert len(calls) == want and bool(want) == (not head)  # (the gated product at least, at all three row counts)
    # five bf16 roundings of a row's values on the way (q k v, attention, o, activation, down), of 2^-9 each, in one and the other
    assert float((outs[0] - outs[1]).norm() / outs[1].norm()) < (2 * 5 * 2.0 ** -9 if want else 1e-12)
