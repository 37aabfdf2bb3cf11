"""Prompts of dense uniform decoders: which products they run on, beside the same step on the library's."""
import pytest
import torch

from src import ops
from src.models.config import resolve_model
from src.models.weights import random_stage_weights
from src.ops import prompt
from src.runtime.executor import StageExecutor

pytestmark = pytest.mark.gpu


# rows at which the tables give qkv to the 128 x 128 tiles and gate / up and down to the larger ones, those two alone, and all four
# (a stage with a head: none, and the same bits)
@pytest.mark.parametrize("T,head", [(300, False), (1000, False), (4330, False), (1000, True)])
def test_products_of_a_prompt(T, head, monkeypatch):
    ops.require_native()
    cfg = resolve_model("llama2-7b")
    w = random_stage_weights(cfg, 0, 1, has_embed=False, has_head=head, device="cuda:0", seed=T)
    x = torch.randn(T, cfg.hidden_size, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).cuda()
    mid = [s for s in prompt.shapes(cfg) if not head and prompt.mid(T, *s)]
    large = [s for s in prompt.shapes(cfg) if not head and s not in mid and (prompt.chosen(T, *s) or prompt.few(T, *s))]
    outs, calls = [], {"_run": [], "_run_mid": []}
    for name in calls:
        monkeypatch.setattr(prompt, name, lambda *a, name=name, run=getattr(prompt, name): calls[name].append(
            (a[3], a[0].shape[1], a[4])) or run(*a))
    for tables in ({n: prompt.table(n) for n in ("table", "few", "mid")}, {"table": {}, "few": {}, "mid": {}}):
        for name, t in tables.items():
            monkeypatch.setitem(prompt._STATE, name, t)
        ex = StageExecutor(cfg, w, "cuda:0", max_sessions=4, max_seq_len=T + 8, kv_cache_bytes=1 << 30, warmup=False)
        outs.append(ex.forward([("a", T - 100), ("b", 100)], x).double())
    # (of the second stage none: it has no tables)
    assert sorted(calls["_run"]) == sorted(large) and sorted(calls["_run_mid"]) == sorted(mid)
    assert bool(large or mid) == (not head) and (T != 300 or (len(large), len(mid)) == (2, 1))
    # five bf16 roundings of a row's values on the way (q k v, attention, o, activation, down), of 2^-9 each, in one and the other
    assert float((outs[0] - outs[1]).norm() / outs[1].norm()) < (2 * 5 * 2.0 ** -9 if large or mid else 1e-12)
