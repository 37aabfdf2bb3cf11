"""Deep prompts of fine-tuning, added in the norm's launch (csrc/train.hip): the bits of the sums that torch rounds one after the other."""
import pytest
import torch

from src import ops
from src.models.config import resolve_model
from src.models.weights import random_stage_weights
from src.ops import train
from src.runtime.autograd_stage import AutogradStage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [8, 4096, 4104, 16384])
@pytest.mark.parametrize("B,T,P", [(1, 1, 1), (1, 5, 2), (3, 7, 7), (3, 4, 1)])
@pytest.mark.parametrize("shared", [True, False])
def test_norm_of_prompted_rows(B, T, P, H, shared):
    ops.require_native()
    g = torch.Generator().manual_seed(B + T + P + H)
    x, y = (torch.randn(B * T, H, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    deep = torch.randn(1 if shared else B, P, H, generator=g).to(torch.bfloat16).cuda()
    w = (torch.rand(H, generator=g) + 0.5).to(torch.bfloat16).cuda()
    for add in (None, y):
        was = x.clone()
        want = x.clone() if add is None else x + add
        want.view(B, T, H)[:, :P] += deep
        total, out = train.norm(x, w, 1e-5, add, deep, T)
        assert torch.equal(total, want) and torch.equal(x, was)
        assert torch.equal(out, train.norm(want, w, 1e-5)[1])


@pytest.mark.parametrize("prompts", [(2, 1, 3, 512), (2, 3, 3, 512), (2, 1, 3, 1), (2, 3, 0, 512)])
def test_shapes_of_prompts(prompts):
    """One prompt for all sequences or one each, one number for a whole row, none: as a prompt of every row of its own; others raise."""
    cfg = resolve_model("small-llama")
    stage = AutogradStage(cfg, random_stage_weights(cfg, 0, 2, has_embed=False, has_head=False, device="cuda:0", seed=1), "cuda:0")
    g = torch.Generator().manual_seed(3)
    x = torch.randn(3, 6, cfg.hidden_size, generator=g).to(torch.bfloat16).cuda()
    p = torch.randn(prompts, generator=g).to(torch.bfloat16).cuda()
    full = p.expand(2, 3, prompts[2], cfg.hidden_size).contiguous()
    assert torch.equal(stage.forward(x, p), stage.forward(x, full))
    with pytest.raises(RuntimeError):
        stage.forward(x, torch.zeros(2, 2, 3, cfg.hidden_size, device="cuda"))
