"""How prompts of head-mixing attention are split, and the merges and choices that follow, at their edges."""
import pytest
import torch

from src.models.config import MoESpec
from src.ops import mixed as xops
from src.ops import moe as eops
from tests import nuvorax_utils as U


@pytest.mark.parametrize("ntoks,starts", [([1], [0]), ([1800], [0]), ([100, 1801, 777], [0, 0, 0]), ([5, 8192], [4000, 0]),
                                          ([40] * 200, [0] * 200), ([300], [30000])])
@pytest.mark.parametrize("tokens,slots", [(16, 256), (8, 512), (16, 1)])
def test_splits_follow_the_work(ntoks, starts, tokens, slots):
    """Whole tiles, every key covered, 16 splits at most; none longer than a slot's share, 256 keys or the cap ask for."""
    ps, n = xops.prompt_splits(ntoks, starts, tokens, slots)
    span = max(a + b for a, b in zip(ntoks, starts))
    keys = sum(s + min(k + tokens, t) for t, s in zip(ntoks, starts) for k in range(0, t, tokens))
    assert ps % xops.KEYS == 0 and 1 <= n <= 16 and ps * n >= span > ps * (n - 1)
    assert ps - xops.KEYS < max(256, -(-span // 16), keys // slots)


@pytest.mark.parametrize("parts", [(256, 1), (256, 16), (288, 9), (32, 11)])
@pytest.mark.parametrize("most", [0, 1, 2, 3, 5, 8, 16, 100])
def test_as_many_splits_as_fit(parts, most):
    """Splits whose scratch is over its limit give way to fewer and longer ones, not to a single one."""
    ps, n = xops.fit_splits(parts, 1000, 1000 * most + 999)
    if parts[1] <= most:
        assert (ps, n) == parts
    elif most < 2:
        assert (ps, n) == (0, 1)
    else:
        assert ps % xops.KEYS == 0 and 2 <= n <= most and ps * n >= parts[0] * parts[1] > ps * (n - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 3, 4, 5, 7, 8, 9, 17])
def test_decode_merges_any_number_of_splits(splits):
    from tests.test_nuvorax_gpu import DEV, near, run_attn

    a = U.Attn([1] * 5, [0, 31, 290, 550, 599], 16, 4, 128, 128, dt=torch.bfloat16, device=DEV, page=64)
    near(run_attn(a, "rows", splits), a.want())


@pytest.mark.gpu
@pytest.mark.parametrize("E,top,groups,keep", [(8, 2, 1, 1), (32, 4, 4, 2), (64, 8, 8, 3), (65, 3, 5, 5), (512, 20, 64, 7)])
@pytest.mark.parametrize("T", [1, 2, 7, 8, 9, 16, 17])
def test_one_workgroup_chooses_and_places(E, top, groups, keep, T):
    """Up to 16 tokens (8 with over 256 experts) one workgroup also places the rows; exact against the CPU's choice."""
    from tests.test_nuvorax_gpu import DEV, check_choice, scratch

    W = 512
    g = torch.Generator().manual_seed(E + T)
    x, w = torch.randn(T, W, generator=g).to(torch.bfloat16), (torch.randn(E, W, generator=g) * 3 / W ** 0.5).to(torch.bfloat16)
    ctx = torch.ones(T, dtype=torch.int32)
    ctx[1::5] = 0  # padding rows
    spec = MoESpec(E, top, 8, 1.0, groups, keep, 1.9)
    p, idx = eops._choose_cpu(x.float(), w.float(), torch.ones_like(ctx), spec)
    c = eops.choose(x.to(DEV), w.to(DEV), ctx.to(DEV), spec, scratch())
    check_choice(c, torch.zeros(T, E).scatter_(1, idx, p), ctx > 0)
