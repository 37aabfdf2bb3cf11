"""How prompts of head-mixing attention are split, and the merges and choices that follow, at their edges."""
import pytest
import torch

from src.models.config import MoESpec
from src.ops import mixed as xops
from src.ops import moe as eops
from tests import nuvorax_utils as U


PROMPTS = [([1], [0]), ([1800], [0]), ([100, 1801, 777], [0, 0, 0]), ([5, 8192], [4000, 0]), ([40] * 200, [0] * 200),
           ([300], [30000]), ([300], [4000]), ([1000], [1000]), ([100] * 4, [3000] * 4), ([500, 100, 0], [500, 2000, 9])]


@pytest.mark.parametrize("ntoks,starts", PROMPTS)
@pytest.mark.parametrize("tokens,cus", [(16, 256), (8, 256), (16, 32), (16, 1)])
def test_splits_take_the_fewest_rounds(ntoks, starts, tokens, cus):
    """Whole tiles, every key covered, 16 splits at most, none under 256 keys.  The denominators': no other number is better
    in rounds of the fullest XCD's workgroups, counted one by one; the values': at most twice that."""
    blk = xops.mixed_blocks(ntoks, starts, tokens)
    span = max(a + b for a, b in zip(ntoks, starts) if a)
    most = min(16, -(-span // 256))
    xcds = [[] for _ in range(8)]  # contexts of every XCD's blocks
    for i, (t, k) in enumerate(blk.T.tolist()):
        if k:
            q, at = 0, 0
            while t >= at + ntoks[q]:
                at, q = at + ntoks[q], q + 1
            xcds[i % 8].append(starts[q] + t + k - at)

    def cost(size):
        rounds = max(-(-sum(-(-c // size) for c in x) // max(1, cus // 8)) for x in xcds)
        return max(rounds * (size + 64), sum(map(sum, xcds)) / cus)

    least = min(cost(xops.KEYS * -(-span // (xops.KEYS * m))) for m in range(1, most + 1))
    for (ps, n), slack in zip(xops.prompt_splits(blk, ntoks, starts, cus), (1.0, 2.0)):
        assert ps % xops.KEYS == 0 and 1 <= n <= most and ps * n >= span > ps * (n - 1)
        assert n == 1 or ps > 256 - xops.KEYS
        assert cost(ps) <= slack * least + 1e-6


def test_splits_of_portions_and_prompts():
    """Contexts alike: as many as one round takes; a long prompt's triangle: the values keep few."""
    for ntoks, starts, tokens, want in (([300], [4000], 16, (11, 11)), ([1000], [4000], 16, (4, 4)), ([1800], [0], 16, (8, 3)),
                                        ([8192], [0], 8, (14, 3)), ([200], [0], 16, (1, 1)), ([], [], 16, (1, 1))):
        got = xops.prompt_splits(xops.mixed_blocks(ntoks, starts, tokens), ntoks, starts)
        assert (got[0][1], got[1][1]) == want, (ntoks, starts, got)


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


@pytest.mark.gpu
@pytest.mark.parametrize("E,top", [(5, 2), (16, 4), (17, 4), (32, 4)])
@pytest.mark.parametrize("W", [64, 256, 2048, 4096, 7168])
@pytest.mark.parametrize("packed", [False, True])
def test_choice_in_one_launch_has_the_same_sums(E, top, W, packed):
    """Up to 16 tokens and 32 experts the choice makes the logits too: the very weights of the same tokens among 17."""
    from src import ops
    from tests.test_nuvorax_gpu import DEV, check_choice, scratch

    ops.require_native()
    g = torch.Generator().manual_seed(E + W)
    x, w = torch.randn(17, W, generator=g).to(torch.bfloat16), (torch.randn(E, W, generator=g) * 3 / W ** 0.5).to(torch.bfloat16)
    spec, xd, wd = MoESpec(E, top, 8, 1.0, 1, 1, 1.9), x.to(DEV), w.to(DEV)
    many = eops.choose(xd, wd, torch.ones(17, dtype=torch.int32, device=DEV), spec, scratch())
    p, idx = eops._choose_cpu(x.float(), w.float(), torch.ones(17, dtype=torch.int32), spec)
    for T in (1, 6, 15, 16):
        rows = ops.pack_act(xd[:T].contiguous()) if packed else xd[:T]
        few = eops.choose(rows, wd, torch.ones(T, dtype=torch.int32, device=DEV), spec, scratch(), packed=packed)
        assert torch.equal(few.weights, many.weights[:T])
        check_choice(few, torch.zeros(T, E).scatter_(1, idx[:T], p[:T]), torch.ones(T, dtype=torch.bool))
