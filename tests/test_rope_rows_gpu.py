"""Rotation and cache write of many rows (csrc/rope_kv.hip, a thread an item): the bits of steps of fewer rows, which a workgroup a row
makes, and the rounded reference."""
import pytest
import torch

from src import ops
from src.ops import reference as ref

pytestmark = pytest.mark.gpu


# 512 rows and one more, items that fill workgroups and not, 32 / 32 heads of 128 (which keep a workgroup a row)
@pytest.mark.parametrize("T", [512, 513, 1030])
@pytest.mark.parametrize("nh,nkv,D", [(32, 8, 128), (64, 8, 128), (5, 1, 128), (12, 12, 64), (3, 3, 16), (4, 2, 24), (32, 32, 128)])
def test_many_rows(T, nh, nkv, D):
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(T + nh + D)
    ps, wide = 16, (nh + 2 * nkv) * D
    pages = T // ps + 2
    angle = torch.rand(2 * T, D // 2, generator=g, device="cuda") * 6.28
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, 2 * T, (T,), generator=g, device="cuda")
    slots = torch.randperm(pages * ps, generator=g, device="cuda")[:T]
    slots[:: 37] = -1  # (rows that are not written)
    x = torch.randn(T, wide + 8, generator=g, device="cuda").to(torch.bfloat16)
    kv = [torch.randn(pages, nkv, ps, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2)]
    many, few, plain = ([x.clone()] + [c.clone() for c in kv] for _ in range(3))
    ops.rope_kv_write(many[0][:, :wide], pos, cos, sin, many[1], many[2], slots, nh, nkv)
    for a in range(0, T, 300):
        part = slice(a, min(T, a + 300))
        ops.rope_kv_write(few[0][part, :wide], pos[part].contiguous(), cos, sin, few[1], few[2], slots[part].contiguous(), nh, nkv)
    assert all(torch.equal(a, b) for a, b in zip(many, few))
    ref.rope_kv_write(plain[0][:, :wide], pos, cos, sin, plain[1], plain[2], slots, nh, nkv)
    # a sum of two products in 32 bits, rounded to bf16 once: a unit of its 8 bits apart at most
    for a, b in zip(many, plain):
        assert bool(((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 1e-6).all())
