"""Kernels of the stateless fine-tuning path (csrc/train.hip): norm, rotary, attention and gate steps of a block with their
gradients, all on [tokens, columns] rows.

The reference differentiates the recomputed forward with autograd (petals/server/block_functions.py:84-141); the weights
are frozen, so a block's backward is the gradient with respect to its input alone and is written out in
``runtime.autograd_stage``.
"""
from __future__ import annotations

import torch

MAX_WIDTH = 16384  # of a norm's row


def shape_ok(cfg) -> bool:
    """Do the kernels cover the blocks of this model?"""
    return (cfg.model_type in ("llama", "mistral") and not cfg.is_moe and cfg.head_dim in (64, 128) and
            cfg.hidden_size % 8 == 0 and cfg.hidden_size <= MAX_WIDTH and cfg.intermediate_size % 16 == 0 and
            cfg.num_attention_heads <= 65535)


def rows_ok(B: int, T: int) -> bool:
    """Do they cover B sequences of T tokens?  (A sequence is a grid's z, a block of 64 tokens its x.)"""
    return 1 <= B <= 65535 and 1 <= T <= 1 << 24


def angles(inv: torch.Tensor, T: int) -> torch.Tensor:
    """[T, D]: cos, then sin of every position's angles, from those of one step, ``inv`` [D / 2] (fp64, on the device)."""
    out = torch.empty(T, 2 * inv.numel(), dtype=torch.float32, device=inv.device)
    torch.ops.mpamd.train_angles(inv, out)
    return out


def norm(x, w, eps, add=None, deep=None, T: int = 0):
    """(x + add, its norm times w); without ``add`` and ``deep`` the first is ``x`` itself.  ``deep`` [1 or B, P, H]: added as well, to
    the first P of every ``T`` rows, after that sum was rounded."""
    out = torch.empty_like(x)
    plain = add is None and deep is None
    total = x if plain else torch.empty_like(x)
    torch.ops.mpamd.train_norm(x, add, w, None if plain else total, out, eps, False, deep, T)
    return total, out


def norm_grad(x, dy, w, eps, dres):
    """dres + the gradient of ``norm``'s second output with respect to the row ``x`` that it normed."""
    out = torch.empty_like(x)
    torch.ops.mpamd.train_norm(x, dy, w, dres, out, eps, True)
    return out


def rope_(qkv, table, heads: int, D: int):
    """The first ``heads`` heads of every row turned in place."""
    torch.ops.mpamd.train_rope(qkv, table, heads, D)
    return qkv


def attention(qkv, B: int, nh: int, nkv: int, D: int, keep: bool):
    """Causal attention of B sequences over turned q, k and v in one matrix: (out, fp32 out, log of the denominators);
    the last two for the gradient (``keep``)."""
    n = qkv.shape[0]
    out = torch.empty(n, nh * D, dtype=qkv.dtype, device=qkv.device)
    out32 = lse = None
    if keep:
        out32 = torch.empty(n, nh * D, dtype=torch.float32, device=qkv.device)
        lse = torch.empty(nh * n, dtype=torch.float32, device=qkv.device)
    torch.ops.mpamd.train_attn(qkv, B, nh, nkv, D ** -0.5, out, None if out32 is None else out32.view(-1), lse)
    return out, out32, lse


def attention_grad(qkv, B: int, nh: int, nkv: int, D: int, out32, lse, dout, table):
    """Gradient of ``attention`` and of the turn before it: [tokens, (nh + 2 nkv) D]."""
    n = qkv.shape[0]
    f32 = dict(dtype=torch.float32, device=qkv.device)
    dqkv = torch.empty_like(qkv)
    torch.ops.mpamd.train_attn_grad(qkv, B, nh, nkv, D ** -0.5, out32.view(-1), lse, dout, torch.empty(nh * n, **f32),
                                    table.view(-1), torch.empty(2 * n * nh * D, **f32), dqkv)
    return dqkv


def glu_grad_(gu, da):
    """Gate / up rows (blocks of 16) replaced by their gradients, from the gradient of silu(gate) * up."""
    torch.ops.mpamd.train_glu_grad(gu, da)
    return gu
