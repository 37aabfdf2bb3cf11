"""Ops of the pre-norm decoders: residual stream with input norms, clamped gated feed-forward, scalar-decay linear
attention (retention, mLSTM) and latent attention.

Same dispatch rule as the package: GPU tensors run the HIP kernels (csrc/pre_norm.hip, csrc/linear_attn.hip,
csrc/latent.hip), CPU tensors the plain-PyTorch forms of ``reference_mixers``.  ``packed`` writes an activation in the
packed decode-GEMM layout.
"""
from __future__ import annotations

import numpy as np
import torch

from . import reference_mixers as rm
from .hybrid import _native, _put


def rope_table(base: float, dims: int, positions: int, device, scaling=None) -> torch.Tensor:
    """fp32 [positions, dims]: cosines, then sines, of position * f_i, f_i = base^(-2i / dims) (angles made in fp64).
    ``scaling`` (factor, low, high, original): frequencies whose wavelength is above original / low are divided by the
    factor, those below original / high are kept, and between them the two are blended linearly in 1 / wavelength."""
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = torch.pow(float(base), -2.0 * i / max(dims, 1))
    if scaling is not None:
        factor, low, high, original = (float(x) for x in scaling)
        keep = ((original * f / (2.0 * torch.pi) - low) / (high - low)).clamp(0.0, 1.0)
        f = keep * f + (1.0 - keep) * f / factor
    a = torch.arange(positions, dtype=torch.float64)[:, None] * f[None]
    return torch.cat([torch.cos(a), torch.sin(a)], 1).float().to(device)


# ------------------------------------------------------------------ residual stream
def _open(res, w, eps, x, center, packed, groups, shift, copy):
    """``x`` of the next sublayer from the stream (CPU)."""
    from .reference_mixed import put_columns

    if copy:
        return put_columns(x, res, 0, copy, packed)
    if w is None:
        return None
    h = rm.norm(res, w, eps, center, groups)
    if shift is not None:
        h = rm.token_shift(h, *shift[:4])
    return _put(x, h, packed)


def put_columns(y, x, col, K, packed=False):
    """Columns [col, ..) of the activation ``x`` [n, K] from fp32 rows."""
    from .reference_mixed import put_columns as put

    if not _native(x):
        return put(x, y, col, K, packed)
    torch.ops.mpamd.put_columns(y, x, int(col), int(K), int(packed))
    return x


def embed_rows_norm(ids, table, res, w, eps, groups=1, x=None, col=0, K=0, packed=False):
    """res[t] = norm(table[ids[t]]) * w (fp32); ``x`` [n, K] gets a copy in columns [col, col + W)."""
    from .reference_mixed import put_columns

    if not _native(table):
        res.copy_(rm.norm(table[ids.long()], w, eps, False, groups))
        return put_columns(x, res, col, K, packed) if x is not None else None
    torch.ops.mpamd.embed_rows_norm(ids, table, res, w, float(eps), int(groups), x, int(col), int(K), int(packed))
    return x


def embed_norm(ids, table, res, w, eps, x, center=False, packed=False, scale=1.0):
    """res[t] = scale * table[ids[t]] (fp32), x = norm(res) * w; ``center``: layer norm, else root mean square."""
    if not _native(table):
        res.copy_(table[ids.long()].float() * scale)
        return _put(x, rm.norm(res, w, eps, center), packed)
    torch.ops.mpamd.embed_norm(ids, table, res, w, x, float(eps), int(center), int(packed), float(scale))
    return x


def add_norm(y, res, mult, w, eps, x, center=False, packed=False, experts=None, groups=1, shift=None, keep=True, copy=0):
    """res += mult * y, then x = norm(res) * w.  ``y``: [n, W], fp32 split-K slabs [S, n, W], or None; ``w`` None:
    the sum alone.  ``experts``: routed experts' outputs that belong to y, (rows, row of every choice [n, top] with -1
    for none, weights [n, top]).  ``groups``: equal parts of a row that are normed alone.  ``keep`` False: res = mult * y.
    ``copy``: x [n, copy] gets the stream itself in its first columns (no norm).  ``shift`` (mu [W], rows [sessions, 2, W],
    q_seq, q_ctx, scratch): x is the norm moved towards the previous token's (``reference_mixers.token_shift``); scratch
    None: every row is one token, else (first [sessions, W], stats [n, groups]) fp32."""
    if not _native(res):
        if not keep:
            res.zero_()
        if y is not None:
            res.add_((y.sum(0) if y.dim() == 3 else y).float() * mult)
        if experts is not None:
            ye, slot, ew = experts
            pick = torch.where((slot >= 0)[..., None], ye[slot.clamp(min=0).long()].float(), 0.0)
            res.add_((pick * ew[..., None]).sum(1) * mult)
        return _open(res, w, eps, x, center, packed, groups, shift, copy)
    if groups == 1 and shift is None and keep and not copy:
        torch.ops.mpamd.add_norm(y, res, w, x, float(mult), float(eps), int(center), int(packed),
                                 *(experts if experts is not None else ()))
        return x
    if experts is not None:
        raise ValueError("routed experts go with a plain norm")
    mu, rows, q_seq, q_ctx, scratch = shift if shift is not None else (None,) * 5
    torch.ops.mpamd.open_norm(y, res, w, x, float(mult), float(eps), int(center), int(packed), int(groups), int(keep), int(copy),
                              mu, rows, q_seq, q_ctx, *(scratch if scratch is not None else (None, None)))
    return x


def rows_norm(res, rows, w, eps, out, center=False, packed=False, groups=1):
    """out[i] = norm(res[rows[i]]) * w."""
    if not _native(res):
        return _put(out, rm.norm(res.index_select(0, rows.long()), w, eps, center, groups), packed)
    torch.ops.mpamd.rows_stream_norm(res, rows, w, out, float(eps), int(center), int(packed), int(groups))
    return out


def clamped_glu(x, out, block, limit, packed=False):
    """g sigmoid(1.702 g) (u + 1) with g <= limit and |u| <= limit, or (limit 0) silu(g) u; ``x`` [n, 2 F] in gate / up
    blocks of ``block``."""
    if not _native(x):
        return _put(out, rm.clamped_glu(x, block, limit), packed)
    torch.ops.mpamd.clamped_glu(x, out, int(block), float(limit), int(packed))
    return out


def softcap(x, cap):
    """cap tanh(x / cap), in place."""
    if not _native(x):
        return x.copy_(cap * torch.tanh(x.float() / cap))
    torch.ops.mpamd.softcap(x, float(cap))
    return x


# ------------------------------------------------------------------ scalar-decay linear attention
def linear_plan(ntoks, heads: int, n_cu: int = 256, seg_tokens: int = None, per_cu: int = 2):
    """Segments of a ragged step, shared with the gated recurrence (``hybrid.hgrn2_plan``)."""
    from .hybrid import hgrn2_plan

    return hgrn2_plan(ntoks, heads, n_cu, seg_tokens, per_cu)


def retention(z, rope, log_decay, state, q_seq, q_ctx, out, eps, plan=None, packed=False):
    """Retention over a ragged step.  ``z`` [T, 2 H (D + V)] projected rows [q | k | v | gate], ``state`` [rows, H, D, V]
    fp32 updated in place for row q_seq[t]; a token of context 1 starts from a zero state, a row of context 0 is
    padding.  ``plan``: None = every row is one token of its own sequence (decode), else the step's device plan."""
    if not _native(z):
        return _put(out, rm.retention(z, rope, log_decay, state, q_seq, q_ctx, eps), packed)
    return _linear(0, z, rope, log_decay, None, None, state, None, q_seq, q_ctx, out, 0.0, eps, 1.0,
                   state.shape[2] ** -0.5, plan, packed)


def mlstm(z, bias, cap, norm_w, state, aux, q_seq, q_ctx, out, eps, plan=None, packed=False):
    """mLSTM over a ragged step, as ``retention``; z rows [q | k | v | gate | i | f], ``bias`` [2, H] of the log gates,
    ``aux`` [rows, H, D + 1]: normalizer and running maximum."""
    if not _native(z):
        return _put(out, rm.mlstm(z, bias, cap, norm_w, state, aux, q_seq, q_ctx, eps), packed)
    return _linear(1, z, None, None, bias, norm_w, state, aux, q_seq, q_ctx, out, cap, eps, state.shape[2] ** -0.5, 1.0,
                   plan, packed)


def _linear(kind, z, rope, decay, bias, norm_w, state, aux, q_seq, q_ctx, out, cap, eps, qs, ks, plan, packed):
    _, H, D, V = state.shape
    head = (kind, z, rope, decay, bias, norm_w, state, aux, q_seq, q_ctx, out, float(cap), float(eps), float(qs), float(ks))
    if plan is not None and not plan.get("scan") and z.dtype == torch.bfloat16 and z.stride(0) % 8 == 0 and \
            torch.ops.mpamd.linear_chunk_ok(D, V, 0 if rope is None else rope.shape[1]):
        slots = plan["slots"]
        ws = torch.empty(slots * H * torch.ops.mpamd.linear_slot(D, V), dtype=torch.float32, device=z.device) \
            if slots else None
        torch.ops.mpamd.linear_chunk(*head, plan["seg"], plan["multi"], slots, ws, int(packed))
        return out
    torch.ops.mpamd.linear_scan(*head, None if plan is None else plan["seqs"], int(packed))
    return out


# ------------------------------------------------------------------ latent attention
LATENT_KEYS = 64  # keys of a tile: splits of a context are multiples of it
LATENT_SPLITS = 64  # most splits of a context


def latent_prep(z, qw, cw, cq, cache, slots, q_ctx, rope, eps, packed=False):
    """Norms of projected rows [q latent | c | rotated key]: ``cq`` gets the q latent, [c | turned key] goes to ``cache``
    at ``slots`` (-1: skip)."""
    if not _native(z):
        return _put(cq, rm.latent_prep(z, qw, cw, cache, slots, q_ctx, rope, eps), packed)
    torch.ops.mpamd.latent_prep(z, qw, cw, cq, cache, slots, q_ctx, rope, float(eps), int(packed))
    return cq


def latent_block(H: int, D: int, R: int, V: int, C: int, page: int) -> int:
    """Tokens of a query block on the MFMA form (0: shape not covered)."""
    return int(torch.ops.mpamd.latent_block(int(H), int(D), int(R), int(V), int(C), int(page)))


def latent_parts(groups: int, span: int, n_cu: int = 256):
    """(keys per split, splits) for ``groups`` workgroups whose queries see at most ``span`` keys: about one workgroup
    per CU, no split under two tiles."""
    span = max(1, int(span))
    n = max(1, min(n_cu // max(1, groups), span // (2 * LATENT_KEYS), LATENT_SPLITS))
    ps = LATENT_KEYS * -(-span // (LATENT_KEYS * n))
    return ps, -(-span // ps)


def latent_attention(q, uk, uv, sink, rope, cache, table, q_seq, q_ctx, out, scale, packed=False, u=None, oc=None,
                     rows=None, blocks=None, parts=(0, 1), ws=None):
    """Causal attention over cached latents, with a sink in the denominator.  ``q`` [T, H (D + R)], ``uk`` [H, C, D],
    ``uv`` [H, V, C].  On the GPU the MFMA form runs when its scratch ``u`` [T, H, C + R] and ``oc`` [T, H, C] is given
    (``rows``: token rows to work on, ``blocks`` [2, n] their query blocks; none: every row a block; ``parts``:
    (keys per split, splits) with ``ws`` fp32 scratch), else the form for any shape and element type."""
    if not _native(q):
        return _put(out, rm.latent_attention(q, uk, uv, sink, rope, cache, table, q_seq, q_ctx, scale), packed)
    torch.ops.mpamd.latent_attention(q, uk, uv, sink, rope, cache, table, q_seq, q_ctx, out, float(scale),
                                     0 if u is None else 1, u, oc, rows, blocks, int(parts[0]), int(parts[1]), ws,
                                     int(packed))
    return out


# a portion of a prompt of this many tokens or more has its context's keys and values made for every head
LATENT_WIDE_TOKENS = 64
WIDE_WAVES = 0  # waves of a workgroup of that form (0: by the portions' length)


def latent_wide_ok(D: int, R: int, V: int, C: int) -> bool:
    """Does the form with every head's own keys and values cover the shape?"""
    return bool(torch.ops.mpamd.latent_wide_ok(int(D), int(R), int(V), int(C)))


def latent_wide_plan(ntoks, starts, heads: int, dim: int, n_cu: int = 256, max_rows: int = 1 << 62):
    """Sequences of a ragged step that take the wide form: (sequence numbers, int32 ``blk`` [3, nblk], waves), None when
    there is none.  ``max_rows``: context rows at most; sequences past it keep the other form."""
    pick, rows, base = [], 0, []
    for i, (n, s) in enumerate(zip(np.asarray(ntoks).tolist(), np.asarray(starts).tolist())):
        if n >= LATENT_WIDE_TOKENS and rows + n + s <= max_rows:
            pick.append(i)
            base.append(rows)
            rows += n + s
    if not pick:
        return None
    off = np.concatenate([[0], np.cumsum(ntoks)[:-1]])
    waves = WIDE_WAVES or (8 if dim > 64 and max(int(ntoks[i]) for i in pick) > 128 else 4)
    tb = 32 * waves
    blk = [(off[i] + k, min(tb, ntoks[i] - k), b) for i, b in zip(pick, base) for k in range(0, int(ntoks[i]), tb)]
    return pick, np.ascontiguousarray(np.asarray(blk, dtype=np.int32).reshape(-1, 3).T), waves


def latent_gather(cache, idx, out):
    """out[i] = cache row idx[i] (slots)."""
    torch.ops.mpamd.latent_gather(cache, idx, out)
    return out


def latent_wide(q, kv, lat, sink, rope, q_ctx, out, D, V, scale, blk, waves, packed=False):
    """The wide form of ``latent_attention`` for the tokens of ``blk``: ``kv`` [N, H (D + V)] keys and values of the
    context rows ``lat`` [N, C + R]."""
    torch.ops.mpamd.latent_wide(q, kv, lat, sink, rope, q_ctx, out, int(D), int(V), float(scale), blk, int(waves),
                                int(packed))
    return out
