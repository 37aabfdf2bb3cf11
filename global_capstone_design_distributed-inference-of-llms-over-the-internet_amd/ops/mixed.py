"""Ops of decoders with head-mixing attention and parallel sublayers (csrc/attention_mixed.hip).

Same dispatch rule as the package: GPU tensors run the HIP kernels, CPU tensors the plain-PyTorch forms of
``reference_mixed``.  Attention and the feed-forward's activation write one buffer [T, K] side by side, the input of the
layer's output projection; ``packed`` writes it in the packed decode-GEMM layout.
"""
from __future__ import annotations

import numpy as np
import torch

from . import reference_mixed as rx
from .hybrid import _native, _put

FF_KINDS = {None: 0, "gelu": 1, "clamped_glu": 2, "gated_glu": 3}


def ffn_act(z, out, kind, F, block=1, limit=0.0, packed=False):
    """Activation of a feed-forward's projected rows: ``gelu`` of [up], the clamped gated form of [gate and up in blocks],
    or (``gated_glu``) that times the sigmoid of the column after them."""
    if not _native(z):
        return _put(out, rx.ffn_act(z, kind, F, block, limit), packed)
    torch.ops.mpamd.ffn_act(z, out, FF_KINDS[kind], int(F), int(block), float(limit), int(packed))
    return out


def mixed_prep(z, q_gain, k_gain, qn, cache, slots, q_ctx, rope, vrope, out, K, eps, ff=None, packed=False):
    """Norms and rotations of projected rows [q | k | v | gate]: ``qn`` gets the queries, keys and turned values go to the
    cache at ``slots`` (-1: skip).  ``ff`` (kind, F, block, column, limit): the feed-forward activation of the row's later
    columns, which goes to columns [H V, H V + F) of ``out`` [T, K]."""
    if not _native(z):
        rx.mixed_prep(z, q_gain, k_gain, qn, cache, slots, q_ctx, rope, vrope, eps)
        if ff is not None:
            kind, F, block, col, limit = ff
            H = qn.shape[1] // q_gain.numel()
            rx.put_columns(out, rx.ffn_act(z[:, col:], kind, F, block, limit), H * vrope.shape[1], K, packed)
        return
    kind, F, block, col, limit = ff if ff is not None else (None, 0, 1, 0, 0.0)
    torch.ops.mpamd.mixed_prep(z, q_gain, k_gain, qn, cache, slots, q_ctx, rope, vrope, out, int(K), FF_KINDS[kind],
                               int(F), int(block), int(col), float(limit), float(eps), int(packed))


KEYS = 32  # keys of a tile: splits of a context are multiples of it
XCDS = 8


def mfma_ok(H, G, D, V, page, cap):
    """(tokens of a query block of the MFMA form for prompts, 0: not covered; does the decode form cover the shape)."""
    r = int(torch.ops.mpamd.mixed_mfma_ok(int(H), int(G), int(D), int(V), int(page), float(cap)))
    return (r >> 8 if r & 1 else 0), bool(r & 2)


def fit_splits(parts, size: int, limit: int):
    """``parts`` (keys per split, splits), or fewer and longer ones whose scratch of ``size`` bytes a split keeps within
    ``limit``; (0, 1) where not even two do."""
    ps, n = parts
    most = limit // max(1, size)
    if n <= most:
        return ps, n
    if most < 2:
        return 0, 1
    longer = KEYS * -(-ps * n // (KEYS * most))
    return longer, -(-ps * n // longer)


def mixed_blocks(ntoks, starts, tokens: int):
    """Query blocks of a ragged step: int32 [2, n] (first flat token, tokens; 0: a filler).  Workgroup i runs on XCD
    i % 8, and every XCD has an L2 of its own: a sequence's blocks stay on one XCD as long as that leaves none with more
    than its share of the keys to read, and the others' blocks even the shares out.  (Spread first, with whole sequences
    on top, the fullest XCD of prompts of 1801, 1401, 750 and 350 tokens had 1.65 shares: their denominators and values took
    94 and 230 us a layer, now 77 and 186.)  Blocks with long
    contexts come first."""
    seqs, off = [], 0
    for n, s in zip(np.asarray(ntoks).tolist(), np.asarray(starts).tolist()):
        b = [(s + min(k + tokens, n), off + k, min(tokens, n - k)) for k in range(0, n, tokens)]
        if b:
            seqs.append((sum(x[0] for x in b), b))
        off += n
    seqs.sort(key=lambda x: -x[0])
    share = sum(w for w, _ in seqs) * 1.05 / XCDS
    bins, load, loose = [[] for _ in range(XCDS)], [0] * XCDS, []
    for w, b in seqs:
        i = load.index(min(load))
        if load[i] + w > share:
            loose += b
            continue
        bins[i] += b
        load[i] += w
    for x in sorted(loose, key=lambda x: -x[0]):
        i = load.index(min(load))
        bins[i].append(x)
        load[i] += x[0]
    depth = max((len(b) for b in bins), default=0)
    out = np.zeros((2, depth, XCDS), dtype=np.int32)
    for i, b in enumerate(bins):
        b.sort(key=lambda x: -x[0])
        for k, (_, t, n) in enumerate(b):
            out[:, k, i] = t, n
    return np.ascontiguousarray(out.reshape(2, -1))


def prompt_splits(blk, ntoks, starts, n_cu: int = 256, least: int = 256, most: int = 16):
    """(keys per split, splits) of a prompt's query blocks ``blk`` (``mixed_blocks``): for the denominators, and for the
    values.  Splits are even, 16 at most, none under 256 keys.

    A workgroup's time is its keys and some 64 more, and an XCD runs ``n_cu`` / 8 at a time.  The denominators' splits are
    those whose rounds on the XCD with the most workgroups are shortest: a few past a round take as long as a round.  The
    values' are a compromise of that and of the keys shared out evenly (whole splits come first and the rest fills the CUs,
    which is what happens to the triangle of a long prompt), and every split of a block that has several costs 128 keys
    more, since it is written and added; within 3 % the fewest.

    us of attention, 16 heads; splits from the mean block over 256 CUs / from all keys over 1.5 workgroups a CU / these:
    1800 tokens 160 / 126 / 120, 300 after 4000 118 / 134 / 92, 1000 after 4000 255 / 265 / 212, 1400 after 700 176 / 136 / 130,
    4 x 100 after 3000 114 / 124 / 92; 4000 tokens of 32 heads 705 / 735 / 687.  It is not the best of all: 500 after 500 beside
    100 after 2000 89 / 98 / 97."""
    seqs = [(n, s) for n, s in zip(np.asarray(ntoks).tolist(), np.asarray(starts).tolist()) if n]
    span, cus = max((n + s for n, s in seqs), default=1), max(1, n_cu // XCDS)
    if span <= least:
        return (KEYS * -(-span // KEYS), 1), (KEYS * -(-span // KEYS), 1)
    ends = np.concatenate([np.arange(s + 1, s + n + 1, dtype=np.int32) for n, s in seqs])
    keys = np.where(blk[1] > 0, ends[blk[0] + blk[1] - 1], 0).reshape(-1, XCDS, 1)
    ps = KEYS * -(-span // (KEYS * np.arange(1, min(most, -(-span // least)) + 1, dtype=np.int32)))
    pieces = keys // ps  # [rows of blocks, XCDS, choices]
    rest = keys - pieces * ps
    whole, rests, longest, share = pieces.sum(0), rest.sum(0), rest.max(0), int(keys.sum()) / n_cu
    pieces += rest > 0
    groups = pieces.sum(0)
    added = groups - (pieces == 1).sum(0)
    full = -(-groups // cus) * (ps + 64)
    over = whole % cus  # whole splits of the last round; the rests fill the other CUs
    tail = np.maximum(np.maximum(np.where(over > 0, ps, 0), longest), (over * ps + rests) / cus)
    even = whole // cus * ps + tail + 64 * -(-groups // cus)

    def first(cost, slack):
        cost = np.maximum(cost.max(0), share)
        best = int(ps[np.flatnonzero(cost <= slack * cost.min())[0]])
        return best, -(-span // best)

    return first(full, 1.0), first((full + even) / 2 + 128 / cus * added, 1.03)


def mixed_parts(groups: int, span: int, n_cu: int = 256, least: int = 2 * KEYS):
    """(keys per split, splits) of ``groups`` workgroups whose queries see at most ``span`` keys: about one workgroup per
    CU, no split under ``least`` keys."""
    span = max(1, int(span))
    n = max(1, min(n_cu // max(1, int(groups)), span // least))
    ps = KEYS * -(-span // (KEYS * n))
    return ps, -(-span // ps)


def mixed_attention(z, qn, talk, cache, table, q_seq, q_ctx, vrope, out, K, scale, cap, packed=False, form=0, blocks=None,
                    parts=(0, 1), sums=None, part=None, sum_parts=(0, 1)):
    """Causal attention over the cache, into columns [0, H V) of ``out`` [T, K]; the head gates come from ``z``.
    On the GPU ``form`` 1 (prompts: ``blocks`` [2, n] first token and tokens of every query block) and 2 (decode: every
    row one token) run on MFMA, with the context in ``parts`` (keys per split, splits) and fp32 scratch ``sums``
    [splits T H] and ``part`` [splits T H V] (prompts of several splits) or [splits T G H V]; a prompt's denominators
    have splits of their own (``sum_parts``, ``sums``).  0 takes any shape."""
    if not _native(z):
        y = rx.mixed_attention(z, qn, talk, cache, table, q_seq, q_ctx, vrope, scale, cap)
        return rx.put_columns(out, y, 0, K, packed)
    torch.ops.mpamd.mixed_attention(z, qn, talk, cache, table, q_seq, q_ctx, vrope, out, int(K), float(scale), float(cap),
                                    int(packed), int(form), blocks, int(parts[0]), int(parts[1]), sums, part, int(sum_parts[0]),
                                    int(sum_parts[1]))
    return out
