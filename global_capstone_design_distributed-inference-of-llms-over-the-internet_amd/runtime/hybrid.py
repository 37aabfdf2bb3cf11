"""Forward step of the hybrid decoders inside a StageExecutor (``ModelConfig.layers``).

The residual stream is fp32 and lives in one buffer; a sublayer f reads an activation ``xb`` made from it.

    post-norm streams   xb = res ;            res += rms(f(xb)) * gain
    pre-norm streams    xb = norm(res) gain ; res += mult * f(xb)

One kernel closes a sublayer: it adds the output projection (rows, or the fp32 split-K slabs of a decode GEMM) to the
stream and writes the next sublayer's ``xb``.  A mixer is one fused input projection z = xb W_in^T, its own ops, and
an output projection; the feed-forward is squared relu, gelu or the clamped gated form, with or without routed experts.

    parallel layers     xb = norm(res) gain ; res += mult * (f(xb) + g(xb))

run as one sublayer: z has the feed-forward's columns too, its activation lies beside the mixer's in the input of one
output projection, and the kernel that closes the layer adds the routed experts' rows.

A pair layer's mixers read columns of one z and write columns of the input of one output projection.  A layer may read its
norm moved towards the previous token's (``LayerSpec.shift``), and a loop's pass may open with a projection of the stream
and the embedding, [res ; res0] W^T, that replaces the stream (``LayerSpec.inject``).

Activations feeding a decode-sized GEMM stay in the packed MFMA-fragment layout where the shape has a native
GEMM (``ops.native_gemm_ok``); other shapes, prompts and fp32 run the library GEMM on row-major activations.
Keys and latents of attention layers live in the executor's paged cache, recurrent states in its ``RecurrentState``:
every layer run has its own, also where a loop runs the same weights again.
"""
from __future__ import annotations

import os
from typing import Optional

import numpy as np
import torch

from .. import ops
from ..ops import gated as gops
from ..ops import hybrid as hops
from ..ops import mixed as xops
from ..ops import mixers as mops
from ..ops import moe as eops
from ..ops import window as wops

# most bytes of fp32 partial sums of a latent attention step whose contexts are split
LATENT_WS_BYTES = 256 << 20
# decode steps of parallel layers run the routed experts beside the mixer
PARALLEL_EXPERTS = os.environ.get("MPAMD_PARALLEL_EXPERTS", "1") != "0"
# most bytes of fp32 partial sums of a head-mixing attention prompt whose contexts are split
MIXED_WS_BYTES = 256 << 20
# most bytes of the keys and values that long portions of prompts make of their contexts' latents, per step
LATENT_KV_BYTES = 4 << 30


class HybridStage:
    """Layer loop of one stage; ``ex`` owns the weights, the cache, the states and the plans."""

    def __init__(self, ex):
        self.ex = ex
        cfg = ex.cfg
        self.W, self.eps = cfg.hidden_size, cfg.rms_norm_eps
        self.pre, self.center, self.mult = cfg.stream == "pre", cfg.norm == "layer", cfg.residual_mult
        self.inv = hops.position_frequencies(self.W, ex.device) if cfg.embed_positions else None
        self.groups = cfg.norm_groups
        # per-layer place in the paged cache and among the states
        self.cache_at, self.state_at, na, nr = [], [], 0, 0
        for sp in cfg.layers[ex.start:ex.end]:
            self.cache_at.append(na)
            self.state_at.append(nr)
            na += sp.cache_row is not None
            nr += bool(sp.state_shapes)
        specs = [sp for lay in ex.w.layers for sp in lay.spec.mixers]
        # angle tables: (base, dimensions, frequency scaling)
        keys = {self._rope_key(sp) for sp in specs if sp.mixer in ("retention", "latent_attention", "mixed_attention",
                                                                          "window_attention")}
        keys |= {(sp.rot_base, sp.vdim, None) for sp in specs if sp.mixer == "mixed_attention"}
        self.rope = {k: mops.rope_table(k[0], k[1], ex.max_seq_len, ex.device, k[2]) for k in keys}
        # query-block tokens of each attention shape's MFMA form (0: the any-shape form)
        self.talk_block, self.latent_block, self.mixed_ok, self.window_rows = {}, {}, {}, {}
        for sp in specs if ex.device.type == "cuda" else ():
            bf16 = ex.dtype == torch.bfloat16
            if sp.mixer == "attention":
                ok = bf16 and ex.cache.page_size >= 32
                self.talk_block[(sp.heads, sp.kv_heads, sp.dim)] = \
                    hops.talk_block(sp.heads, sp.kv_heads, sp.dim) if ok else 0
            elif sp.mixer == "latent_attention":
                key = self._latent_key(sp)
                self.latent_block[key] = mops.latent_block(*key, ex.cache.page_size) if bf16 else 0
            elif sp.mixer == "mixed_attention":
                key = self._mixed_key(sp)
                self.mixed_ok[key] = xops.mfma_ok(*key[:4], ex.cache.page_size, key[4]) if bf16 else (0, False)
            elif sp.mixer == "window_attention":
                key = self._window_key(sp)
                self.window_rows[key] = wops.mfma_ok(*key, ex.cache.page_size) if bf16 and sp.scale > 0 else 0
        self.windows = sorted({(self._window_key(sp), sp.reach) for sp in specs if sp.mixer == "window_attention"})
        self.side = torch.cuda.Stream(ex.device) if ex.device.type == "cuda" and PARALLEL_EXPERTS and \
            any(sp.parallel and sp.moe for sp in specs) else None
        # heads of the layer whose prompts fill the CUs with the fewest segments, and workgroups of it that share a CU (one,
        # where a state is past 128 x 128)
        most = lambda *kinds: max([(sp.heads, 1 if max(sp.dim, sp.vdim) > 128 else 2) for sp in specs if sp.mixer in kinds],  # noqa: E731
                                  key=lambda x: x[0] / x[1], default=None)
        self.rec_fill, self.lin_fill = most("hgrn2"), most("retention", "mlstm")
        self.gated = any(sp.mixer in ("gated_delta", "mamba2", "gla") for sp in specs)
        self.gated_waves = min([sp.heads * -(-sp.vdim // 16) for sp in specs if sp.mixer in ("mamba2", "gla")], default=0)
        self.max_chunk = max([sp.reach for sp in specs if sp.reach], default=1)

    @staticmethod
    def _rope_key(sp):
        return sp.rot_base, sp.rot_dims, sp.rot_scaling

    @staticmethod
    def _mixed_key(sp):
        return sp.heads, sp.kv_heads, sp.dim, sp.vdim, sp.softcap

    @staticmethod
    def _window_key(sp):
        return sp.heads, sp.kv_heads, sp.dim, sp.vdim

    @staticmethod
    def _latent_key(sp):
        return sp.heads, sp.dim, sp.rot_dim, sp.vdim, sp.kv_rank

    def autotune(self) -> None:
        """Decode-GEMM kernel choices for this stage's shapes (none while tuning is off)."""
        if ops.autotune_mode() == "off":
            return
        up = {"relu2": 4, "clamped_glu": 1, "silu_glu": 1, "gelu": 0}
        shapes = {(getattr(lay, n).shape[0], getattr(lay, n).shape[1],
                   up[lay.spec.ffn] if n == "w_up" and not lay.spec.moe else 0)
                  for lay in self.ex.w.layers for n in lay.GEMMS if getattr(lay, n + "_p") is not None}
        if self.ex.w.loop_in_p is not None:
            shapes.add((self.W, 2 * self.W, 0))
        if self.ex.w.lm_head_p is not None:
            shapes.add((self.ex.w.lm_head.shape[0], self.W, 0))
        # (small products are launch-bound whatever kernel runs them)
        ops.autotune_gemm([s for s in sorted(shapes) if s[0] * s[1] >= 1 << 22], self.ex.device)

    # ------------------------------------------------------------------ GEMMs
    def _packed(self, T: int, w, wp) -> bool:
        """Does the GEMM over ``w`` take a packed T-row activation?"""
        return (wp is not None and self.ex.device.type == "cuda" and ops.gemm_policy() != "hipblaslt" and
                ops.native_gemm_ok(T, w.shape[0], w.shape[1], 0))

    def _act(self, e, name: str, T: int, K: int, packed: bool):
        if packed:
            return e(f"{name}_p{K}", (ops.packed_numel(T, K),))
        return e(f"{name}_{K}", (T, K))

    def _mm(self, x, w, wp, T: int, packed: bool, out):
        if packed:
            return ops.linear(x, None, wp=wp, a_rows=T, out=out)
        return ops.linear(x, w, out=out, tiles=True)

    def _add(self, y_in, w, wp, packed: bool, T: int, res, gain, nxt, e, experts=None, join=None, keep=True):
        """Close a sublayer: add y = y_in w^T to the stream (``keep`` False: replace it) and write the next sublayer's
        ``xb``.  ``gain``: the sublayer's own norm gain, ``nxt``: what opens the next one (``_entry``; None after the last).  A packed projection with a split-K
        form hands its fp32 slabs straight to the kernel (no reduce launch, no rounding of y).  ``experts``: routed
        experts' rows that belong to y (``y_in`` None: the only ones); ``join``: the stream that waits for them."""
        if y_in is None:
            y = None
        elif packed and ops.rwk_split(T, w.shape[0], w.shape[1]) > 0:
            y = ops.linear_partials(y_in, T, wp=wp, out=e("y", (T, self.W)), rot=ops.partials_turned(*w.shape))
        else:
            y = self._mm(y_in, w, wp, T, packed, e("y", (T, self.W)))
        if join is not None:
            join.wait_stream(self.side)
        if self.pre:
            n = nxt or {"gain": None, "xb": None, "packed": False, "shift": None, "copy": 0}
            mops.add_norm(y, res, self.mult if keep else 1.0, n["gain"], self.eps, n["xb"], self.center, packed=n["packed"],
                          experts=experts, groups=self.groups, shift=n["shift"], keep=keep, copy=n["copy"])
        else:
            hops.residual_norm(y, res, gain, self.eps, nxt["xb"], packed=nxt["packed"])

    def _enter(self, res, nxt) -> None:
        """``xb`` of a sublayer from the stream alone."""
        if nxt is None:
            return
        if self.pre:
            mops.add_norm(None, res, 0.0, nxt["gain"], self.eps, nxt["xb"], self.center, packed=nxt["packed"],
                          groups=self.groups, shift=nxt["shift"], copy=nxt["copy"])
            return
        y = res.to(self.ex.dtype)
        if nxt["packed"]:
            ops.pack_act(y, out=nxt["xb"])
        else:
            nxt["xb"].copy_(y)

    def _entry(self, i: int, m, e, inject: bool = True):
        """What the kernel ahead of layer ``i`` writes: the norm that its input projection reads (moved towards the previous
        token's where the layer shifts), or, ahead of a loop's pass, the stream's half of [stream, embedding].  After the last
        layer of a pre-norm stream the head's input where every row has logits (a launch less in a decode step: 8 of Nuvorax' 4345 ->
        4318 us), else None."""
        layers, T, W = self.ex.w.layers, m["T"], self.W
        if i >= len(layers):
            if m["head"]:
                pk = self._packed(T, self.ex.w.lm_head, self.ex.w.lm_head_p)
                return {"gain": self.ex.w.final_norm, "xb": self._act(e, "fn", T, W, pk), "packed": pk, "shift": None, "copy": 0}
            return None if self.pre else {"gain": None, "xb": e(f"xb_{W}", (T, W)), "packed": False}
        lay = layers[i]
        if inject and self._spec(i).inject:
            pk = self._packed(T, self.ex.w.loop_in, self.ex.w.loop_in_p)
            return {"gain": None, "xb": self._act(e, "cat", T, 2 * W, pk), "packed": pk, "shift": None, "copy": 2 * W}
        pk, shift = self._packed(T, lay.w_in, lay.w_in_p), None
        if lay.shift is not None:
            rows = self.ex.state.layer(self.state_at[i])[-1]
            scratch = None
            if m["plan"] is not None and self.ex.device.type == "cuda":
                scratch = (e("shift_first", (rows.shape[0], W), torch.float32),
                           e("shift_stats", (T, self.groups), torch.float32))
            shift = (lay.shift, rows, m["q_seq"], m["q_ctx"], scratch)
        return {"gain": lay.n1, "xb": self._act(e, "xb", T, W, pk), "packed": pk, "shift": shift, "copy": 0}

    def _spec(self, i: int):
        """Spec of layer run ``i`` (runs of one checkpoint layer share the weight object, not the run's own fields)."""
        return self.ex.cfg.layers[self.ex.start + i]

    # ------------------------------------------------------------------ mixers: z -> the output projection's input
    def _hgrn2(self, i, lay, z, o, pko, m, e):
        hops.hgrn2(z, lay.f_bias, lay.f_lower, lay.o_norm, self.ex.state.layer(self.state_at[i])[0], m["q_seq"], m["q_ctx"],
                   o, self.eps, plan=m["plan"], packed=pko)

    def _retention(self, i, lay, z, o, pko, m, e):
        sp = lay.spec
        mops.retention(z, self.rope[self._rope_key(sp)], lay.log_decay, self.ex.state.layer(self.state_at[i])[0],
                       m["q_seq"], m["q_ctx"], o, self.eps, plan=m["linear"], packed=pko)

    def _mlstm(self, i, lay, z, o, pko, m, e):
        state, aux = self.ex.state.layer(self.state_at[i])
        mops.mlstm(z, lay.gate_bias, lay.spec.gate_cap, lay.o_norm, state, aux, m["q_seq"], m["q_ctx"], o, self.eps,
                   plan=m["linear"], packed=pko)

    def _attention(self, i, lay, z, o, pko, m, e):
        ex, sp, T, plan = self.ex, lay.spec, m["T"], m["plan"]
        kv, rk = ex.cache.layer(self.cache_at[i])
        qn = e(f"qn{sp.out_cols}", (T, sp.out_cols))
        hops.talk_prep(z, lay.w_qk, qn, kv, rk, m["slots"], self.eps)
        tb = self.talk_block.get((sp.heads, sp.kv_heads, sp.dim), 0)
        blocks = parts = ws = None
        if tb and plan is not None:
            blocks = plan["blocks"][tb]
        elif tb:
            parts = hops.talk_parts(T, sp.heads, sp.kv_heads, sp.dim, min(m["span"], sp.chunk), ex._n_cu)
            if parts[1] > 1:
                ws = e("talk_ws", (parts[1] * T * sp.heads * (sp.dim + 2),), torch.float32)
        hops.talk_attention(z, qn, lay.talk, kv, rk, m["table"], m["q_seq"], m["q_ctx"], o, sp.chunk, sp.scale,
                            packed=pko, sigma=lay.sigma, blocks=blocks, parts=parts, ws=ws)

    def _latent(self, i, lay, z, o, pko, m, e):
        ex, sp, T, plan = self.ex, lay.spec, m["T"], m["plan"]
        kv, _ = ex.cache.layer(self.cache_at[i])
        rope = self.rope[self._rope_key(sp)]
        pkq = self._packed(T, lay.w_uq, lay.w_uq_p)
        cq = self._act(e, "cq", T, sp.q_rank, pkq)
        mops.latent_prep(z, lay.q_norm, lay.c_norm, cq, kv, m["slots"], m["q_ctx"], rope, self.eps, packed=pkq)
        q = self._mm(cq, lay.w_uq, lay.w_uq_p, T, pkq, e(f"q{sp.q_rows}", (T, sp.q_rows)))
        key = self._latent_key(sp)
        lp = plan["latent"][key] if plan is not None and self.latent_block.get(key, 0) else None
        if lp is not None and lp["wide"] is not None:  # long portions: every head's own keys and values
            wd = lp["wide"]
            lat = mops.latent_gather(kv, wd["idx"], e("lat_rows", (wd["idx"].numel(), kv.shape[3])))
            own = e("lat_kv", (lat.shape[0], lay.w_ukv.shape[0]))
            torch.mm(lat[:, :sp.kv_rank], lay.w_ukv.t(), out=own)
            mops.latent_wide(q, own, lat, lay.sink, rope, m["q_ctx"], o, sp.dim, sp.vdim, sp.scale, wd["blk"],
                             wd["waves"], packed=pko)
            if lp["blocks"] is None:
                return
        kw = {}
        if self.latent_block.get(key, 0):
            H, C, R = sp.heads, sp.kv_rank, sp.rot_dim
            kw = dict(u=e("lat_u", (T, H, C + R)), oc=e("lat_oc", (T, H, C)))
            if lp is not None:
                kw.update(blocks=lp["blocks"], rows=lp["rows"], parts=lp["parts"])
            else:
                kw["parts"] = mops.latent_parts(T * -(-H // 32), m["span"], ex._n_cu)
            if kw["parts"][1] > 1:
                kw["ws"] = e("lat_ws", (kw["parts"][1] * T * H * (C + 2),), torch.float32)
        mops.latent_attention(q, lay.w_uk, lay.w_uv, lay.sink, rope, kv, m["table"], m["q_seq"], m["q_ctx"], o, sp.scale,
                              packed=pko, **kw)

    def _mixed(self, i, lay, z, o, pko, m, e):
        ex, sp, T = self.ex, lay.spec, m["T"]
        kv, _ = ex.cache.layer(self.cache_at[i])
        rope, vrope = self.rope[self._rope_key(sp)], self.rope[(sp.rot_base, sp.vdim, None)]
        qn = e(f"qn{sp.heads * sp.dim}", (T, sp.heads * sp.dim))
        ff = (self._ff_kind(sp), sp.ff, lay.ffn_block or 1, sp.mix_rows, sp.limit) if sp.parallel and sp.ff else None
        xops.mixed_prep(z, lay.q_gain, lay.k_gain, qn, kv, m["slots"], m["q_ctx"], rope, vrope, o, sp.o_cols, self.eps,
                        ff=ff, packed=pko)
        (tb, dec), kw, plan, f32 = self.mixed_ok.get(self._mixed_key(sp), (0, False)), {}, m["plan"], torch.float32
        H, V = sp.heads, sp.vdim
        if plan is not None and tb:
            mp = plan["mixed"][tb]
            parts = xops.fit_splits(mp["parts"], T * H * V * 4, MIXED_WS_BYTES)
            kw = dict(form=1, blocks=mp["blocks"], parts=parts, sum_parts=mp["sums"],
                      sums=e("mix_sums", (mp["sums"][1] * T * H,), f32))
            if parts[1] > 1:
                kw["part"] = e("mix_part", (parts[1] * T * H * V,), f32)
        elif plan is None and dec:
            parts = xops.mixed_parts(T, m["span"], ex._n_cu)
            kw = dict(form=2, parts=parts, sums=e("mix_sums", (parts[1] * T * H,), f32),
                      part=e("mix_part", (parts[1] * T * sp.kv_heads * H * V,), f32))
        xops.mixed_attention(z, qn, lay.talk, kv, m["table"], m["q_seq"], m["q_ctx"], vrope, o, sp.o_cols, sp.scale,
                             sp.softcap, packed=pko, **kw)

    # mixers that may be part of a pair: z, and columns [col, ..) of o [T, K]
    def _window(self, i, sp, part, z, o, col, K, mult, states, pko, m, e):
        ex, T = self.ex, m["T"]
        kv, _ = ex.cache.layer(self.cache_at[i])
        qn = e(f"qn{sp.heads * sp.dim}", (T, sp.heads * sp.dim))
        wops.window_prep(z, qn, kv, m["slots"], m["q_ctx"], self.rope[self._rope_key(sp)], sp.vdim, sp.neighbours,
                         self.eps if sp.qk_norm else None)
        kw, plan = {}, m["plan"]
        rows = self.window_rows.get(self._window_key(sp), 0) if col % 4 == 0 and K % 4 == 0 else 0
        if rows and plan is not None:
            blocks, rows = plan["window"][self._window_key(sp), sp.reach]
            kw = dict(form=1, blocks=blocks, parts=(rows, 1))
        elif rows:
            parts = wops.window_parts(T * sp.kv_heads, min(m["span"], sp.reach), ex._n_cu)
            kw = dict(form=2, parts=parts)
            if parts[1] > 1:
                kw["ws"] = e("window_ws", (parts[1] * T * sp.heads * (sp.vdim + 2),), torch.float32)
        wops.window_attention(qn, part["head"], kv, m["table"], m["q_seq"], m["q_ctx"], o, col, K, sp.vdim, sp.scale, mult,
                              sp.window, sp.keep_first, sp.weights == "sigmoid", packed=pko, **kw)

    def _gated(self, i, sp, part, z, o, col, K, mult, states, pko, m, e):
        head = {"gla": (sp.tau,), "gated_delta": (sp.kv_heads,), "mamba2": (sp.kv_heads, sp.norm_groups)}[sp.mixer]
        getattr(gops, sp.mixer)(z, part, *head, *states, m["q_seq"], m["q_ctx"], o, col, K, self.eps, plan=m["gated"],
                                packed=pko, e=e)

    def _parts(self, i, lay, z, o, pko, m, e):
        """A mixer of ``parts``, or a pair's two side by side."""
        spec, row, col, at = lay.spec, 0, 0, 0
        states = self.ex.state.layer(self.state_at[i]) if spec.state_shapes else ()
        scales = (spec.left_scale, spec.right_scale) if spec.mixer == "pair" else (1.0,)
        for sp, part, mult in zip(spec.mixers, lay.parts, scales):
            n = len(sp.state_shapes) - (1 if sp.shift else 0)
            self.PART[sp.mixer](self, i, sp, part, z[:, row:row + sp.mix_rows], o, col, spec.o_cols, mult,
                                states[at:at + n], pko, m, e)
            row, col, at = row + sp.mix_rows, col + sp.out_cols, at + n

    PART = {"window_attention": _window, "gated_delta": _gated, "mamba2": _gated, "gla": _gated}
    MIX = {"hgrn2": _hgrn2, "retention": _retention, "mlstm": _mlstm, "attention": _attention,
           "latent_attention": _latent, "mixed_attention": _mixed, "pair": _parts, **dict.fromkeys(PART, _parts)}

    @staticmethod
    def _ff_kind(sp):
        """Activation of a feed-forward that the decode GEMM's epilogues do not cover."""
        return "gated_glu" if sp.moe else sp.ffn

    def _fork(self, lay, x, packed: bool, m, e):
        """``_experts`` of a parallel layer beside its mixer: decode steps run them on a stream of their own (both paths
        are chains of short launches), joined before the layer closes."""
        if self.side is None or m["plan"] is not None:
            return self._experts(lay, x, packed, m, e), None
        cur = torch.cuda.current_stream()
        self.side.wait_stream(cur)
        with torch.cuda.stream(self.side):
            return self._experts(lay, x, packed, m, e), cur

    def _experts(self, lay, x, packed: bool, m, e):
        """Routed experts of the rows ``x``: (rows, row of every choice, weights)."""
        c = eops.choose(x, lay.w_r, m["q_ctx"], lay.spec.moe, e, packed=packed)
        y = eops.experts(x, c, lay.w_eu, lay.w_ed, lay.w_eu_p, lay.w_ed_p, lay.expert_block, e, packed=packed)
        return y, c.slot, c.weights

    def _ffn(self, lay, xu, pku: bool, T: int, e):
        """Feed-forward activation (what ``w_down`` reads) and whether it is packed."""
        sp = lay.spec
        if lay.w_down is None:  # routed experts alone
            return None, False
        pkd = self._packed(T, lay.w_down, lay.w_down_p)
        a = self._act(e, "act", T, sp.ff, pkd)
        rows = lay.w_up.shape[0]
        if sp.moe or sp.ffn == "gelu":
            u = self._mm(xu, lay.w_up, lay.w_up_p, T, pku, e(f"u{rows}", (T, rows)))
            return xops.ffn_act(u, a, self._ff_kind(sp), sp.ff, lay.ffn_block or 1, sp.limit, packed=pkd), pkd
        glu = sp.glu
        fused = dict(epilogue=1, glu_limit=sp.limit) if glu else dict(epilogue=4)
        if pku and (not glu or lay.ffn_block == ops.GU_BLOCK) and \
                ops.native_gemm_ok(T, rows, self.W, fused["epilogue"], pkd):
            ops.linear(xu, None, wp=lay.w_up_p, a_rows=T, out=a, out_packed=pkd, **fused)  # in the GEMM's epilogue
            return a, pkd
        if not pku and not pkd and (not glu or lay.ffn_block == ops.GU_BLOCK) and \
                ops.gemm_policy() != "hipblaslt" and ops.prompt.ok(xu, lay.w_up, fused["epilogue"]):
            return ops.linear(xu, lay.w_up, out=a, tiles=True, **fused), False
        u = self._mm(xu, lay.w_up, lay.w_up_p, T, pku, e(f"u{rows}", (T, rows)))
        if glu:
            mops.clamped_glu(u, a, lay.ffn_block, sp.limit, packed=pkd)
        else:
            hops.relu2(u, a, packed=pkd)
        return a, pkd

    # ------------------------------------------------------------------ the step
    def forward(self, x, positions, slots, q_seq, q_ctx, last_rows, T, bufs: Optional[dict] = None, plan=None,
                span: int = 0, prompt=None, every: bool = False):
        """``plan``: the ragged step's ``plan`` (None: a decode step, every row one token); ``span``: most keys a
        query sees.  Returns the fp32
        residual rows [T, W] (non-last stage) or the logits of ``last_rows`` (``every``: which are all rows in order)."""
        ex, W, eps = self.ex, self.W, self.eps
        dev, dt = ex.device, ex.dtype
        layers = ex.w.layers
        cache: dict = {} if bufs is None else bufs

        def e(name, shape, dtype=dt):
            t = cache.get(name)
            if t is None or tuple(t.shape) != tuple(shape) or t.dtype != dtype:
                t = cache[name] = torch.empty(shape, dtype=dtype, device=dev)
            return t

        m = {"T": T, "slots": slots, "q_seq": q_seq, "q_ctx": q_ctx, "plan": plan, "span": span,
             "linear": plan.get("linear") if plan else None, "gated": plan.get("gated") if plan else None,
             "table": ex.sessions.table_dev, "head": every and self.pre and ex.is_last and bool(layers)}
        res = torch.empty(T, W, dtype=torch.float32, device=dev)
        nxt, res0 = self._entry(0, m, e), None
        if ex.cfg.embed_norm:
            res0 = self._embed(x, res, e, T)
            self._enter(res, nxt)
        elif not ex.is_first:
            res.copy_(x)
            if layers:
                self._enter(res, nxt)
        elif not self.pre:
            hops.embed_pos(x, ex.w.embed, positions, self.inv, res, nxt["xb"], packed=nxt["packed"])
        elif layers:
            mops.embed_norm(x, ex.w.embed, res, nxt["gain"], eps, nxt["xb"], self.center, packed=nxt["packed"],
                            scale=ex.cfg.embed_scale)
        else:
            res.copy_(ex.w.embed[x.long()].float() * ex.cfg.embed_scale)
        for i, lay in enumerate(layers):
            sp = lay.spec
            if prompt is not None:  # deep prompt: the block input += prompt[i]
                res.index_add_(0, prompt[0], prompt[1][i].float())
                self._enter(res, nxt)
            if self._spec(i).inject:
                nin, nxt = nxt, self._entry(i, m, e, inject=False)
                self._add(nin["xb"], ex.w.loop_in, ex.w.loop_in_p, nin["packed"], T, res, None, nxt, e, keep=False)
            xb, pk = nxt["xb"], nxt["packed"]
            rows, join = self._fork(lay, xb, pk, m, e) if sp.moe and sp.parallel else (None, None)
            z = self._mm(xb, lay.w_in, lay.w_in_p, T, pk, e(f"z{sp.in_rows}", (T, sp.in_rows)))
            pko = self._packed(T, lay.w_o, lay.w_o_p)
            o = self._act(e, "o", T, sp.o_cols, pko)
            self.MIX[sp.mixer](self, i, lay, z, o, pko, m, e)
            if (sp.ff or sp.moe) and not sp.parallel:
                pku = lay.w_up is not None and self._packed(T, lay.w_up, lay.w_up_p)
                xu = self._act(e, "xb", T, W, pku)
                self._add(o, lay.w_o, lay.w_o_p, pko, T, res, lay.n1,
                          {"gain": lay.n2, "xb": xu, "packed": pku, "shift": None, "copy": 0}, e)
                a, pkd = self._ffn(lay, xu, pku, T, e)
                rows = self._experts(lay, xu, pku, m, e) if sp.moe else None
                nxt = self._entry(i + 1, m, e)
                self._add(a, lay.w_down, lay.w_down_p, pkd, T, res, lay.n2, nxt, e, rows)
            else:
                nxt = self._entry(i + 1, m, e)
                self._add(o, lay.w_o, lay.w_o_p, pko, T, res, lay.n1, nxt, e, rows, join)
        if not ex.is_last:
            return torch.cat([res, res0], 1) if ex.cfg.injects else res
        S, V = last_rows.numel(), ex.cfg.vocab_size
        head = ex.w.lm_head
        if S == 0:
            return torch.empty(0, V, dtype=dt, device=dev)
        pkh = self._packed(S, head, ex.w.lm_head_p)
        fn = self._act(e, "fn", S, W, pkh)
        if m["head"]:
            pass  # (the last layer closed with it)
        elif self.pre:
            mops.rows_norm(res, last_rows, ex.w.final_norm, eps, fn, self.center, packed=pkh, groups=self.groups)
        else:
            hops.rows_norm(res, last_rows, ex.w.final_norm, eps, fn, packed=pkh)
        logits = self._mm(fn, head, ex.w.lm_head_p, S, pkh, torch.empty(S, head.shape[0], dtype=dt, device=dev))
        if ex.cfg.logit_softcap > 0:
            mops.softcap(logits, ex.cfg.logit_softcap)
        return logits[:, :V]

    def _embed(self, x, res, e, T: int):
        """The normed embedding into the stream (first stage) or the stream that came in; returns the embedding where later
        layers or stages read it, its activation copy in place in [stream, embedding]."""
        ex, W = self.ex, self.W
        here = any(self._spec(i).inject for i in range(len(ex.w.layers)))
        cat, pk = None, False
        if here:
            pk = self._packed(T, ex.w.loop_in, ex.w.loop_in_p)
            cat = self._act(e, "cat", T, 2 * W, pk)
        if ex.is_first:
            mops.embed_rows_norm(x, ex.w.embed, res, ex.w.embed_norm, self.eps, self.groups, cat, W, 2 * W, pk)
            return res.clone() if ex.cfg.injects and not ex.is_last else None
        res.copy_(x[:, :W])
        if not ex.cfg.injects:
            return None
        if here:
            mops.put_columns(x[:, W:], cat, W, 2 * W, pk)
        return x[:, W:]

    # ------------------------------------------------------------------ plans
    def plan(self, ntoks, starts, rows, up=None) -> dict:
        """Device description of a ragged step (not one token per session): ``ntoks`` tokens per session after the
        ``starts`` it already holds; ``rows``: the sessions' rows of the block table; ``up``: host array -> device tensor, there
        when the step runs."""
        if self.ex.device.type != "cuda":
            return {}
        up = up or (lambda a: torch.from_numpy(a).to(self.ex.device, non_blocking=True))
        p = {"blocks": {tb: up(hops.talk_blocks(ntoks, tb)) for tb in set(self.talk_block.values()) if tb}}
        if self.rec_fill:
            h = hops.hgrn2_plan(ntoks, self.rec_fill[0], self.ex._n_cu, per_cu=self.rec_fill[1])
            p.update(seqs=up(h["seqs"]), seg=up(h["seg"]), multi=up(h["multi"]) if h["slots"] else None,
                     slots=h["slots"])
        if self.lin_fill:
            h = mops.linear_plan(ntoks, self.lin_fill[0], self.ex._n_cu, per_cu=self.lin_fill[1])
            p["linear"] = {"seqs": up(h["seqs"]), "seg": up(h["seg"]), "slots": h["slots"],
                           "multi": up(h["multi"]) if h["slots"] else None}
        p["window"] = {}
        for key, reach in self.windows:
            rep, rows = key[0] // key[1], self.window_rows[key]
            if rows:
                rows = wops.window_rows(ntoks, rep, key[1], rows, self.ex._n_cu)
                p["window"][key, reach] = up(wops.window_blocks(ntoks, starts, rep, rows, reach)), rows
        if self.gated:
            c = gops.chunk_plan(ntoks, self.gated_waves, self.ex._n_cu)
            p["gated"] = {k: up(v) for k, v in c.items()}
        p["mixed"] = {}
        for tb in {t for t, _ in self.mixed_ok.values() if t}:
            blk = xops.mixed_blocks(ntoks, starts, tb)
            sums, parts = xops.prompt_splits(blk, ntoks, starts, self.ex._n_cu)
            p["mixed"][tb] = {"blocks": up(blk), "sums": sums, "parts": parts}
        p["latent"] = {key: self._latent_plan(key, tb, ntoks, starts, rows, up)
                       for key, tb in self.latent_block.items() if tb}
        return p

    def _latent_plan(self, key, tb, ntoks, starts, rows, up) -> dict:
        """Which sessions' tokens go which way: long portions on the wide form, the rest in query blocks of the other."""
        H, D, R, V, C = key
        ntoks, starts = np.asarray(ntoks), np.asarray(starts)
        off = np.concatenate([[0], np.cumsum(ntoks)[:-1]])
        wide = mops.latent_wide_plan(ntoks, starts, H, D, self.ex._n_cu, LATENT_KV_BYTES // (2 * H * (D + V))) \
            if mops.latent_wide_ok(D, R, V, C) else None
        out = {"wide": None, "blocks": None, "rows": None, "parts": (0, 1)}
        rest = np.arange(len(ntoks))
        if wide is not None:
            pick, blk, waves = wide
            ps, table = self.ex.cache.page_size, self.ex.sessions.table
            idx = np.concatenate([(table[rows[i], np.arange(n) // ps].astype(np.int64) * ps + np.arange(n) % ps)
                                  for i in pick for n in [int(starts[i] + ntoks[i])]])
            out["wide"] = {"idx": up(idx), "blk": up(blk), "waves": waves}
            rest = np.setdiff1d(rest, pick)
        rest = rest[ntoks[rest] > 0]
        if not rest.size:
            return out
        blk = np.concatenate([hops.talk_blocks(ntoks[i:i + 1], tb) + [[off[i]], [0]] for i in rest], 1).astype(np.int32)
        if wide is not None:
            out["rows"] = up(np.concatenate([np.arange(off[i], off[i] + ntoks[i]) for i in rest]).astype(np.int32))
        n, T = int((starts + ntoks)[rest].max()), int(ntoks.sum())
        parts = mops.latent_parts(blk.shape[1] * -(-H // 32), n, self.ex._n_cu)
        if parts[1] > 1 and parts[1] * T * H * (C + 2) * 4 <= LATENT_WS_BYTES:
            out["parts"] = parts
        out["blocks"] = up(np.ascontiguousarray(blk))
        return out

    def span(self, max_ctx: int) -> int:
        """Most keys a decode query of context <= max_ctx can see."""
        return max(1, min(int(max_ctx), self.max_chunk))
