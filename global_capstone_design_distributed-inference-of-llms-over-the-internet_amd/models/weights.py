"""Per-stage weights: synthetic random init or HF checkpoint loading of ONLY the stage's keys.

The reference loads the whole HF model on CPU in every stage process and then prunes
``model.layers`` (reference src/llama_partition.py:495-530); the vendored Petals server
instead reads only ``model.layers.{i}.*`` from the sharded checkpoint
(reference petals/server/from_pretrained.py:35-128).  Here a stage reads only its own
blocks (plus embeddings / final norm / lm_head when its role needs them) straight from
the safetensors shards, and lays them out for the MI355X kernels:

* q/k/v fused into one ``qkv`` matrix [(nh + 2 nkv) * D, H] -> one GEMM per layer;
* gate/up fused into ``gate_up`` [2F, H] with rows interleaved in 16-row blocks
  ([g0..g15, u0..u15, g16..g31, ...]) so the GEMM epilogue can apply SwiGLU in registers;
* everything resident on the GPU (no per-forward CPU<->GPU streaming, unlike
  src/llama_partition.py:169-180, :233-293 of the reference).

Random init is deterministic per (seed, block index): a model split into any number of
stages gets bit-identical weights, which the pipeline-equivalence tests rely on.
"""
from __future__ import annotations

import dataclasses
import glob
import json
import os
from typing import Dict, List, Optional, Tuple

import torch

from .config import PAIRED, LayerSpec, ModelConfig
from ..ops.reference import GU_BLOCK

INIT_STD = 0.02


def interleave_gate_up(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    F, H = gate.shape
    assert F % GU_BLOCK == 0, "intermediate_size must be a multiple of 16"
    return torch.stack([gate.view(F // GU_BLOCK, GU_BLOCK, H), up.view(F // GU_BLOCK, GU_BLOCK, H)], 1).reshape(2 * F, H)


def split_gate_up(gu: torch.Tensor):
    F2, H = gu.shape
    v = gu.view(F2 // (2 * GU_BLOCK), 2, GU_BLOCK, H)
    return v[:, 0].reshape(F2 // 2, H), v[:, 1].reshape(F2 // 2, H)


@dataclasses.dataclass
class LlamaLayer:
    input_norm: torch.Tensor
    qkv: torch.Tensor
    o: torch.Tensor
    post_norm: torch.Tensor
    gate_up: torch.Tensor
    down: torch.Tensor
    # fragment-native packed copies for the decode GEMM (ops.pack_weight); None until packed
    qkv_p: Optional[torch.Tensor] = None
    o_p: Optional[torch.Tensor] = None
    gate_up_p: Optional[torch.Tensor] = None
    down_p: Optional[torch.Tensor] = None
    # fp8 e4m3 W8A8 copies (ops.pack_weight_fp8): packed uint8 + per-output-channel fp32 scale
    qkv_q: Optional[torch.Tensor] = None
    qkv_s: Optional[torch.Tensor] = None
    o_q: Optional[torch.Tensor] = None
    o_s: Optional[torch.Tensor] = None
    gate_up_q: Optional[torch.Tensor] = None
    gate_up_s: Optional[torch.Tensor] = None
    down_q: Optional[torch.Tensor] = None
    down_s: Optional[torch.Tensor] = None
    # fp8 W8A16 copies (ops.w8_from_fp8: the bf16 fragment order at 1 byte per weight) + fp32
    # per-output-channel scales, for the fused-norm decode GEMMs of an fp8 stage
    qkv_w8: Optional[torch.Tensor] = None
    qkv_ws: Optional[torch.Tensor] = None
    o_w8: Optional[torch.Tensor] = None
    o_ws: Optional[torch.Tensor] = None
    gate_up_w8: Optional[torch.Tensor] = None
    gate_up_ws: Optional[torch.Tensor] = None
    down_w8: Optional[torch.Tensor] = None
    down_ws: Optional[torch.Tensor] = None
    # Mixtral sparse-MoE block (HF MixtralSparseMoeBlock): ``router`` [E, H]; gate_up / down
    # (and their packed copies) are then stacked per expert: [E, 2F, H] / [E, H, F]
    router: Optional[torch.Tensor] = None
    folded: bool = False  # qkv_p / gate_up_p carry the input / post-attention norm weights

    PROJ = ("qkv", "o", "gate_up", "down")

    @property
    def moe(self) -> bool:
        return self.router is not None

    @property
    def fp8(self) -> bool:
        return self.qkv_q is not None or self.qkv_w8 is not None

    @property
    def w8(self) -> bool:
        return self.qkv_w8 is not None

    def dense(self, name: str, dtype=torch.bfloat16) -> torch.Tensor:
        """Row-major weight ``name`` (dequantized on the fly when only an fp8 copy is kept; a
        W8A16 layer's qkv / gate_up then carry the folded norm weights, see ``folded``)."""
        w = getattr(self, name)
        if w is not None:
            return w
        from .. import ops

        if getattr(self, name + "_w8") is not None:
            return ops.unpack_weight_w8(getattr(self, name + "_w8"), getattr(self, name + "_ws"), dtype)
        return ops.unpack_weight_fp8(getattr(self, name + "_q"), getattr(self, name + "_s"), dtype)


@dataclasses.dataclass
class GPT2Layer:
    ln1_w: torch.Tensor
    ln1_b: torch.Tensor
    attn_w: torch.Tensor  # [3H, H] (HF Conv1D weight transposed)
    attn_b: torch.Tensor
    proj_w: torch.Tensor
    proj_b: torch.Tensor
    ln2_w: torch.Tensor
    ln2_b: torch.Tensor
    fc_w: torch.Tensor
    fc_b: torch.Tensor
    fc2_w: torch.Tensor
    fc2_b: torch.Tensor


@dataclasses.dataclass
class HybridLayer:
    """A layer of a hybrid decoder.  GEMM weights have the stage's dtype; norms, gates and mixing matrices
    are fp32.  ``w_in`` fuses the mixer's input projections (``LayerSpec.in_rows``); ``*_p`` are the
    fragment-native copies for the decode GEMM where the shape allows one.  In a parallel layer the feed-forward's
    projections are part of ``w_in`` (rows from ``mix_rows`` on) and ``w_o`` (columns from ``out_cols`` on).  Expert
    weights are held in one form: packed (``w_eu_p``, ``w_ed_p``) where the MFMA kernels cover the shape."""
    spec: LayerSpec
    w_in: torch.Tensor                       # [in_rows, W]
    w_o: torch.Tensor                        # [W, heads * vdim]
    n1: torch.Tensor                         # [W] norm gain of the mixer's output x layer scale, or of its input
    w_up: Optional[torch.Tensor] = None      # [ff, W]; gated: [2 ff, W] gate and up rows in blocks of ``ffn_block``
    w_down: Optional[torch.Tensor] = None    # [W, ff]
    n2: Optional[torch.Tensor] = None        # [W]
    f_bias: Optional[torch.Tensor] = None    # hgrn2 [heads * dim]
    f_lower: Optional[torch.Tensor] = None   # hgrn2 [heads * dim]
    o_norm: Optional[torch.Tensor] = None    # hgrn2 [vdim]
    w_qk: Optional[torch.Tensor] = None      # attention [heads * dim]: query norm x its kv head's key norm
    talk: Optional[torch.Tensor] = None      # attention [heads, heads]
    sigma: Optional[torch.Tensor] = None     # attention [heads]: talk @ the heads' distance slopes
    q_norm: Optional[torch.Tensor] = None    # latent_attention [q_rank]
    c_norm: Optional[torch.Tensor] = None    # latent_attention [kv_rank]
    w_uq: Optional[torch.Tensor] = None      # latent_attention [heads * (dim + rot_dim), q_rank]
    w_uk: Optional[torch.Tensor] = None      # latent_attention [heads, kv_rank, dim]: a query head into latent space
    w_uv: Optional[torch.Tensor] = None      # latent_attention [heads, vdim, kv_rank]: a head's latent sum to its value
    w_ukv: Optional[torch.Tensor] = None     # latent_attention [heads * (dim + vdim), kv_rank]: keys and values, by head
    sink: Optional[torch.Tensor] = None      # latent_attention [heads]
    log_decay: Optional[torch.Tensor] = None  # retention [heads]: log2 of the decay
    gate_bias: Optional[torch.Tensor] = None  # mlstm [2, heads]: input and forget gate
    q_gain: Optional[torch.Tensor] = None    # mixed_attention [dim]
    k_gain: Optional[torch.Tensor] = None    # mixed_attention [dim]
    w_r: Optional[torch.Tensor] = None       # experts: router [experts, W]
    w_eu: Optional[torch.Tensor] = None      # experts [experts, 2 ff, W]: gate and up rows in blocks of ``expert_block``
    w_ed: Optional[torch.Tensor] = None      # experts [experts, W, ff]
    expert_block: int = 0
    w_eu_p: Optional[torch.Tensor] = None    # [experts, 2 ff / 16, W / 32, 64, 8]
    w_ed_p: Optional[torch.Tensor] = None    # [experts, W / 16, ff / 32, 64, 8]
    ffn_block: int = 0                       # gated feed-forward: rows of a gate / up block of ``w_up``
    w_in_p: Optional[torch.Tensor] = None
    w_o_p: Optional[torch.Tensor] = None
    w_up_p: Optional[torch.Tensor] = None
    w_down_p: Optional[torch.Tensor] = None
    w_uq_p: Optional[torch.Tensor] = None
    shift: Optional[torch.Tensor] = None     # [W] token shift
    # what the mixers of ``spec.mixers`` read besides the projections (the first, then a pair's second), by name
    parts: Tuple[Dict[str, torch.Tensor], ...] = ()

    GEMMS = ("w_in", "w_o", "w_up", "w_down", "w_uq")


@dataclasses.dataclass
class StageWeights:
    cfg: ModelConfig
    start: int
    end: int
    layers: list
    embed: Optional[torch.Tensor] = None        # [V, H] (gpt2: wte)
    pos_embed: Optional[torch.Tensor] = None    # gpt2 wpe [P, H]
    final_norm: Optional[torch.Tensor] = None   # llama [H]; gpt2 ln_f weight
    final_norm_b: Optional[torch.Tensor] = None  # gpt2 ln_f bias
    lm_head: Optional[torch.Tensor] = None      # [V, H]
    lm_head_p: Optional[torch.Tensor] = None    # packed lm_head (V padded to a multiple of 16)
    lm_head_folded: bool = False                # lm_head_p carries final_norm in its K columns
    embed_norm: Optional[torch.Tensor] = None   # hybrid decoders: gain of the embedding's norm [H]
    loop_in: Optional[torch.Tensor] = None      # hybrid decoders: projection of [stream, embedding] ahead of a pass [H, 2 H]
    loop_in_p: Optional[torch.Tensor] = None

    @property
    def has_embed(self) -> bool:
        return self.embed is not None

    @property
    def has_head(self) -> bool:
        return self.lm_head is not None

    def nbytes(self) -> int:
        n = 0
        for t in self.tensors():
            n += t.numel() * t.element_size()
        return n

    def pack_for_decode(self, fold_norms: bool = False) -> None:
        """Add fragment-native copies of every projection (MI355X decode GEMM layout).

        The row-major weights stay for the hipBLASLt prefill path: 2x weight bytes, which
        288 GB of HBM affords (13.5 GB -> 27 GB for Llama-2-7B on one GPU).

        ``fold_norms``: the packed qkv / gate_up copies carry the RMSNorm weight folded into
        their K columns (W' = W diag(g)) for the fused-norm decode path, whose GEMMs take the raw
        residual stream and apply rsqrt(mean x^2) per row in the epilogue (ops/csrc/gemm.hip).
        """
        from .. import ops

        for lay in self.layers:
            if isinstance(lay, HybridLayer):
                for name in HybridLayer.GEMMS:
                    w = getattr(lay, name)
                    if w is not None and w.dtype == torch.bfloat16 and w.shape[0] % 16 == 0 and w.shape[1] % 128 == 0 \
                            and getattr(lay, name + "_p") is None:
                        setattr(lay, name + "_p", ops.pack_weight(w))
                if lay.w_eu is not None and ops.expert_mfma_ok(lay.spec.moe.ff, self.cfg.hidden_size, lay.w_eu.dtype):
                    lay.w_eu_p = torch.stack([ops.pack_weight(w) for w in lay.w_eu])
                    lay.w_ed_p = torch.stack([ops.pack_weight(w) for w in lay.w_ed])
                    lay.w_eu = lay.w_ed = None
            if isinstance(lay, LlamaLayer) and lay.qkv_p is None and lay.qkv is not None:
                if fold_norms and not lay.moe:
                    lay.qkv_p = ops.pack_weight((lay.qkv.float() * lay.input_norm.float()[None, :])
                                                .to(lay.qkv.dtype).contiguous())
                    lay.o_p = ops.pack_weight(lay.o)
                    lay.gate_up_p = ops.pack_weight((lay.gate_up.float() * lay.post_norm.float()[None, :])
                                                    .to(lay.gate_up.dtype).contiguous())
                    lay.down_p = ops.pack_weight(lay.down)
                    lay.folded = True
                    continue
                lay.qkv_p = ops.pack_weight(lay.qkv)
                lay.o_p = ops.pack_weight(lay.o)
                if lay.moe:
                    lay.gate_up_p = torch.stack([ops.pack_weight(w) for w in lay.gate_up])
                    lay.down_p = torch.stack([ops.pack_weight(w) for w in lay.down])
                    lay.router = lay.router.contiguous()
                else:
                    lay.gate_up_p = ops.pack_weight(lay.gate_up)
                    lay.down_p = ops.pack_weight(lay.down)
        w = self.loop_in
        if w is not None and self.loop_in_p is None and w.dtype == torch.bfloat16 and w.shape[0] % 16 == 0 and \
                w.shape[1] % 128 == 0:
            self.loop_in_p = ops.pack_weight(w)
        if self.lm_head is not None and self.lm_head_p is None and self.cfg.model_type != "gpt2":
            V, H = self.lm_head.shape
            if H % 32 == 0 and self.lm_head.dtype == torch.bfloat16:
                pad = (-V) % 16
                w = self.lm_head if pad == 0 else torch.cat([self.lm_head, self.lm_head.new_zeros(pad, H)])
                # fused-norm decode: the final RMSNorm weight folded in as for qkv / gate_up, so a
                # decode step's lm_head reads the packed residual stream + its row statistics
                # (no final norm launch); other steps normalise with a unit weight first
                fold = fold_norms and self.final_norm is not None
                if fold:
                    w = (w.float() * self.final_norm.float()[None, :]).to(w.dtype)
                self.lm_head_p = ops.pack_weight(w.contiguous())
                self.lm_head_folded = fold

    def quantize_fp8(self, drop_dense: bool = True) -> None:
        """fp8 (OCP e4m3) W8A8 weights for every projection (the 70B fp8 MFMA path).

        ``drop_dense`` frees the bf16 copies (the prefill path then dequantizes one layer at a
        time), halving resident weight bytes: Llama-3-70B fits ONE MI355X (~70 GB) with room
        for a large KV cache.  Embeddings, norms and lm_head stay bf16.
        """
        from .. import ops

        if self.cfg.is_moe:
            raise ValueError("fp8 W8A8 weights are not supported for MoE (Mixtral) models")
        for lay in self.layers:
            if not isinstance(lay, LlamaLayer) or lay.fp8:
                continue
            for name in LlamaLayer.PROJ:
                q, sc = ops.pack_weight_fp8(getattr(lay, name))
                setattr(lay, name + "_q", q)
                setattr(lay, name + "_s", sc)
                if drop_dense:
                    setattr(lay, name, None)
                    setattr(lay, name + "_p", None)

    def prepare_w8a16(self, fold_norms: bool = True) -> None:
        """Convert every fp8 layer to the W8A16 layout (ops.w8_from_fp8) and drop the W8A8
        copies.  ``fold_norms``: qkv / gate_up are dequantized, multiplied by the input /
        post-attention RMSNorm weight along K and re-quantized (W' = W diag(g), per-output-channel
        scales), as the bf16 fused-norm path folds them into its packed weights; ``folded`` is set
        and every path over these weights normalises with a unit RMSNorm weight."""
        from .. import ops

        for lay in self.layers:
            if not isinstance(lay, LlamaLayer) or lay.w8 or lay.qkv_q is None:
                continue
            for name, g in (("qkv", lay.input_norm), ("o", None), ("gate_up", lay.post_norm), ("down", None)):
                q, sc = getattr(lay, name + "_q"), getattr(lay, name + "_s")
                if fold_norms and g is not None:
                    w = ops.unpack_weight_fp8(q, sc, torch.float32) * g.float()[None, :]
                    q, sc = ops.pack_weight_fp8(w)
                    del w
                setattr(lay, name + "_w8", ops.w8_from_fp8(q))
                setattr(lay, name + "_ws", sc)
                setattr(lay, name + "_q", None)
                setattr(lay, name + "_s", None)
            lay.folded = bool(fold_norms)

    @property
    def fp8(self) -> bool:
        return bool(self.layers) and all(isinstance(L, LlamaLayer) and L.fp8 for L in self.layers)

    @property
    def w8(self) -> bool:
        return bool(self.layers) and all(isinstance(L, LlamaLayer) and L.w8 for L in self.layers)

    def tensors(self):
        seen = set()
        for lay in self.layers:
            for f in dataclasses.fields(lay):
                t = getattr(lay, f.name)
                if isinstance(t, torch.Tensor) and id(t) not in seen:
                    seen.add(id(t))
                    yield t
            for t in (t for part in getattr(lay, "parts", ()) for t in part.values()):
                if id(t) not in seen:
                    seen.add(id(t))
                    yield t
        for t in (self.embed, self.pos_embed, self.final_norm, self.final_norm_b, self.lm_head, self.lm_head_p,
                  self.embed_norm, self.loop_in, self.loop_in_p):
            if t is not None and id(t) not in seen:
                seen.add(id(t))
                yield t


def _gen(device, seed: int):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _randn(shape, g, device, dtype, std=INIT_STD):
    t = torch.empty(shape, dtype=torch.float32, device=device)
    t.normal_(0.0, std, generator=g)
    return t.to(dtype)


def _random_llama_layer(cfg: ModelConfig, idx: int, device, dtype, seed: int) -> LlamaLayer:
    g = _gen(device, seed * 100003 + idx + 1)
    H, F = cfg.hidden_size, cfg.intermediate_size
    qkv = _randn((cfg.q_dim + 2 * cfg.kv_dim, H), g, device, dtype)
    o = _randn((H, cfg.q_dim), g, device, dtype)
    ones = torch.ones(H, dtype=dtype, device=device)
    if cfg.is_moe:
        E = cfg.num_local_experts
        router = _randn((E, H), g, device, dtype)
        gu = torch.empty((E, 2 * F, H), dtype=dtype, device=device)
        dn = torch.empty((E, H, F), dtype=dtype, device=device)
        for e in range(E):
            gu[e] = interleave_gate_up(_randn((F, H), g, device, dtype), _randn((F, H), g, device, dtype))
            dn[e] = _randn((H, F), g, device, dtype)
        return LlamaLayer(ones, qkv, o, ones.clone(), gu, dn, router=router)
    gate = _randn((F, H), g, device, dtype)
    up = _randn((F, H), g, device, dtype)
    down = _randn((H, F), g, device, dtype)
    return LlamaLayer(ones, qkv, o, ones.clone(), interleave_gate_up(gate, up), down)


def _random_gpt2_layer(cfg: ModelConfig, idx: int, device, dtype, seed: int) -> GPT2Layer:
    g = _gen(device, seed * 100003 + idx + 1)
    H, F = cfg.hidden_size, cfg.intermediate_size
    z = lambda n: torch.zeros(n, dtype=dtype, device=device)  # noqa: E731
    o = lambda n: torch.ones(n, dtype=dtype, device=device)  # noqa: E731
    return GPT2Layer(o(H), z(H), _randn((3 * H, H), g, device, dtype), z(3 * H), _randn((H, H), g, device, dtype),
                     z(H), o(H), z(H), _randn((F, H), g, device, dtype), z(F), _randn((H, F), g, device, dtype), z(H))


# ------------------------------------------------------------------ hybrid decoders
def _ffn_prefix(spec: LayerSpec) -> str:
    return "mlp.shared." if spec.moe else "mlp."


def _mixer_names(sp: LayerSpec, width: int) -> Dict[str, tuple]:
    """Tensors of a mixer that may be part of a pair (after its own prefix) -> shape."""
    H, G, D, V = sp.heads, sp.kv_heads, sp.dim, sp.vdim
    n: Dict[str, tuple] = {"o": (width, H * V)}
    if sp.mixer == "window_attention":
        n.update({"q": (H * D, width), "k": (G * D, width), "v": (G * V, width),
                  "sink" if sp.weights == "sink" else "pb": (H,)})
    elif sp.mixer == "gated_delta":
        A, R = sp.decay_rank, sp.gate_rank
        n.update({"q": (G * D, width), "k": (G * D, width), "v": (H * V, width), "q.conv": (G * D, sp.conv),
                  "k.conv": (G * D, sp.conv), "v.conv": (H * V, sp.conv), "b": (H, width), "A_log": (H,),
                  "norm": (V,), "a1": (A, width), "a2": (H * D, A), "dt_bias": (H * D,), "g1": (R, width),
                  "g2": (H * V, R)})
    elif sp.mixer == "mamba2":
        C = sp.conv_cols
        n.update({"in": (sp.inner + C + H, width), "conv": (C, sp.conv), "conv.b": (C,), "dt_bias": (H,), "A_log": (H,),
                  "D": (H,), "norm": (sp.inner,)})
    else:
        A = sp.decay_rank
        n.update({"q": (H * D, width), "k": (H * D, width), "v": (H * V, width), "g": (H * V, width), "norm": (V,),
                  "a1": (A, width), "a2": (H * D, A), "a2.b": (H * D,)})
    return n


def _mixer_part(sp: LayerSpec, scale: float, get, dtype) -> Dict[str, torch.Tensor]:
    """What such a mixer's ops read; ``get(name)``: a tensor.  ``scale``: the factor of its output, which goes into the
    gain of its last norm (attention without one takes it as an argument)."""
    f = lambda k: get(k).float().contiguous()  # noqa: E731
    if sp.mixer == "window_attention":
        return {"head": f("sink" if sp.weights == "sink" else "pb")}
    p = {"norm": f("norm") * scale}
    if sp.mixer == "gated_delta":
        p.update(conv=torch.cat([f("q.conv"), f("k.conv"), f("v.conv")]).t().contiguous(), decay=torch.exp(f("A_log")),
                 dt_bias=f("dt_bias"), a2=get("a2").to(dtype).contiguous(), g2=get("g2").to(dtype).contiguous())
    elif sp.mixer == "mamba2":
        p.update(conv=f("conv").t().contiguous(), conv_b=f("conv.b"), decay=torch.exp(f("A_log")), dt_bias=f("dt_bias"),
                 skip=f("D"))
    else:
        p.update(a2=get("a2").to(dtype).contiguous(), a2_b=f("a2.b"))
    for k in [k for k in ("a2", "g2") if k in p]:  # (prompts take the matrix as it is, token by token the packed form)
        from ..ops.gated import pack_low_rank

        p[k + "_p"] = pack_low_rank(p[k], sp.heads)
    return p


def _hybrid_names(spec: LayerSpec, cfg: ModelConfig) -> Dict[str, tuple]:
    """Checkpoint tensors of one layer (after its 'l<i>.' prefix) -> shape."""
    width = cfg.hidden_size
    norm = (width,) if cfg.stream == "pre" else ()
    scaled = cfg.stream == "post"  # post-norm streams have a layer scale per sublayer
    n: Dict[str, tuple] = {"norm1": norm}
    H, D, V = spec.heads, spec.dim, spec.vdim
    if spec.mixer == "pair":
        for p, sp in zip(("left.", "right."), spec.mixers):
            n.update({"mix." + p + k: s for k, s in _mixer_names(sp, width).items()})
    elif spec.mixer in PAIRED:
        n.update({"mix." + k: s for k, s in _mixer_names(spec, width).items()})
    elif spec.mixer == "hgrn2":
        n.update({"mix.q": (H * D, width), "mix.f": (H * D, width), "mix.f.b": (H * D,), "mix.lower": (H * D,),
                  "mix.v": (H * V, width), "mix.norm": (V,), "mix.o": (width, H * V)})
    elif spec.mixer == "latent_attention":
        C, R, Q = spec.kv_rank, spec.rot_dim, spec.q_rank
        n.update({"mix.dq": (Q, width), "mix.dq.norm": (Q,), "mix.uq": (H * (D + R), Q), "mix.dkv": (C + R, width),
                  "mix.dkv.norm": (C,), "mix.uk": (H * D, C), "mix.uv": (H * V, C), "mix.sink": (H,),
                  "mix.o": (width, H * V)})
    elif spec.mixer in ("retention", "mlstm"):
        n.update({"mix.q": (H * D, width), "mix.k": (H * D, width), "mix.v": (H * V, width), "mix.g": (H * V, width),
                  "mix.o": (width, H * V)})
        if spec.mixer == "mlstm":
            n.update({"mix.norm": (H * V,), "mix.i": (H, width), "mix.i.b": (H,), "mix.f": (H, width), "mix.f.b": (H,)})
    elif spec.mixer == "mixed_attention":
        G = spec.kv_heads
        n.update({"mix.q": (H * D, width), "mix.k": (G * D, width), "mix.v": (G * V, width), "mix.q.norm": (D,),
                  "mix.k.norm": (D,), "mix.talk": (H, H), "mix.g": (H, width), "mix.o": (width, H * V)})
    else:
        KD = spec.kv_heads * D
        n.update({"mix.q": (H * D, width), "mix.k": (KD, width), "mix.q.norm": (H * D,), "mix.k.norm": (KD,),
                  "mix.talk": (H, H), "mix.g": (H * D, width), "mix.o": (width, H * D)})
    if spec.ff:
        p = _ffn_prefix(spec)
        n.update({p + "up": (spec.ff, width), p + "down": (width, spec.ff)})
        if spec.glu:
            n[p + "gate"] = (spec.ff, width)
        if spec.moe:
            n[p + "sg"] = (1, width)
    if spec.moe:
        n["mlp.router"] = (spec.moe.experts, width)
        for e in range(spec.moe.experts):
            n.update({f"mlp.e{e}.gate": (spec.moe.ff, width), f"mlp.e{e}.up": (spec.moe.ff, width),
                      f"mlp.e{e}.down": (width, spec.moe.ff)})
    if (spec.ff or spec.moe) and not spec.parallel:
        n["norm2"] = norm
    if spec.shift:
        n["shift"] = (width,)
    if scaled:
        n["ls1"] = (width,)
        if spec.ff:
            n["ls2"] = (width,)
    return n


# a mixer's input projections in the order in which ``w_in`` fuses them
_IN_PARTS = {"hgrn2": ("q", "f", "v"), "attention": ("q", "k", "g"), "latent_attention": ("dq", "dkv"),
             "retention": ("q", "k", "v", "g"), "mlstm": ("q", "k", "v", "g", "i", "f"),
             "mixed_attention": ("q", "k", "v", "g"), "window_attention": ("q", "k", "v"),
             "gated_delta": ("q", "k", "v", "a1", "g1", "b"), "mamba2": ("in",), "gla": ("q", "k", "v", "g", "a1")}


def _stacked_gate_up(gate: torch.Tensor, up: torch.Tensor):
    """Gate and up rows in alternating blocks, and the block: one kernel tile where the width has whole ones."""
    F = gate.shape[0]
    if F % GU_BLOCK == 0:
        return interleave_gate_up(gate, up), GU_BLOCK
    return torch.cat([gate, up], 0), F


def _fill_rows(w: torch.Tensor, rows: int) -> torch.Tensor:
    return w if w.shape[0] == rows else torch.cat([w, w.new_zeros(rows - w.shape[0], w.shape[1])], 0)


def _hybrid_layer(spec: LayerSpec, cfg: ModelConfig, get, device, dtype) -> HybridLayer:
    """``get(name)``: checkpoint tensor of this layer (any device / dtype)."""
    raw = {}
    for name, shape in _hybrid_names(spec, cfg).items():
        t = get(name)
        if shape == () and t.numel() == 1:
            t = t.reshape(())
        if tuple(t.shape) != shape:
            raise ValueError(f"{name}: shape {tuple(t.shape)}, expected {shape}")
        raw[name] = t.to(device)
    f32 = lambda n: raw[n].float().contiguous()  # noqa: E731
    g = lambda n: raw[n].to(dtype).contiguous()  # noqa: E731
    gain = lambda n, ls: f32(n) * f32(ls) if ls in raw else f32(n)  # noqa: E731
    pre = ("mix.left.", "mix.right.") if spec.mixer == "pair" else ("mix.",)
    w_in = torch.cat([_fill_rows(torch.cat([raw[p + k].to(dtype) for k in _IN_PARTS[sp.mixer]], 0), sp.mix_rows)
                      for p, sp in zip(pre, spec.mixers)], 0)
    lay = HybridLayer(spec, w_in.contiguous(), torch.cat([g(p + "o") for p in pre], 1).contiguous(), gain("norm1", "ls1"))
    if spec.mixer == "pair" or spec.mixer in PAIRED:
        scales = (spec.left_scale, spec.right_scale) if spec.mixer == "pair" else (1.0,)
        lay.parts = tuple(_mixer_part(sp, c, lambda k, p=p: raw[p + k], dtype)
                          for p, sp, c in zip(pre, spec.mixers, scales))
    if spec.shift:
        lay.shift = f32("shift")
    if spec.ff:
        p = _ffn_prefix(spec)
        lay.w_up, lay.w_down = g(p + "up"), g(p + "down")
        if spec.glu:
            lay.w_up, lay.ffn_block = _stacked_gate_up(g(p + "gate"), lay.w_up)
        if spec.moe:
            lay.w_up = torch.cat([lay.w_up, g(p + "sg")], 0)
        lay.w_up = _fill_rows(lay.w_up, spec.ff_rows).contiguous()
        if spec.parallel:
            lay.w_in, lay.w_o = torch.cat([lay.w_in, lay.w_up], 0), torch.cat([lay.w_o, lay.w_down], 1).contiguous()
            lay.w_up = lay.w_down = None
    if spec.moe:
        E, F, W = spec.moe.experts, spec.moe.ff, cfg.hidden_size
        lay.w_r = g("mlp.router")
        lay.w_eu = torch.empty(E, 2 * F, W, dtype=dtype, device=device)
        lay.w_ed = torch.empty(E, W, F, dtype=dtype, device=device)
        for e in range(E):
            up, lay.expert_block = _stacked_gate_up(raw[f"mlp.e{e}.gate"], raw[f"mlp.e{e}.up"])
            lay.w_eu[e].copy_(up)
            lay.w_ed[e].copy_(raw[f"mlp.e{e}.down"])
    if "norm2" in raw:
        lay.n2 = gain("norm2", "ls2")
    H, D, V = spec.heads, spec.dim, spec.vdim
    if lay.parts:
        pass
    elif spec.mixer == "hgrn2":
        lay.f_bias, lay.f_lower, lay.o_norm = f32("mix.f.b"), f32("mix.lower"), f32("mix.norm")
    elif spec.mixer == "latent_attention":
        C = spec.kv_rank
        lay.q_norm, lay.c_norm, lay.w_uq, lay.sink = f32("mix.dq.norm"), f32("mix.dkv.norm"), g("mix.uq"), f32("mix.sink")
        uk, uv = g("mix.uk").view(H, D, C), g("mix.uv").view(H, V, C)
        lay.w_uk, lay.w_uv = uk.transpose(1, 2).contiguous(), uv
        lay.w_ukv = torch.cat([uk, uv], 1).reshape(H * (D + V), C).contiguous()
    elif spec.mixer == "retention":
        lay.log_decay = torch.log2(torch.tensor(spec.decay, dtype=torch.float64)).clamp(min=-1e30).float().to(device)
    elif spec.mixer == "mlstm":
        lay.o_norm, lay.gate_bias = f32("mix.norm"), torch.stack([f32("mix.i.b"), f32("mix.f.b")])
    elif spec.mixer == "mixed_attention":
        lay.q_gain, lay.k_gain, lay.talk = f32("mix.q.norm"), f32("mix.k.norm"), f32("mix.talk")
    else:
        kn = f32("mix.k.norm").view(spec.kv_heads, 1, spec.dim)
        kn = kn.expand(spec.kv_heads, spec.heads // spec.kv_heads, spec.dim).reshape(-1)
        lay.w_qk, lay.talk = (f32("mix.q.norm") * kn).contiguous(), f32("mix.talk")
        from ..ops.hybrid import talk_sigma

        lay.sigma = talk_sigma(lay.talk)
    return lay


def random_hybrid_tensors(cfg: ModelConfig, idx: int, device="cpu", dtype=torch.bfloat16,
                          seed: int = 0) -> Dict[str, torch.Tensor]:
    """Synthetic checkpoint tensors of layer ``idx`` (names without the layer prefix)."""
    spec = cfg.layers[idx]
    src = idx if spec.source is None else spec.source
    g = _gen(device, seed * 100003 + src + 1)
    out = {}
    for name, shape in _hybrid_names(spec, cfg).items():
        if name.endswith("norm") or name in ("norm1", "norm2", "ls1", "ls2"):
            t = torch.ones(shape, device=device)
        elif name == "mix.talk":
            t = torch.eye(shape[0], device=device) + _randn(shape, g, device, torch.float32, 0.3 / shape[0] ** 0.5)
        elif name == "mix.f.b":  # forget gates near 1: the state remembers
            t = 2.0 + _randn(shape, g, device, torch.float32, 1.0)
        elif name.endswith((".A_log", ".dt_bias")):  # decays between forgetting at once and hardly at all
            t = _randn(shape, g, device, torch.float32, 1.0) - (2.0 if name.endswith("dt_bias") else 0.0)
        elif name.endswith(".a2.b"):
            t = 2.0 + _randn(shape, g, device, torch.float32, 1.0)
        elif name == "shift":
            t = torch.empty(shape, device=device).uniform_(0.0, 0.5, generator=g)
        elif name in ("mix.i.b", "mix.sink") or name.endswith((".sink", ".pb", ".D", ".conv.b")):
            t = _randn(shape, g, device, torch.float32, 1.0)
        elif name == "mix.lower":
            t = torch.empty(shape, device=device).uniform_(0.0, 0.9, generator=g)
        else:
            t = _randn(shape, g, device, torch.float32, shape[-1] ** -0.5)
        out[name] = t.to(dtype)
    return out


def _hybrid_layers(cfg: ModelConfig, start: int, end: int, make) -> List[HybridLayer]:
    """Layers [start, end): runs of one checkpoint layer share one object, so its weights are held once."""
    made: Dict[int, HybridLayer] = {}
    out = []
    for i in range(start, end):
        src = i if cfg.layers[i].source is None else cfg.layers[i].source
        if src not in made:
            made[src] = make(i, src)
        out.append(made[src])
    return out


def _random_hybrid_layer(cfg: ModelConfig, idx: int, device, dtype, seed: int) -> HybridLayer:
    raw = random_hybrid_tensors(cfg, idx, device, dtype, seed)
    return _hybrid_layer(cfg.layers[idx], cfg, raw.__getitem__, device, dtype)


def _pad_rows(w: torch.Tensor, m: int) -> torch.Tensor:
    """``w`` with zero rows up to a multiple of ``m`` (an lm_head whose logits rows stay 16-B aligned)."""
    pad = (-w.shape[0]) % m
    return w if pad == 0 else torch.cat([w, w.new_zeros(pad, w.shape[1])])


def random_stage_weights(cfg: ModelConfig, start: int, end: int, *, has_embed: bool, has_head: bool, device,
                         dtype=torch.bfloat16, seed: int = 0, fp8: bool = False) -> StageWeights:
    """``fp8``: quantize each block as soon as it is generated (bf16 copies dropped), so a
    70B stage never holds its full bf16 weights."""
    device = torch.device(device)
    mk = _random_gpt2_layer if cfg.model_type == "gpt2" else _random_llama_layer
    layers = _hybrid_layers(cfg, start, end, lambda i, _: _random_hybrid_layer(cfg, i, device, dtype, seed)) \
        if cfg.hybrid else []
    for i in range(start, end) if not cfg.hybrid else ():
        lay = mk(cfg, i, device, dtype, seed)
        if fp8 and isinstance(lay, LlamaLayer):
            one = StageWeights(cfg, i, i + 1, [lay])
            one.quantize_fp8(drop_dense=True)
        layers.append(lay)
    sw = StageWeights(cfg, start, end, layers)
    H, V = cfg.hidden_size, cfg.vocab_size
    if has_embed or (has_head and cfg.tie_word_embeddings):
        g = _gen(device, seed * 100003 + 7919)
        emb = _randn((V, H), g, device, dtype)
        if has_embed:
            sw.embed = emb
            if cfg.embed_norm:
                sw.embed_norm = torch.ones(H, dtype=torch.float32, device=device)
        if cfg.model_type == "gpt2" and has_embed:
            sw.pos_embed = _randn((cfg.max_position_embeddings, H), _gen(device, seed * 100003 + 7927), device,
                                  dtype, std=0.01)
        if has_head and cfg.tie_word_embeddings:
            sw.lm_head = emb
    if any(lay.inject for lay in (cfg.layers or ())[start:end]):
        sw.loop_in = _randn((H, 2 * H), _gen(device, seed * 100003 + 7949), device, dtype, (2 * H) ** -0.5)
    if has_head:
        sw.final_norm = torch.ones(H, dtype=torch.float32 if cfg.hybrid else dtype, device=device)
        if cfg.hybrid:
            sw.final_norm *= cfg.logit_scale
        if cfg.model_type == "gpt2":
            sw.final_norm_b = torch.zeros(H, dtype=dtype, device=device)
        if sw.lm_head is None:
            sw.lm_head = _randn((V, H), _gen(device, seed * 100003 + 7937), device, dtype)
        if cfg.hybrid:
            sw.lm_head = _pad_rows(sw.lm_head, 16)
    return sw


# ------------------------------------------------------------------ checkpoint loading
SAFE_INDEX = "model.safetensors.index.json"
BIN_INDEX = "pytorch_model.bin.index.json"


def checkpoint_files(path: str) -> Optional[str]:
    """Which weight format a local HF directory holds: "safetensors", "bin" or None.

    Same lookup order as upstream Petals ``INDEX_FILES`` / ``_find_index_file``
    (reference petals/server/from_pretrained.py:131-159): sharded safetensors, sharded
    ``.bin``, then single-file variants."""
    if os.path.exists(os.path.join(path, SAFE_INDEX)) or glob.glob(os.path.join(path, "*.safetensors")):
        return "safetensors"
    if os.path.exists(os.path.join(path, BIN_INDEX)) or glob.glob(os.path.join(path, "*.bin")):
        return "bin"
    return None


class _Checkpoint:
    """Key -> shard lookup over a local HF directory (sharded or single-file; safetensors or
    ``pytorch_model*.bin``).

    ``.bin`` shards are read with ``torch.load(weights_only=True, mmap=True)``: the restricted
    unpickler executes nothing from the file, and the memory map means only the tensors a stage
    actually asks for are paged in (upstream ``_load_state_dict_from_local_file``,
    petals/server/from_pretrained.py:216-224, loads whole shards)."""

    def __init__(self, path: str):
        self.path = path
        self._handles: Dict[str, object] = {}
        self.kind = checkpoint_files(path)
        if self.kind is None:
            raise FileNotFoundError(f"no safetensors or pytorch_model*.bin weights under {path}")
        self.key_to_file: Dict[str, str] = {}
        index = os.path.join(path, SAFE_INDEX if self.kind == "safetensors" else BIN_INDEX)
        if os.path.exists(index):
            with open(index) as f:
                wm = json.load(f)["weight_map"]
            self.key_to_file = {k: os.path.join(path, v) for k, v in wm.items()}
        else:
            pattern = "*.safetensors" if self.kind == "safetensors" else "*.bin"
            for fn in sorted(glob.glob(os.path.join(path, pattern))):
                for k in self._open(fn).keys():
                    self.key_to_file[k] = fn

    def _open(self, fn: str):
        h = self._handles.get(fn)
        if h is not None:
            return h
        if self.kind == "safetensors":
            from safetensors import safe_open

            h = safe_open(fn, framework="pt")
        else:
            try:
                h = torch.load(fn, map_location="cpu", weights_only=True, mmap=True)
            except RuntimeError:  # legacy (non-zip) serialization cannot be memory-mapped
                h = torch.load(fn, map_location="cpu", weights_only=True)
            if not isinstance(h, dict):
                raise ValueError(f"{fn}: expected a state dict, got {type(h).__name__}")
        self._handles[fn] = h
        return h

    def has(self, key: str) -> bool:
        return key in self.key_to_file

    def get(self, key: str) -> torch.Tensor:
        h = self._open(self.key_to_file[key])
        return h.get_tensor(key) if self.kind == "safetensors" else h[key]


def checkpoint_shape(path: str, key: str) -> tuple:
    """Shape of a checkpoint tensor (safetensors: from the header alone)."""
    if checkpoint_files(path) is None:
        raise ValueError(f"{path}: the shape of {key} takes the checkpoint")
    ck = _Checkpoint(path)
    if not ck.has(key):
        raise ValueError(f"{path}: no tensor {key}")
    h = ck._open(ck.key_to_file[key])
    return tuple(h.get_slice(key).get_shape() if ck.kind == "safetensors" else h[key].shape)


def load_stage_weights(cfg: ModelConfig, path: str, start: int, end: int, *, has_embed: bool, has_head: bool,
                       device, dtype=torch.bfloat16) -> StageWeights:
    ck = _Checkpoint(path)
    dev = torch.device(device)

    def t(key):
        return ck.get(key).to(device=dev, dtype=dtype)

    layers: List = []
    if cfg.hybrid:
        W = cfg.hidden_size
        layers = _hybrid_layers(cfg, start, end, lambda i, src: _hybrid_layer(
            cfg.layers[i], cfg, lambda n: ck.get(f"l{src}.{n}"), dev, dtype))
        sw = StageWeights(cfg, start, end, layers)
        if has_embed:
            sw.embed = t("embed").contiguous()
            if cfg.embed_norm:
                sw.embed_norm = ck.get("embed.norm").to(dev).float().contiguous()
                if tuple(sw.embed_norm.shape) != (W,):
                    raise ValueError(f"embed.norm: shape {tuple(sw.embed_norm.shape)}, expected {(W,)}")
        if any(sp.inject for sp in cfg.layers[start:end]):
            sw.loop_in = t("loop.in").contiguous()
            if tuple(sw.loop_in.shape) != (W, 2 * W):
                raise ValueError(f"loop.in: shape {tuple(sw.loop_in.shape)}, expected {(W, 2 * W)}")
        if has_head:
            fn = ck.get("final.norm").to(dev).float().reshape(-1)
            sw.final_norm = (fn * cfg.logit_scale).expand(W).contiguous()  # (one gain for all, or one each)
            sw.lm_head = _pad_rows(t("head"), 16).contiguous()
        return sw
    if cfg.model_type == "gpt2":
        pre = "transformer." if ck.has("transformer.wte.weight") else ""
        for i in range(start, end):
            p = f"{pre}h.{i}."
            layers.append(GPT2Layer(t(p + "ln_1.weight"), t(p + "ln_1.bias"), t(p + "attn.c_attn.weight").t().contiguous(),
                                    t(p + "attn.c_attn.bias"), t(p + "attn.c_proj.weight").t().contiguous(),
                                    t(p + "attn.c_proj.bias"), t(p + "ln_2.weight"), t(p + "ln_2.bias"),
                                    t(p + "mlp.c_fc.weight").t().contiguous(), t(p + "mlp.c_fc.bias"),
                                    t(p + "mlp.c_proj.weight").t().contiguous(), t(p + "mlp.c_proj.bias")))
        sw = StageWeights(cfg, start, end, layers)
        if has_embed:
            sw.embed = t(pre + "wte.weight")
            sw.pos_embed = t(pre + "wpe.weight")
        if has_head:
            sw.final_norm, sw.final_norm_b = t(pre + "ln_f.weight"), t(pre + "ln_f.bias")
            sw.lm_head = sw.embed if sw.embed is not None else t(pre + "wte.weight")
        return sw
    for i in range(start, end):
        p = f"model.layers.{i}."
        qkv = torch.cat([t(p + "self_attn.q_proj.weight"), t(p + "self_attn.k_proj.weight"),
                         t(p + "self_attn.v_proj.weight")], 0).contiguous()
        if cfg.is_moe:  # HF MixtralSparseMoeBlock: gate = router, experts.j.{w1 gate, w3 up, w2 down}
            m = p + "block_sparse_moe."
            E = cfg.num_local_experts
            gu = torch.stack([interleave_gate_up(t(f"{m}experts.{j}.w1.weight"), t(f"{m}experts.{j}.w3.weight"))
                              for j in range(E)])
            dn = torch.stack([t(f"{m}experts.{j}.w2.weight") for j in range(E)])
            layers.append(LlamaLayer(t(p + "input_layernorm.weight"), qkv, t(p + "self_attn.o_proj.weight"),
                                     t(p + "post_attention_layernorm.weight"), gu, dn, router=t(m + "gate.weight")))
            continue
        gu = interleave_gate_up(t(p + "mlp.gate_proj.weight"), t(p + "mlp.up_proj.weight")).contiguous()
        layers.append(LlamaLayer(t(p + "input_layernorm.weight"), qkv, t(p + "self_attn.o_proj.weight"),
                                 t(p + "post_attention_layernorm.weight"), gu, t(p + "mlp.down_proj.weight")))
    sw = StageWeights(cfg, start, end, layers)
    if has_embed:
        sw.embed = t("model.embed_tokens.weight")
    if has_head:
        sw.final_norm = t("model.norm.weight")
        if ck.has("lm_head.weight"):
            sw.lm_head = t("lm_head.weight")
        else:  # tied embeddings
            sw.lm_head = sw.embed if sw.embed is not None else t("model.embed_tokens.weight")
    return sw


def build_stage_weights(cfg: ModelConfig, model: str, start: int, end: int, *, has_embed: bool, has_head: bool,
                        device, dtype=torch.bfloat16, seed: int = 0) -> StageWeights:
    """Checkpoint weights when ``model`` is a local HF directory, synthetic weights for presets.

    A directory without loadable weights is an error: silently serving a real config with
    random weights would produce garbage that looks like a working server."""
    if os.path.isdir(model):
        if checkpoint_files(model) is None:
            raise FileNotFoundError(f"--model {model!r} is a directory without *.safetensors or pytorch_model*.bin "
                                    f"weights (pass a preset name such as llama2-7b for synthetic weights)")
        return load_stage_weights(cfg, model, start, end, has_embed=has_embed, has_head=has_head, device=device,
                                  dtype=dtype)
    return random_stage_weights(cfg, start, end, has_embed=has_embed, has_head=has_head, device=device, dtype=dtype,
                                seed=seed)
