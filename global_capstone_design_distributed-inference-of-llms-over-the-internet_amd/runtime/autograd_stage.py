"""Stateless, differentiable stage forward/backward: the fine-tuning half of the Petals server.

Reference (vendored upstream server):
* ``run_rpc_forward`` (petals/server/block_functions.py:32-81) runs the span's blocks on a
  ``[B, T, H]`` hidden state with optional *deep prompts* ``[n_blocks, B, P, H]``. Before block i,
  ``hidden[:, :P] += prompts[i]``. No KV cache is involved.
* ``run_rpc_backward`` (:84-141) recomputes that forward with autograd and returns the gradient
  w.r.t. the input hidden state and w.r.t. the prompts. For block i, the prompt gradient is
  the gradient flowing into ``hidden[:, :P]`` at its input.
* handler endpoints ``rpc_forward(_stream)`` / ``rpc_backward(_stream)``
  (petals/server/handler.py:352-488). Server weights are frozen. Clients train prompts or
  adapters on their side.

The inference hot path (paged KV, HIP kernels, hipGraphs) is not differentiable and does not
need to be. This module is the training-time path on the stage's resident weights (the same
tensors the executor uses; no copies), in two forms:
* kernels (``ops/train.py``): bf16 LLaMA / Mistral blocks on the GPU. The weights are frozen, so a
  block's backward is written out: the forward of the span is made again, keeping per block its
  input, q / k / v, the attention's output and gate / up rows, then the blocks are run backwards.
  Attention never holds a [heads, T, T] tensor.
* plain PyTorch ops and library GEMMs for everything else (CPU, fp32, experts, GPT-2, callers that differentiate
  ``forward`` themselves): attention is an explicit causal softmax in fp32, backward = recompute
  forward + ``torch.autograd.grad``, as upstream.
Either way no activations are held between the two RPCs.
"""
from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
import torch.nn.functional as F

from .. import ops
from ..models.weights import split_gate_up
from ..ops import prompt, train
from ..ops.moe import moe_mlp_torch
from ..ops.reference import rope_cos_sin, rope_inv


def _rms(x, w, eps):
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype) * w


def _plain(*tensors) -> bool:
    """Are these ordinary tensors in an ordinary call: no subclass, no transform (vmap, grad, forward mode), no tracing and
    no dispatch mode that has to see every operation?"""
    return (all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors) and
            not torch.compiler.is_compiling() and not torch.jit.is_tracing() and
            torch._C._functorch.peek_interpreter_stack() is None and
            torch.autograd.forward_ad._current_level < 0 and
            torch._C._len_torch_dispatch_stack() == 0 and
            torch.overrides._get_current_function_mode() is None)


def _rows(t: torch.Tensor) -> torch.Tensor:
    """[B, T, H] as rows that the kernels read: contiguous and 16-byte aligned."""
    t = t.reshape(-1, t.shape[-1]).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class AutogradStage:
    """Differentiable view of a stage's blocks (LLaMA-family and GPT-2)."""

    def __init__(self, cfg, weights, device, dtype=None):
        if cfg.hybrid:
            raise ValueError("training RPCs cover the uniform decoder families, not hybrid decoders")
        self.cfg = cfg
        self.w = weights
        self.device = torch.device(device)
        self.dtype = dtype or (weights.layers[0].input_norm.dtype if cfg.model_type != "gpt2"
                               else weights.layers[0].ln1_w.dtype)
        self._cache = {}  # per-layer (gate, up) views, made once
        self._inv = None  # the kernel form's rotary angles of one position, on the device (made once)

    @property
    def n_blocks(self) -> int:
        return len(self.w.layers)

    # ------------------------------------------------------------------ blocks
    def _attn(self, q, k, v):
        """q [B,T,nh,D], k/v [B,T,nkv,D] -> [B,T,nh*D], causal, fp32 softmax."""
        B, T, nh, D = q.shape
        rep = nh // k.shape[2]
        k = k.repeat_interleave(rep, 2) if rep > 1 else k
        v = v.repeat_interleave(rep, 2) if rep > 1 else v
        s = torch.einsum("bqhd,bkhd->bhqk", q.float(), k.float()) / math.sqrt(D)
        mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
        p = torch.softmax(s.masked_fill(mask, float("-inf")), -1)
        return torch.einsum("bhqk,bkhd->bqhd", p, v.float()).to(q.dtype).reshape(B, T, nh * D)

    def _llama_block(self, i, x, cos, sin):
        cfg, lay = self.cfg, self.w.layers[i]
        nh, nkv, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
        B, T, _ = x.shape
        h = _rms(x, lay.input_norm, cfg.rms_norm_eps)
        qkv = h @ lay.qkv.t()
        q = qkv[..., : nh * D].view(B, T, nh, D)
        k = qkv[..., nh * D: (nh + nkv) * D].view(B, T, nkv, D)
        v = qkv[..., (nh + nkv) * D:].view(B, T, nkv, D)
        c, s = cos[:T].view(1, T, 1, D // 2).to(x.dtype), sin[:T].view(1, T, 1, D // 2).to(x.dtype)

        def rot(t):
            t1, t2 = t[..., : D // 2], t[..., D // 2:]
            return torch.cat([t1 * c - t2 * s, t2 * c + t1 * s], -1)

        x = x + self._attn(rot(q), rot(k), v) @ lay.o.t()
        h = _rms(x, lay.post_norm, cfg.rms_norm_eps)
        if lay.router is not None:
            return x + moe_mlp_torch(h, lay.router, lay.gate_up, lay.down, cfg.num_experts_per_tok)
        if i not in self._cache:
            self._cache[i] = split_gate_up(lay.gate_up)
        g, u = self._cache[i]
        return x + (F.silu(h @ g.t()) * (h @ u.t())) @ lay.down.t()

    def _gpt2_block(self, i, x):
        cfg, lay = self.cfg, self.w.layers[i]
        H, nh, D = cfg.hidden_size, cfg.num_attention_heads, cfg.head_dim
        B, T, _ = x.shape
        a = F.layer_norm(x, (H,), lay.ln1_w, lay.ln1_b, cfg.layer_norm_eps)
        q, k, v = [t.reshape(B, T, nh, D) for t in (a @ lay.attn_w.t() + lay.attn_b).split(H, -1)]
        x = x + self._attn(q, k, v) @ lay.proj_w.t() + lay.proj_b
        m = F.layer_norm(x, (H,), lay.ln2_w, lay.ln2_b, cfg.layer_norm_eps)
        m = F.gelu(m @ lay.fc_w.t() + lay.fc_b, approximate="tanh")
        return x + m @ lay.fc2_w.t() + lay.fc2_b

    # ------------------------------------------------------------------ blocks on kernels
    def _kernels(self, hidden, prompts, *more) -> bool:
        """Does the kernel form cover this call?  bf16 blocks it knows the shape of, whole weights on one GPU, at least one
        token; a caller that differentiates the call itself (``backward`` does it without autograd) takes the other."""
        given = [t for t in (hidden, prompts) + more if t is not None]
        if self.device.type != "cuda" or self.dtype != torch.bfloat16 or not train.shape_ok(self.cfg) or not self.w.layers:
            return False
        if not _plain(*given) or hidden.dim() != 3 or not train.rows_ok(*hidden.shape[:2]) or \
                hidden.shape[2] != self.cfg.hidden_size:
            return False
        for lay in self.w.layers:
            mats = [getattr(lay, n, None) for n in ("input_norm", "qkv", "o", "post_norm", "gate_up", "down")]
            if any(m is None or m.dtype != torch.bfloat16 or not m.is_contiguous() or m.data_ptr() % 16 or m.requires_grad or
                   m.device.type != "cuda" or m.device != mats[0].device for m in mats):
                return False
        ops.require_native()
        return True

    def _kernel_blocks(self, x, prompts, B, T, table, keep: bool):
        """The span's blocks over the rows ``x`` [B T, H]: (rows out, what ``_kernel_grads`` reads of every block).  With
        ``keep`` the last block ends at its gate / up rows: nothing of a gradient depends on what follows."""
        cfg = self.cfg
        nh, nkv, D, eps = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.rms_norm_eps
        kept, y = [], None
        for i, lay in enumerate(self.w.layers):
            deep = None
            if prompts is not None and prompts.shape[2]:
                deep = prompts[i]
                if deep.shape[0] not in (1, B) or deep.shape[2] != cfg.hidden_size:  # (what broadcasts, or raises)
                    deep = deep.expand(B, deep.shape[1], cfg.hidden_size)
                deep = _rows(deep).view(deep.shape)
            x, h = train.norm(x, lay.input_norm, eps, y, deep, T)
            qkv = train.rope_(ops.linear(h, lay.qkv, tiles=True), table, nh + nkv, D)
            a, a32, lse = train.attention(qkv, B, nh, nkv, D, keep)
            x2, h = train.norm(x, lay.post_norm, eps, ops.linear(a, lay.o, tiles=True))
            if keep:
                gu = ops.linear(h, lay.gate_up, tiles=True)
                kept.append((x, qkv, a32, lse, x2, gu))
                if i == len(self.w.layers) - 1:
                    return None, kept
                act = ops.swiglu(gu)
            else:
                act = ops.linear(h, lay.gate_up, epilogue=1, tiles=True)
            x, y = x2, ops.linear(act, lay.down, tiles=True)
        return x + y, kept

    def _kernel_grads(self, g, kept, prompts, B, T, table):
        """Gradients of the blocks' input and of the prompts from the gradient ``g`` [B T, H] of their output."""
        cfg = self.cfg
        nh, nkv, D, eps = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.rms_norm_eps
        gp = None if prompts is None else torch.empty_like(prompts)
        for i in reversed(range(len(kept))):
            lay, (x, qkv, a32, lse, x2, gu) = self.w.layers[i], kept.pop()
            dgu = train.glu_grad_(gu, prompt.gemm_columns(g, lay.down))
            g = train.norm_grad(x2, prompt.gemm_columns(dgu, lay.gate_up), lay.post_norm, eps, g)
            dqkv = train.attention_grad(qkv, B, nh, nkv, D, a32, lse, prompt.gemm_columns(g, lay.o), table)
            g = train.norm_grad(x, prompt.gemm_columns(dqkv, lay.qkv), lay.input_norm, eps, g)
            if gp is not None:
                d = g.view(B, T, -1)[:, :gp.shape[2]]
                gp[i] = d.sum(0, keepdim=True) if gp.shape[1] == 1 else d
        return g, gp

    def _angles(self, T: int):
        if self._inv is None:
            self._inv = rope_inv(self.cfg.head_dim, self.cfg.rope_theta, self.cfg.rope_scaling).to(self.device)
        return train.angles(self._inv, T)

    # ------------------------------------------------------------------ public API
    def forward(self, hidden: torch.Tensor, prompts: Optional[torch.Tensor] = None) -> torch.Tensor:
        """hidden [B, T, H]; prompts None or [n_blocks, B|1, P, H] (P <= T). Returns [B, T, H]."""
        x = hidden.to(self.device, self.dtype)
        if prompts is not None:
            prompts = prompts.to(self.device, self.dtype)
            if prompts.dim() != 4 or prompts.shape[0] != self.n_blocks or prompts.shape[2] > x.shape[1]:
                raise ValueError(f"prompts must be [{self.n_blocks}, B, P<=T, H], got {tuple(prompts.shape)}")
        T = x.shape[1]
        if self._kernels(x, prompts) and not (torch.is_grad_enabled() and (
                x.requires_grad or (prompts is not None and prompts.requires_grad))):
            B = x.shape[0]
            y, _ = self._kernel_blocks(_rows(x), prompts, B, T, self._angles(T), False)
            return y.view(B, T, -1)
        cos = sin = None
        if self.cfg.model_type != "gpt2":
            cos, sin = rope_cos_sin(self.cfg.head_dim, T, self.cfg.rope_theta, self.device, self.cfg.rope_scaling)
        for i in range(self.n_blocks):
            if prompts is not None:
                P = prompts.shape[2]
                x = torch.cat([x[:, :P] + prompts[i], x[:, P:]], 1)
            x = self._gpt2_block(i, x) if self.cfg.model_type == "gpt2" else self._llama_block(i, x, cos, sin)
        return x

    def backward(self, hidden: torch.Tensor, grad_output: torch.Tensor,
                 prompts: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
        """Recompute the forward and return (grad_hidden, grad_prompts)."""
        got = self._backward_kernels(hidden, grad_output, prompts)
        if got is not None:
            return got
        with torch.enable_grad():
            x = hidden.detach().to(self.device, self.dtype).requires_grad_(True)
            p = None
            if prompts is not None:
                p = prompts.detach().to(self.device, self.dtype).requires_grad_(True)
            out = self.forward(x, p)
            inputs = [x] if p is None else [x, p]
            grads = torch.autograd.grad(out, inputs, grad_output.to(self.device, out.dtype), allow_unused=True)
        gp = None
        if p is not None:
            gp = grads[1] if grads[1] is not None else torch.zeros_like(p)
        return grads[0], gp

    def _backward_kernels(self, hidden, grad_output, prompts):
        """``backward`` on the kernels, or None where they do not cover the call (the other form then raises what is to be
        raised)."""
        if not self._kernels(hidden, prompts, grad_output) or grad_output.shape != hidden.shape:
            return None
        B, T, H = hidden.shape
        if prompts is not None and (prompts.dim() != 4 or prompts.shape[0] != self.n_blocks or prompts.shape[2] > T or
                                    prompts.shape[1] not in (1, B) or prompts.shape[3] != H):
            return None
        with torch.no_grad():
            x = _rows(hidden.to(self.device, self.dtype))
            g = _rows(grad_output.to(self.device, self.dtype))
            p = prompts.to(self.device, self.dtype) if prompts is not None else None
            table = self._angles(T)
            _, kept = self._kernel_blocks(x, p, B, T, table, True)
            gx, gp = self._kernel_grads(g, kept, p, B, T, table)
            return gx.view(B, T, H), gp
