"""The calls whose speed this framework is judged by: decode steps, prompts, short generations and fine-tuning requests of
the model families it serves, through ``StageExecutor``, ``BatchSampler`` and ``AutogradStage``.

A case names a preset of ``src.models.config``, the blocks of it that the stage holds, and what the stage is asked for:

* ``step``      one decode step of sessions that already hold a context (the ordinary call of a serving loop);
* ``prompt``    the prompts of new sessions in one ragged step (time to first token);
* ``generate``  prompts of new sessions and some decode steps after them, next tokens given.  Sessions with recurrent state
                cannot go back, so this is the pass of theirs that can be repeated;
* ``tune``      a fine-tuning client's forward and backward request with deep prompts.

``role`` is the stage's place: ``full`` (token ids to logits), ``segment`` (hidden rows to hidden rows) or ``last`` (hidden
rows to logits).  ``shortest`` and ``longest`` bound the sessions' lengths, which spread over that range.
"""
import dataclasses
import math

import torch
import torch.nn.functional as F

from src.models.config import resolve_model
from src.models.weights import random_hybrid_tensors, random_stage_weights
from src.runtime.autograd_stage import AutogradStage
from src.runtime.executor import StageExecutor
from src.runtime.sampler import BatchSampler, SamplingParams

MOE_FAMILIES = ("mixtral-8x7b", "nuvorax-7b")  # (a decode batch reads most experts: fewer steps keep the cost of a pass alike)


def _case(kind, model, first, last, role, sessions, shortest, longest, steps=0, weights="bf16", sample=False, prefix=0):
    return {"kind": kind, "model": model, "first": first, "last": last, "role": role, "sessions": sessions,
            "shortest": shortest, "longest": longest, "steps": steps, "weights": weights, "sample": sample, "prefix": prefix}


def listed():
    named = {
        # a small model answering one user: launches and latency, hardly any bytes
        "step-small": _case("step", "small-llama", 0, 8, "full", 1, 100, 100),
        # the interactive case: one session of an 8B model, weights streamed for a single token
        "step-one": _case("step", "llama3-8b", 0, 4, "full", 1, 900, 900),
        # the serving benchmark's shape: 64 chats of a 7B model in the last stage, tokens sampled there
        "step-batch": _case("step", "llama2-7b", 28, 32, "last", 64, 64, 256, sample=True),
        # long documents in a middle stage with fp8 weights: the cache is most of the traffic
        "step-long": _case("step", "llama3-8b", 8, 12, "segment", 12, 1500, 6000, weights="fp8"),
        # a wave of new chats of all lengths arriving at a middle stage
        "prompt-ragged": _case("prompt", "llama2-7b", 8, 10, "segment", 20, 7, 601),
        # one long document, the longest prompt that fits a step
        "prompt-long": _case("prompt", "llama3-8b", 0, 2, "full", 1, 7995, 7995),
        # routed experts over a few prompts, then a small decode batch
        "generate-mixtral": _case("generate", "mixtral-8x7b", 4, 6, "segment", 6, 40, 700, 6),
        # a client tuning soft prompts through a span of blocks
        "tune": _case("tune", "mistral-7b", 4, 6, "segment", 2, 777, 777, prefix=16),
        # the hybrid decoders: recurrent and attention layers side by side
        "generate-kafunex": _case("generate", "kafunex-7b", 2, 4, "full", 4, 100, 1801, 8),
        "generate-fubapel": _case("generate", "fubapel-7b", 0, 3, "full", 4, 100, 1801, 8),
        "generate-nuvorax": _case("generate", "nuvorax-7b", 0, 3, "full", 4, 100, 1801, 8),
        "generate-debuzen": _case("generate", "debuzen-7b", 4, 7, "full", 4, 100, 1801, 8),
    }
    return [{"name": n, **c} for n, c in named.items()]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of lo .. hi."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(("step", "step", "prompt", "prompt", "generate", "generate", "generate", "tune"))
    if kind == "step":
        model, fp8 = rng.choice((("small-llama", False), ("llama2-7b", False), ("llama3-8b", False), ("llama3-8b", True)))
        role, n = rng.choice(("full", "segment", "last")), _log(rng, 1, 64)
        longest = _log(rng, 20, min(2000 if model == "small-llama" else 4000 if model == "llama2-7b" else 7000, 72000 // n))
        return _case("step", model, 0, rng.randint(2, 4), role, n, max(1, longest // 3), longest,
                     weights="fp8" if fp8 else "bf16", sample=role != "segment" and n >= 16 and rng.random() < 0.5)
    if kind == "prompt":
        model, n = rng.choice(("small-llama", "llama2-7b", "llama3-8b")), _log(rng, 1, 40)
        longest = _log(rng, 4, min(1900 if model == "small-llama" else 4000 if model == "llama2-7b" else 7900, 7900 // n))
        return _case("prompt", model, 0, 2, rng.choice(("full", "segment", "last")), n, max(1, longest // 20), longest)
    if kind == "tune":
        longest = _log(rng, 16, 700)
        return _case("tune", rng.choice(("small-llama", "mistral-7b")), 4, 6, "segment", rng.randint(1, 2), longest, longest,
                     prefix=rng.choice((0, 1, 8, 16)))
    model, first, last = rng.choice((("mixtral-8x7b", 4, 6), ("kafunex-7b", 2, 4), ("fubapel-7b", 0, 3), ("nuvorax-7b", 0, 3),
                                     ("debuzen-7b", 4, 7)))
    n = _log(rng, 1, 16)
    longest = _log(rng, 8, min(1800, 4000 // n))
    role = "segment" if model == "mixtral-8x7b" else "full"
    return _case("generate", model, first, last, role, n, max(1, longest // 10), longest,
                 rng.randint(1, 5 if model in MOE_FAMILIES else 8))


# ------------------------------------------------------------------ what a pass works on
def _lengths(case):
    n, a, b = case["sessions"], case["shortest"], case["longest"]
    return [b - round((b - a) * ((i * 0.6180339887) % 1.0)) for i in range(n)]


def _config(case):
    """The preset; a hybrid decoder's blocks as a model of their own (layers of one model differ, a short one stands for a
    stack of them)."""
    cfg = resolve_model(case["model"])
    if not cfg.hybrid:
        return cfg
    layers = tuple(cfg.layers[case["first"]:case["last"]])
    return dataclasses.replace(cfg, layers=layers, num_hidden_layers=len(layers))


def _weights(case, seed, cfg):
    first, last = (0, cfg.num_hidden_layers) if cfg.hybrid else (case["first"], case["last"])
    w = random_stage_weights(cfg, first, last, has_embed=case["role"] == "full", has_head=case["role"] != "segment",
                             device="cuda:0", seed=seed % 10007, fp8=case["weights"] == "fp8")
    if case["sample"]:  # a trained head is decided: few tokens share most of the probability
        w.lm_head = w.lm_head * 4
    if cfg.hybrid:
        _decide(w, cfg, torch.Generator().manual_seed(seed))
    return w


def _decide(w, cfg, gen):
    """Tokens lean towards some experts of every block, of as many groups as are kept: a trained router is decided, and its
    choices do not turn on the last bit of a sum."""
    lean = torch.zeros_like(w.embed, dtype=torch.float32)
    for sp, lay in zip(cfg.layers, w.layers):
        if sp.moe is None:
            continue
        m, size = sp.moe, sp.moe.experts // sp.moe.groups
        score = torch.rand(cfg.vocab_size, m.groups, size, generator=gen)
        drop = torch.topk(torch.rand(cfg.vocab_size, m.groups, generator=gen), m.groups - m.keep).indices
        wish = torch.topk(score.scatter_(1, drop[:, :, None].expand(-1, -1, size), -1.0).flatten(1), m.top).indices.cuda()
        for k in range(m.top):
            lean += (16.0 / cfg.embed_scale) * lay.w_r.float()[wish[:, k]]
    w.embed = (w.embed.float() + lean).to(w.embed.dtype)


def _rows(n, case, cfg, gen):
    """Token ids, or rows of a residual stream: unit size with a few large channels."""
    if case["role"] == "full":
        return torch.randint(0, cfg.vocab_size, (n,), generator=gen)
    x = torch.randn(n, cfg.hidden_size, generator=gen)
    x[:, torch.randperm(cfg.hidden_size, generator=gen)[: cfg.hidden_size // 128]] *= 8.0
    return x.to(torch.bfloat16)


def _decided(x, w, gen):
    """Rows that lean towards some experts of every block, popular ones more often (see ``_decide``)."""
    for lay in w.layers if w.cfg.is_moe else ():
        r = lay.router.float()
        wish = torch.multinomial(torch.linspace(1.0, 0.3, r.shape[0]).expand(x.shape[0], -1), w.cfg.num_experts_per_tok,
                                 generator=gen).cuda()
        for k, much in zip(range(wish.shape[1]), (12.0, 9.0)):
            x = (x.float() + much * r[wish[:, k]]).to(x.dtype)
    return x


def _inputs(case, seed, cfg, w):
    """Per session the rows it holds or brings, and the rows of each later step."""
    gen = torch.Generator().manual_seed(seed)
    steps = 1 if case["kind"] == "step" else case["steps"]
    first = [_decided(_rows(n, case, cfg, gen).cuda(), w, gen) for n in _lengths(case)]
    return first, [_decided(_rows(case["sessions"], case, cfg, gen).cuda(), w, gen) for _ in range(steps)], gen


def _tune_inputs(case, seed, cfg):
    gen = torch.Generator().manual_seed(seed)
    B, T, P, H = case["sessions"], case["longest"], case["prefix"], cfg.hidden_size
    hidden = _rows(B * T, case, cfg, gen).view(B, T, H).cuda()
    grad = (torch.randn(B, T, H, generator=gen) / T).to(torch.bfloat16).cuda()
    prompts = (0.5 * torch.randn(case["last"] - case["first"], B, P, H, generator=gen)).to(torch.bfloat16).cuda()
    return hidden, grad, prompts if P else None


@torch.no_grad()
def prepare(case, seed):
    cfg = _config(case)
    w = _weights(case, seed, cfg)
    if case["kind"] == "tune":
        hidden, grad, prompts = _tune_inputs(case, seed, cfg)
        return {"case": case, "stage": AutogradStage(cfg, w, "cuda:0"), "hidden": hidden, "grad": grad, "prompts": prompts}
    n, lens = case["sessions"], _lengths(case)
    ex = StageExecutor(cfg, w, "cuda:0", max_sessions=max(n, 4), max_seq_len=min(cfg.max_position_embeddings,
                                                                                 max(lens) + case["steps"] + 1),
                       kv_cache_bytes=6 << 30, max_tokens_per_step=8192, warmup=False)
    first, later, gen = _inputs(case, seed, cfg, w)
    sids = [f"chat-{i}" for i in range(n)]
    state = {"case": case, "ex": ex, "sids": sids, "lens": lens, "first": torch.cat(first), "later": later}
    if case["kind"] == "step":
        ex.forward(list(zip(sids, lens)), state["first"], reset=[True] * n)
    if case["sample"]:
        state["sampler"] = BatchSampler("cuda:0", max_rows=n)
        state["params"] = [SamplingParams(1.0, 0.92, 50, 1.5)] * n
        state["histories"] = torch.randint(0, cfg.vocab_size, (n, 50), generator=gen).tolist()
        state["seeds"] = torch.randint(0, 1 << 60, (n,), generator=gen).tolist()
    return state


@torch.no_grad()
def run(state):
    case = state["case"]
    if case["kind"] == "tune":
        out = state["stage"].forward(state["hidden"], state["prompts"])
        grads = state["stage"].backward(state["hidden"], state["grad"], state["prompts"])
        return [out] + [g for g in grads if g is not None]
    ex, sids, lens = state["ex"], state["sids"], state["lens"]
    if case["kind"] == "step":
        out = ex.forward([(s, 1) for s in sids], state["later"][0], starts=lens)
        if not case["sample"]:
            return out
        return [out, state["sampler"](out, state["params"], state["histories"], state["seeds"])]
    out = ex.forward(list(zip(sids, lens)), state["first"], reset=[True] * len(sids))
    if case["kind"] == "prompt":
        return out
    outs = [out]
    for rows in state["later"]:  # (a step's logits are a buffer that the next step writes again)
        outs.append(ex.forward([(s, 1) for s in sids], rows).clone())
    return outs


# ------------------------------------------------------------------ what a pass cannot do without
def _used_params(case, cfg, rows):
    """(bytes of weights that ``rows`` tokens read, multiply-adds of one token) over the stage's blocks."""
    H, size = cfg.hidden_size, 1 if case["weights"] == "fp8" else 2
    read = macs = 0
    for i in range(case["first"], case["last"]):
        if cfg.hybrid:
            sp = cfg.layers[i - case["first"]]
            n, moe = sp.param_count(H), (sp.moe.experts, sp.moe.top, 3 * sp.moe.ff * H) if sp.moe else None
        else:
            moe = (cfg.num_local_experts, cfg.num_experts_per_tok, 3 * H * cfg.intermediate_size) if cfg.is_moe else None
            n = cfg.layer_param_bytes(1)
        macs += n - (moe[0] - moe[1]) * moe[2] if moe else n
        read += n - round(moe[0] * (1 - moe[1] / moe[0]) ** rows) * moe[2] if moe else n
    return read * size, macs


def _pairs(n, start=0):
    """Query-key pairs of tokens start .. start + n - 1 of a causal sequence."""
    return n * start + n * (n + 1) // 2


def work(case):
    cfg = _config(case)
    H, lens, n = cfg.hidden_size, _lengths(case), case["sessions"]
    if case["kind"] == "tune":
        T, rows, layers = case["longest"], case["longest"] * n, case["last"] - case["first"]
        read, macs = _used_params(case, cfg, rows)
        attn = 2 * cfg.q_dim * _pairs(T) * n * layers  # scores and values; backward recomputes them and has four products
        return {"bytes": 2 * read + rows * H * 2 * 5 + 2 * layers * n * case["prefix"] * H * 2 * 2,
                "flops": 2 * (3 * rows * macs + 4 * attn)}
    prompt = case["kind"] != "step"
    calls = ([(lens, [0] * n)] if prompt else []) + \
        [([1] * n, [x + k for x in lens]) for k in range(1 if not prompt else case["steps"])]
    total = {"bytes": 0, "flops": 0}
    for ntoks, starts in calls:
        rows = sum(ntoks)
        read, macs = _used_params(case, cfg, rows)
        width = cfg.hidden_width * (4 if cfg.hybrid else 2)
        b = read + rows * (8 if case["role"] == "full" else width)
        f = 2 * rows * macs
        if case["role"] == "full":
            b += rows * H * 2
        if case["role"] != "segment":
            b += cfg.vocab_size * H * 2 + n * cfg.vocab_size * 2
            f += 2 * n * cfg.vocab_size * H
        else:
            b += rows * width
        for i in range(case["first"], case["last"]):
            for sp in cfg.layers[i - case["first"]].mixers if cfg.hybrid else (None,):
                if sp is not None and sp.recurrent:
                    b += sp.state_elems * 4 * n * (1 if starts[0] == 0 else 2)
                    f += 4 * rows * sp.heads * sp.dim * sp.vdim
                    continue
                heads, dims = (sp.heads, sp.dim + sp.vdim) if sp is not None else (cfg.num_attention_heads, 2 * cfg.head_dim)
                reach = sp.reach if sp is not None else 1 << 30
                row = sp.cache_bytes(2) if sp is not None else cfg.kv_bytes_per_token_per_layer(2)
                b += row * (rows + sum(min(s, reach) for s in starts))
                f += 2 * heads * dims * sum(_pairs(t, s) if t + s <= reach else t * min(reach, s + t)
                                            for t, s in zip(ntoks, starts))
        total["bytes"] += b
        total["flops"] += f
    return total


def tolerance(case):
    """bf16 activations between 32-bit sums.  Against ``exact`` the uniform families are 0.003 to 0.02 off (a bf16 stream), the
    hybrid decoders 0.0035 to 0.011 (a 32-bit one); a token sampled from such logits may be another one."""
    out = {"rel": 0.06 if not _config(case).hybrid else 0.04}
    return {**out, "differ": 0.6} if case["sample"] else out


# ------------------------------------------------------------------ the same in 64 bits, plain torch
def _d(t):
    return t.double()


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, eps):
    return _rms(x - x.mean(-1, keepdim=True), eps)


def _group_norm(x, eps, groups):
    return _rms(x.view(*x.shape[:-1], groups, -1), eps).reshape(x.shape)


def _turns(L, dims, base, scaling=None):
    """cos and sin [L, 1, dims / 2] of every position's angles."""
    f = float(base) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device="cuda") / dims)
    if scaling is not None:
        factor, low, high, original = scaling
        wave = 2 * math.pi / f
        s = ((original / wave - low) / (high - low)).clamp(0, 1)
        f = (1 - s) * f / factor + s * f
    a = torch.arange(L, dtype=torch.float64, device="cuda")[:, None] * f
    return torch.cos(a)[:, None], torch.sin(a)[:, None]


def _rotate(x, turns, neighbours=False, sign=1.0):
    """x [L, heads, n], its first entries turned in pairs: neighbours, or entry i with entry i + half."""
    c, s = turns
    half = c.shape[-1]
    a, b = (x[..., 0:2 * half:2], x[..., 1:2 * half:2]) if neighbours else (x[..., :half], x[..., half:2 * half])
    u, v = a * c - sign * b * s, b * c + sign * a * s
    y = torch.stack([u, v], -1).flatten(-2) if neighbours else torch.cat([u, v], -1)
    return torch.cat([y, x[..., 2 * half:]], -1)


def _see(L, window=None, keep=0, chunk=None):
    i = torch.arange(L, device="cuda")
    see = i[None, :] <= i[:, None]
    if window is not None:
        see &= (i[:, None] - i[None, :] < window) | (i[None, :] < keep)
    if chunk is not None:
        see &= i[:, None] // chunk == i[None, :] // chunk
    return see


def _per_head(q, k, v, weigh):
    """Outputs [L, H, V] of heads that share kv heads; ``weigh(scores, head)`` makes weights of q k."""
    rep = q.shape[1] // k.shape[1]
    return torch.stack([weigh(q[:, h] @ k[:, h // rep].t(), h) @ v[:, h // rep] for h in range(q.shape[1])], 1)


def _sink_softmax(s, sink):
    top = torch.maximum(s.amax(-1, keepdim=True), sink)
    e = torch.exp(s - top)
    return e / (e.sum(-1, keepdim=True) + torch.exp(sink - top))


def _llama_weights(case, cfg, lay, fresh):
    """The layer's matrices as they multiply: q, k, v fused, gate and up apart (16 rows of each in turn), fp8 weights as
    the nearest of their format with a scale per output."""
    def mat(name, e=None):
        w = getattr(fresh, name)
        w = w if e is None else w[e]
        if case["weights"] == "fp8":
            s = w.float().abs().amax(1, keepdim=True) / 448.0
            w = (w.float() / s).to(torch.float8_e4m3fn).double() * s.double()
        return w.double()

    def glu(e=None):
        gu = mat("gate_up", e)
        gu = gu.view(-1, 2, 16, gu.shape[1])
        return gu[:, 0].flatten(0, 1), gu[:, 1].flatten(0, 1), mat("down", e)
    return mat, glu


def _llama_block(x, mat, glu, cfg, router=None):
    """x [L, W] -> [L, W]."""
    L, H, G, D, eps = x.shape[0], cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.rms_norm_eps
    z = _rms(x, eps) @ mat("qkv").t()
    turns = _turns(L, D, cfg.rope_theta)
    q, k = _rotate(z[:, :H * D].view(L, H, D), turns), _rotate(z[:, H * D:(H + G) * D].view(L, G, D), turns)
    hide = ~_see(L)
    o = _per_head(q, k, z[:, (H + G) * D:].view(L, G, D),
                  lambda s, h: torch.softmax((s * D ** -0.5).masked_fill(hide, -math.inf), -1))
    x = x + o.reshape(L, H * D) @ mat("o").t()
    h = _rms(x, eps)
    if router is None:
        g, u, d = glu()
        return x + (F.silu(h @ g.t()) * (h @ u.t())) @ d.t()
    p, e = torch.topk(torch.softmax(h @ router.t(), -1), cfg.num_experts_per_tok, -1)
    p = p / p.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for j in range(cfg.num_local_experts):
        t, c = (e == j).nonzero(as_tuple=True)
        g, u, d = glu(j)
        y[t] += ((F.silu(h[t] @ g.t()) * (h[t] @ u.t())) @ d.t()) * p[t, c, None]
    return x + y


def _scan(decay, k, v, q, S0=None, delta=None):
    """S <- decay S + k v^T, o = S^T q, token by token; [L, H, D] (values [L, H, V], ``decay`` of the keys' shape).  ``delta``
    [L, H]: the delta rule's step size, which writes v - S^T k."""
    L, H, D = k.shape
    S = torch.zeros(H, D, v.shape[-1], dtype=k.dtype, device=k.device)
    o = torch.empty(L, H, v.shape[-1], dtype=k.dtype, device=k.device)
    for t in range(L):
        S = S * decay[t][:, :, None]
        u = v[t]
        if delta is not None:
            u = delta[t][:, None] * (u - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    return o


def _clamped(g, u, limit):
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1)


def _hgrn2(h, w, sp, eps):
    L, H, D, V = h.shape[0], sp.heads, sp.dim, sp.vdim
    f = w["lower"] + (1 - w["lower"]) * torch.sigmoid(h @ w["f"].t() + w["f.b"])
    o = _scan(f.view(L, H, D), (1 - f).view(L, H, D), (h @ w["v"].t()).view(L, H, V), F.silu(h @ w["q"].t()).view(L, H, D))
    return (_rms(o, eps) * w["norm"]).reshape(L, H * V)


def _talking(h, w, sp, eps):
    L, H, G, D = h.shape[0], sp.heads, sp.kv_heads, sp.dim
    kr = h @ w["k"].t()
    q = (_rms(h @ w["q"].t(), eps) * w["q.norm"]).view(L, H, D)
    k, v = (_rms(kr, eps) * w["k.norm"]).view(L, G, D), kr.view(L, G, D)
    o = torch.empty(L, H, D, dtype=h.dtype, device=h.device)
    sl = 2.0 ** (-8.0 * torch.arange(1, H + 1, dtype=torch.float64, device="cuda") / H)
    for a in range(0, L, sp.chunk):
        b, i = min(L, a + sp.chunk), torch.arange(a, min(L, a + sp.chunk), dtype=torch.float64, device="cuda")
        raw = torch.einsum("ihd,jhd->hij", q[a:b], k[a:b].repeat_interleave(H // G, 1)) * sp.scale
        raw = raw - sl[:, None, None] * (i[:, None] - i[None, :])
        s = torch.einsum("hg,gij->hij", w["talk"], raw).masked_fill(~_see(b - a), -math.inf)
        o[a:b] = torch.einsum("hij,jhd->ihd", torch.softmax(s, -1), v[a:b].repeat_interleave(H // G, 1))
    return o.reshape(L, H * D) * torch.sigmoid(h @ w["g"].t())


def _latent(h, w, sp, eps):
    L, H, D, R, V, C = h.shape[0], sp.heads, sp.dim, sp.rot_dim, sp.vdim, sp.kv_rank
    turns = _turns(L, sp.rot_dims, sp.rot_base)
    q = ((_rms(h @ w["dq"].t(), eps) * w["dq.norm"]) @ w["uq"].t()).view(L, H, D + R)
    z = h @ w["dkv"].t()
    c, kr = _rms(z[:, :C], eps) * w["dkv.norm"], _rotate(z[:, None, C:], turns)
    q = torch.cat([q[..., :D], _rotate(q[..., D:], turns)], -1)
    k = torch.cat([(c @ w["uk"].t()).view(L, H, D), kr.expand(L, H, R)], -1)
    hide = ~_see(L)
    return _per_head(q, k, (c @ w["uv"].t()).view(L, H, V),
                     lambda s, i: _sink_softmax((s * sp.scale).masked_fill(hide, -math.inf), w["sink"][i])).reshape(L, H * V)


def _mlstm(h, w, sp, eps):
    L, H, D, V = h.shape[0], sp.heads, sp.dim, sp.vdim
    q, k, v = (h @ w["q"].t() * D ** -0.5).view(L, H, D), (h @ w["k"].t()).view(L, H, D), (h @ w["v"].t()).view(L, H, V)
    cap = lambda z: sp.gate_cap * torch.tanh(z / sp.gate_cap)  # noqa: E731
    i, f = cap(h @ w["i"].t() + w["i.b"]), F.logsigmoid(cap(h @ w["f"].t() + w["f.b"]))
    m, top = torch.zeros(H, dtype=h.dtype, device=h.device), []
    for t in range(L):
        m = torch.maximum(f[t] + m, i[t])
        top.append(m)
    m = torch.stack(top)
    a = torch.exp(f + torch.cat([torch.zeros_like(m[:1]), m[:-1]]) - m)[:, :, None].expand(L, H, D)
    y = _scan(a, k * torch.exp(i - m)[:, :, None], torch.cat([v, torch.ones_like(v[..., :1])], -1), q)
    den = torch.maximum(y[..., V:].abs(), torch.exp(-m)[:, :, None]) + 1e-6
    return _rms(y[..., :V] / den, eps).reshape(L, H * V) * w["norm"] * torch.sigmoid(h @ w["g"].t())


def _retention(h, w, sp, eps):
    L, H, D, V = h.shape[0], sp.heads, sp.dim, sp.vdim
    turns = _turns(L, sp.rot_dims, sp.rot_base)
    q, k = (_rotate((h @ w[n].t()).view(L, H, D), turns) for n in "qk")
    decay = torch.tensor(sp.decay, dtype=h.dtype, device="cuda")[None, :, None].expand(L, H, D)
    o = _scan(decay, k * D ** -0.5, (h @ w["v"].t()).view(L, H, V), q)
    return _rms(o, eps).reshape(L, H * V) * F.silu(h @ w["g"].t())


def _mixed(h, w, sp, eps):
    L, H, G, D, V = h.shape[0], sp.heads, sp.kv_heads, sp.dim, sp.vdim
    turns, vt = _turns(L, sp.rot_dims, sp.rot_base, sp.rot_scaling), _turns(L, V, sp.rot_base)
    q = _rotate(_rms((h @ w["q"].t()).view(L, H, D), eps) * w["q.norm"], turns)
    k = _rotate(_rms((h @ w["k"].t()).view(L, G, D), eps) * w["k.norm"], turns)
    v = _rotate((h @ w["v"].t()).view(L, G, V), vt)
    hide, zero = ~_see(L), torch.zeros((), dtype=h.dtype, device=h.device)
    p = torch.stack([_sink_softmax((sp.softcap * torch.tanh(q[:, i] @ k[:, i // (H // G)].t() * sp.scale / sp.softcap))
                                   .masked_fill(hide, -math.inf), zero) for i in range(H)])
    o = torch.stack([torch.einsum("g,gij->ij", w["talk"][i], p) @ v[:, i // (H // G)] for i in range(H)], 1)
    return (_rotate(o, vt, sign=-1.0) * torch.sigmoid(h @ w["g"].t())[:, :, None]).reshape(L, H * V)


def _window(h, w, sp, eps):
    L, H, G, D, V = h.shape[0], sp.heads, sp.kv_heads, sp.dim, sp.vdim
    turns = _turns(L, sp.rot_dims, sp.rot_base)
    q, k = (_rotate((h @ w[n].t()).view(L, m, D), turns, sp.neighbours) for n, m in (("q", H), ("k", G)))
    if sp.qk_norm:
        q, k = _rms(q, eps), _rms(k, eps)
    see = _see(L, sp.window, sp.keep_first)
    if sp.weights == "sigmoid":
        weigh = lambda s, i: torch.sigmoid(s * sp.scale + w["pb"][i]) * see  # noqa: E731
    else:
        weigh = lambda s, i: _sink_softmax((s * sp.scale).masked_fill(~see, -math.inf), w["sink"][i])  # noqa: E731
    return _per_head(q, k, (h @ w["v"].t()).view(L, G, V), weigh).reshape(L, H * V)


def _conv(x, w, bias=0.0):
    taps = w.shape[1]
    x = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return F.silu(sum(x[j:x.shape[0] - taps + 1 + j] * w[:, j] for j in range(taps)) + bias)


def _delta(h, w, sp, eps):
    L, H, G, D, V = h.shape[0], sp.heads, sp.kv_heads, sp.dim, sp.vdim
    q, k, v = (_conv(h @ w[n].t(), w[n + ".conv"]) for n in "qkv")
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = (unit(x.view(L, G, D)).repeat_interleave(H // G, 1) for x in (q, k))
    z = F.softplus((h @ w["a1"].t()) @ w["a2"].t() + w["dt_bias"]).view(L, H, D)
    o = _scan(torch.exp(-torch.exp(w["A_log"])[:, None] * z), k, v.view(L, H, V), q * D ** -0.5,
              delta=torch.sigmoid(h @ w["b"].t()))
    return (_rms(o, eps) * w["norm"]).reshape(L, H * V) * torch.sigmoid((h @ w["g1"].t()) @ w["g2"].t())


def _mamba(h, w, sp, eps):
    L, H, V, N, G, inner = h.shape[0], sp.heads, sp.vdim, sp.dim, sp.kv_heads, sp.inner
    z, xbc, dt = (h @ w["in"].t()).split([inner, inner + 2 * G * N, H], -1)
    x, B, C = _conv(xbc, w["conv"], w["conv.b"]).split([inner, G * N, G * N], -1)
    x = x.reshape(L, H, V)
    B, C = (t.reshape(L, G, N).repeat_interleave(H // G, 1) for t in (B, C))
    dt = F.softplus(dt + w["dt_bias"])
    a = torch.exp(-torch.exp(w["A_log"]) * dt)[:, :, None].expand(L, H, N)
    y = _scan(a, B * dt[:, :, None], x, C) + w["D"][:, None] * x
    return _group_norm(y.reshape(L, inner) * F.silu(z), eps, sp.norm_groups) * w["norm"]


def _gla(h, w, sp, eps):
    L, H, D, V = h.shape[0], sp.heads, sp.dim, sp.vdim
    a = torch.sigmoid((h @ w["a1"].t()) @ w["a2"].t() + w["a2.b"]) ** (1 / sp.tau)
    o = _scan(a.view(L, H, D), (h @ w["k"].t()).view(L, H, D), (h @ w["v"].t()).view(L, H, V),
              (h @ w["q"].t()).view(L, H, D) * D ** -0.5)
    return (_rms(o, eps) * w["norm"]).reshape(L, H * V) * F.silu(h @ w["g"].t())


_MIXERS = {"hgrn2": _hgrn2, "attention": _talking, "latent_attention": _latent, "mlstm": _mlstm, "retention": _retention,
           "mixed_attention": _mixed, "window_attention": _window, "gated_delta": _delta, "mamba2": _mamba, "gla": _gla}


def _sub(w, prefix):
    return {k[len(prefix):]: t for k, t in w.items() if k.startswith(prefix)}


def _mix(h, w, sp, eps):
    if sp.mixer != "pair":
        return _MIXERS[sp.mixer](h, w, sp, eps) @ w["o"].t()
    return sum(s * _mix(h, _sub(w, p), m, eps) for s, p, m in ((sp.left_scale, "left.", sp.left),
                                                             (sp.right_scale, "right.", sp.right)))


def _feed(h, w, sp):
    if sp.moe is not None:
        m = sp.moe
        s = torch.softmax(h @ w["router"].t(), -1)
        groups = s.view(-1, m.groups, m.experts // m.groups)
        keep = torch.zeros_like(groups[..., 0]).scatter_(1, torch.topk(groups.amax(-1), m.keep, -1).indices, 1.0)
        p, e = torch.topk((groups * keep[..., None]).flatten(1), m.top, -1)
        p = p / (p.sum(-1, keepdim=True) + 1e-20) * m.scale
        y = torch.sigmoid(h @ w["shared.sg"].t()) * (_clamped(h @ w["shared.gate"].t(), h @ w["shared.up"].t(), sp.limit)
                                                     @ w["shared.down"].t())
        for j in range(m.experts):
            t, c = (e == j).nonzero(as_tuple=True)
            a = _clamped(h[t] @ w[f"e{j}.gate"].t(), h[t] @ w[f"e{j}.up"].t(), m.limit)
            y[t] += (a @ w[f"e{j}.down"].t()) * p[t, c, None]
        return y
    if sp.ffn == "relu2":
        a = torch.relu(h @ w["up"].t()) ** 2
    elif sp.ffn == "gelu":
        a = F.gelu(h @ w["up"].t())
    elif sp.ffn == "silu_glu":
        a = F.silu(h @ w["gate"].t()) * (h @ w["up"].t())
    else:
        a = _clamped(h @ w["gate"].t(), h @ w["up"].t(), sp.limit)
    return a @ w["down"].t()


def _hybrid(ids, cfg, layers, top, rows):
    """Logits of ``rows`` of one sequence."""
    eps, W = cfg.rms_norm_eps, cfg.hidden_size
    norm = (lambda x: _layer_norm(x, eps)) if cfg.norm == "layer" else (lambda x: _group_norm(x, eps, cfg.norm_groups))
    x = top["embed"][ids] * cfg.embed_scale
    if cfg.embed_positions:
        c, s = _turns(len(ids), W, 10000.0)
        x = x + torch.stack([s, c], -1).view(len(ids), W)
    if cfg.embed_norm:
        x = norm(x)
    x0 = x
    for sp, w in zip(cfg.layers, layers):
        mixer, mlp = _sub(w, "mix."), _sub(w, "mlp.")
        if cfg.stream == "post":
            x = x + _rms(_mix(x, mixer, sp, eps), eps) * w["norm1"] * w["ls1"]
            if sp.ff:
                x = x + _rms(_feed(x, mlp, sp), eps) * w["norm2"] * w["ls2"]
            continue
        if sp.inject:
            x = torch.cat([x, x0], -1) @ top["loop_in"].t()
        h = norm(x) * w["norm1"]
        if sp.shift:
            h = h + (torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h) * w["shift"]
        y = _mix(h, mixer, sp, eps)
        if sp.parallel:
            y = y + _feed(h, mlp, sp)
        x = x + cfg.residual_mult * y
        if sp.ff and not sp.parallel:
            x = x + cfg.residual_mult * _feed(norm(x) * w["norm2"], mlp, sp)
    z = norm(x[rows]) * cfg.logit_scale @ top["head"][:cfg.vocab_size].t()
    return cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap) if cfg.logit_softcap else z


def exact(case, seed):
    cfg = _config(case)
    plain = dict(case, weights="bf16")
    w = _weights(plain, seed, cfg)
    if case["kind"] == "tune":
        return _exact_tune(case, seed, cfg, w)
    with torch.no_grad():
        first, later, _ = _inputs(case, seed, cfg, w)
        seqs = [torch.cat([f] + [r[i:i + 1] for r in later]) for i, f in enumerate(first)]
        if case["kind"] == "step":
            rows = [slice(n, n + 1) for n in _lengths(case)]
        elif case["role"] == "segment":
            rows = [slice(0, n + len(later)) for n in _lengths(case)]
        else:
            rows = [slice(n - 1, n + len(later)) for n in _lengths(case)]
        if cfg.hybrid:
            made = [{k: _d(t) for k, t in random_hybrid_tensors(cfg, i, "cuda:0", torch.bfloat16, seed % 10007).items()}
                    for i in range(len(cfg.layers))]
            top = {"embed": _d(w.embed), "head": _d(w.lm_head), "loop_in": None if w.loop_in is None else _d(w.loop_in)}
            outs = [_hybrid(ids, cfg, made, top, r) for ids, r in zip(seqs, rows)]
        else:
            xs = [_d(w.embed)[s] if case["role"] == "full" else _d(s) for s in seqs]
            for lay in w.layers:
                mat, glu = _llama_weights(case, cfg, lay, lay)
                xs = [_llama_block(x, mat, glu, cfg, None if lay.router is None else _d(lay.router)) for x in xs]
            outs = [x[r] for x, r in zip(xs, rows)]
            if case["role"] != "segment":
                head = _d(w.lm_head)
                outs = [_rms(x, cfg.rms_norm_eps) @ head.t() for x in outs]
        if case["kind"] == "generate" and case["role"] == "segment":
            ends = _lengths(case)
            return [torch.cat([o[:n] for o, n in zip(outs, ends)])] + \
                [torch.stack([o[n + k] for o, n in zip(outs, ends)]) for k in range(case["steps"])]
        if case["kind"] == "generate":
            return [torch.stack([o[k] for o in outs]) for k in range(case["steps"] + 1)]
        out = torch.cat(outs)
        return [out, None] if case["sample"] else out


def _exact_tune(case, seed, cfg, w):
    hidden, grad, prompts = _tune_inputs(case, seed, cfg)
    x0 = _d(hidden).requires_grad_(True)
    p0 = _d(prompts).requires_grad_(True) if prompts is not None else None
    outs = []
    with torch.enable_grad():
        for b in range(case["sessions"]):
            x = x0[b]
            for i, lay in enumerate(w.layers):
                if p0 is not None:
                    x = torch.cat([x[:case["prefix"]] + p0[i, b], x[case["prefix"]:]])
                x = _llama_block(x, *_llama_weights(case, cfg, lay, lay), cfg)
            outs.append(x)
        out = torch.stack(outs)
        grads = torch.autograd.grad(out, [x0] if p0 is None else [x0, p0], _d(grad))
    return [out.detach(), *grads]
