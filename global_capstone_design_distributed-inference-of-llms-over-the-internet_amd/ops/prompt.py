"""Products of prompt-sized steps (csrc/gemm_prompt.hip) and when they run in place of the library's.

``gemm``: y = epilogue(x w^T) over row-major bf16 operands, the gate / relu epilogues of a feed-forward in the same kernel;
``gemm_columns``: y = x w, a gradient's way back through a projection.
The library's rate depends on its choice of solution, from 0.55 to 1.65 PFLOP/s over neighbouring row counts; this kernel's
on how its tiles, 256 wide and 128 to 256 high, fill 256 CUs, 1.2 to 1.6.  So the choice is measured, as it is for the decode GEMMs, for
the callers that ask (``tiles`` of ``ops.linear``: stages and fine-tuning): shapes in the committed table
(``python -m src.ops.tune --prompt``: every projection of every preset, steps of 257 to 8192 rows, weights that no cache holds,
as a model's do not stay there from one step to the next) run here at the row-tile
counts where this kernel was at least as fast at all three row counts timed inside the tile, and 3 % faster on average, in
both of two sweeps (one sweep differs from the next in about a third of the shapes, at counts where the two are close; the
committed table of more than 256 rows also holds 49 counts, of 919, that an earlier pair of sweeps had given to tiles of 256 rows, and
that were at least as fast at all three row counts when they were timed once more, with the heights that they have now).

Up to 384 rows there are tiles of 128 x 128 as well (csrc/gemm_mid.hip), by a table of theirs, timed against what runs without
them: 66 rows of Mistral-7B, forward and backward, 1031 -> 832 us.  The library's call costs the host 21 us, theirs 13, so they stay
where they are up to 3 % slower on the GPU.  Weights of less than 4M elements go there by a rule (``mid``): a prompt of 153 tokens
of a 512-wide model, 503 -> 381 us for two blocks.  (Ranges that were timed at 8, 16 and 32 rows hold at 1 to 7 too: 1.0 to 1.7 times as
fast as the library's at 33 of 36 shapes, 0.93 at the worst.)
A third table holds those few of 1 to 256 rows that are best on the large tiles.

Everything else keeps the library.  (No rule on the shape alone holds at the shapes that were timed: "less than a wave of
tiles, K from 10240 on, parts that fill 218 CUs or more" picks the slower one at 10 of 31 row-tile counts.)
"""
from __future__ import annotations

import itertools
import json
import os
import threading
from typing import Dict, FrozenSet, Iterable, Optional, Tuple

import torch

TABLE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned", "prompt_gemm_gfx950.json")
FEW_TABLE = TABLE.replace("prompt_gemm", "prompt_few")  # the same of few rows: 1 to 4 for up to 32, 64, 128, 256
MID_TABLE = TABLE.replace("prompt_gemm", "prompt_mid")  # those that the 128 x 128 tiles make, in ``MID``'s ranges
COLUMNS = 8  # in an epilogue's place: x w
EPILOGUES = (0, 1, 4, COLUMNS)
TILE, MAX_ROWS = 256, 8192
FEW = (32, 64, 128, TILE)  # (a tile of up to 128 rows takes half the products; the library's times jump at all four)
MID = (32, 64, 96, 128, 192, 256, 384)
SMALL = 1 << 22  # elements of a weight that no table holds
Shape = Tuple[int, int, int]  # N, K, epilogue

_LOCK = threading.Lock()
_STATE: dict = {"table": None, "few": None, "mid": None}
_PATHS = {"table": TABLE, "few": FEW_TABLE, "mid": MID_TABLE}


def _key(shape: Shape) -> str:
    return "N%dxK%de%d" % shape


def _load(path: str) -> Dict[Shape, FrozenSet[int]]:
    with open(path) as f:
        t = json.load(f)
    out = {}
    for s, tiles in t.get("tiles", {}).items():
        n, rest = s[1:].split("xK")
        k, e = rest.split("e")
        out[(int(n), int(k), int(e))] = frozenset(tiles)
    return out


def table(name: str = "table") -> Dict[Shape, FrozenSet[int]]:
    """(N, K, epilogue) -> row-tile counts at which the kernel runs (read once; MPAMD_KERNEL_TABLE=0: none); ``few``: the
    same of ``FEW``'s ranges; ``mid``: of ``MID``'s, those at which ``gemm_mid`` does."""
    with _LOCK:
        if _STATE[name] is None:
            path = _PATHS[name]
            on = os.environ.get("MPAMD_KERNEL_TABLE") != "0" and os.path.exists(path)
            _STATE[name] = _load(path) if on else {}
        return _STATE[name]


def shape_ok(M: int, N: int, K: int, epilogue: int) -> bool:
    """Does the kernel cover the shape?  (Byte offsets of a piece are 32 bits.)"""
    return (epilogue in EPILOGUES and M >= 1 and K >= 64 and K % 64 == 0 and N % (32 if epilogue == 1 else 16) == 0 and
            N >= 16 and M * K < 1 << 31 and N * K < 1 << 31)


def chosen(M: int, N: int, K: int, epilogue: int) -> bool:
    """Does a step of M rows run this product here?"""
    return TILE < M <= MAX_ROWS and shape_ok(M, N, K, epilogue) and -(-M // TILE) in table().get((N, K, epilogue), ())


def few(M: int, N: int, K: int, epilogue: int) -> bool:
    """The same of a step of few rows, whose weights have no packed copy."""
    return M <= TILE and shape_ok(M, N, K, epilogue) and \
        next(i for i, n in enumerate(FEW, 1) if M <= n) in table("few").get((N, K, epilogue), ())


def mid(M: int, N: int, K: int, epilogue: int) -> bool:
    """Does a step of M rows run this product on the 128 x 128 tiles?"""
    if not shape_ok(M, N, K, epilogue) or M > MAX_ROWS:
        return False
    if N * K < SMALL:
        # Up to 8192 stages of all tiles they take 6 % less than the library's on average, and where they take more (1280 x 1280
        # of 300 rows 13.7, 7.5 us) no more than its call costs the host beyond theirs; past that only where K is small, or the library's
        # pass over what it wrote is saved: 8192 x 768 x 4096 65.7, 50.5 us, but 4096 x 16384 x 128 40.4, 39.8 and 8192 x 4064 x 1024
        # gated 69.4, 113.  That pass moves both lines to twice as much (4096 x 2048 x 1984 gated 34.6, 39.7, of 5000 rows 49.1, 45.7).
        more = 2 if epilogue in (1, 4) else 1
        stages = -(-M // 128) * -(-N // 128) * (K // 64)
        return (K <= 512 * more or stages <= 8192 * more) and os.environ.get("MPAMD_KERNEL_TABLE") != "0"
    return M <= MID[-1] and next(i for i, n in enumerate(MID, 1) if M <= n) in table("mid").get((N, K, epilogue), ())


def ahead(M: int, N: int, K: int) -> bool:
    """Are the 128 x 128 tiles ahead of packing M rows for the decode kernels, where the weights are there packed as well?  Those
    stream large weights of few rows faster (us of the tiles, of packing and the decode kernel): 8 rows of 4096 x 11008 21.4, 19.3, of
    6144 x 4096 13.7, 15.2; 16 rows of 8192 x 8192 28.3, 25.3, of 28672 x 4096 gated 41.6, 42.0; 17 rows of 4096 x 11008 22.0, 25.5, of
    8192 x 8192 28.4, 27.2; 24 rows of 57344 x 8192 gated 163, 146, 32 rows 164, 161, 48 rows 165, 201."""
    return N * K <= 1 << 25 or M > 32 or (M > 16 and N * K <= 1 << 28)


def reads(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Are these operands that the kernel reads (types, strides, alignments), in a call that is not differentiated?"""
    if x.dim() != 2 or w.dim() != 2 or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        return False
    if not (x.is_cuda and w.device == x.device and w.is_contiguous() and x.stride(1) == 1 and x.stride(0) % 8 == 0 and
            x.stride(0) >= x.shape[1] and x.shape[0] * x.stride(0) < 1 << 31):
        return False
    return x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and not (
        torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))


def ok(x: torch.Tensor, w: Optional[torch.Tensor], epilogue: int) -> bool:
    """Is this product of rows [M, K] with weights [N, K] one that runs here?  Callers that differentiate it, and operands
    the kernel does not read, keep the library's."""
    if w is None or x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1]:
        return False
    shape = x.shape[0], w.shape[0], w.shape[1], epilogue
    return (mid(*shape) or chosen(*shape) or few(*shape)) and reads(x, w)


def _run(x, w, y, N: int, epilogue: int, limit: float = 0.0, frags: int = 0):
    """``frags``: tiles of 32 times as many rows (4 to 8; 0: what the estimate says)."""
    need = torch.ops.mpamd.gemm_prompt_ws(x.shape[0], N, x.shape[1], frags)
    ws = torch.empty(need, dtype=torch.float32, device=x.device) if need else None
    torch.ops.mpamd.gemm_prompt(x, w, y, ws, epilogue, limit, frags)
    return y


def _run_mid(x, w, y, N: int, epilogue: int, limit: float = 0.0):
    need = torch.ops.mpamd.gemm_mid_ws(x.shape[0], N, x.shape[1])
    ws = torch.empty(need, dtype=torch.float32, device=x.device) if need else None
    torch.ops.mpamd.gemm_mid(x, w, y, ws, epilogue, limit)
    return y


def gemm(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None, epilogue: int = 0, limit: float = 0.0,
         mid: bool = False):
    """epilogue 0: x w^T; 1: the gated forms over gate / up rows in blocks of 16 (``limit`` 0: silu); 4: max(., 0)^2."""
    M, N = x.shape[0], w.shape[0]
    cols = N // 2 if epilogue == 1 else N
    y = out if out is not None and out.is_contiguous() and out.dtype == x.dtype and out.data_ptr() % 16 == 0 else \
        torch.empty(M, cols, dtype=x.dtype, device=x.device)
    (_run_mid if mid else _run)(x, w, y, N, epilogue, limit)
    return y if out is None or y is out else out.copy_(y)


def gemm_columns(x: torch.Tensor, w: torch.Tensor, always: bool = False) -> torch.Tensor:
    """x w of rows [M, K] and weights [K, N]: on the kernel where the table says so (or ``always``), else the library's."""
    run = _run if always else None
    if not always and x.dim() == 2 and w.dim() == 2 and x.shape[1] == w.shape[0]:
        shape = x.shape[0], w.shape[1], w.shape[0], COLUMNS
        run = _run_mid if mid(*shape) else _run if chosen(*shape) or few(*shape) else None
    if run and (always or reads(x, w)):
        return run(x, w, torch.empty(x.shape[0], w.shape[1], dtype=x.dtype, device=x.device), w.shape[1], COLUMNS)
    return torch.mm(x, w)


# ------------------------------------------------------------------ the table
def shapes(cfg) -> Iterable[Shape]:
    """Row-major projections of a model's prompts."""
    H = cfg.hidden_size
    out = set()
    if cfg.hybrid:
        for sp in cfg.layers:
            out |= {(sp.in_rows, H, 0), (H, sp.o_cols, 0)}
            if sp.mixer == "latent_attention":
                out.add((sp.q_rows, sp.q_rank, 0))
            if sp.ff and not sp.parallel:
                out |= {(sp.ff_rows, H, 1 if sp.glu else 4 if sp.ffn == "relu2" else 0), (H, sp.ff, 0)}
        if cfg.injects:
            out.add((H, 2 * H, 0))
    elif cfg.model_type != "gpt2":
        out = {(cfg.q_dim + 2 * cfg.kv_dim, H, 0), (H, cfg.q_dim, 0)}
        if not cfg.is_moe:
            out |= {(2 * cfg.intermediate_size, H, 1), (H, cfg.intermediate_size, 0)}
    return sorted(s for s in out if shape_ok(MAX_ROWS, *s) and s[0] * s[1] >= 1 << 22)


def train_shapes(cfg) -> Iterable[Shape]:
    """What fine-tuning adds: gate / up rows as they are, and every projection's way back."""
    from . import train

    H, F, Q, A = cfg.hidden_size, cfg.intermediate_size, cfg.q_dim, cfg.q_dim + 2 * cfg.kv_dim
    out = {(2 * F, H, 0), (F, H, COLUMNS), (H, 2 * F, COLUMNS), (Q, H, COLUMNS), (H, A, COLUMNS)} if train.shape_ok(cfg) else set()
    return sorted(s for s in out if shape_ok(MAX_ROWS, *s) and s[0] * s[1] >= 1 << 22)


def agreed(sweeps: Iterable[Dict[Shape, list]]) -> Dict[Shape, list]:
    """The row-tile counts that all sweeps give."""
    first, *rest = sweeps
    return {s: [m for m in v if all(m in r[s] for r in rest)] for s, v in first.items()}


ROWS = {m: (TILE * m - 251, TILE * m - 124, TILE * m) for m in range(2, MAX_ROWS // TILE + 1)}
FEW_ROWS = {1: (8, 16, 32), 2: (33, 48, 64), 3: (65, 96, 128), 4: (129, 192, 256)}
MID_ROWS = {1: (8, 16, 32), 2: (33, 48, 64), 3: (65, 80, 96), 4: (97, 112, 128), 5: (129, 160, 192), 6: (193, 224, 256),
            7: (257, 320, 384)}


def tune(todo: Iterable[Shape], device="cuda", log=None, rows=ROWS, kernel=None) -> Dict[Shape, list]:
    """The row-tile counts of every shape at which the kernel is faster, in both of two sweeps (``rows``: what is timed of
    each; ``kernel``: ``_run_mid``, else ``_run``)."""
    todo = list(todo)
    return agreed([sweep(todo, device, log, rows, kernel or _run) for _ in range(2)])


def sweep(todo: Iterable[Shape], device="cuda", log=None, rows=ROWS, kernel=None) -> Dict[Shape, list]:
    """Time both products over the row-tile counts of every shape, best of three rounds in turn: the kernel and the library's, or
    ``_run_mid`` and what would run in its place, where the library's call costs the host 8 us more, which is what the 3 % are for
    elsewhere."""
    from . import hybrid, require_native, swiglu, use_tuned_gemms

    kernel = kernel or _run
    require_native()
    use_tuned_gemms()

    def ms(f, n=4):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        f()
        a.record()
        for _ in range(n):
            f()
        b.record()
        b.synchronize()
        return a.elapsed_time(b) / n

    got = {}
    for N, K, epi in todo:
        # (as many weights as push each other out of the 256 MB of cache; what a step's rows are was just written)
        many = max(1, min(8, -(-(600 << 20) // (2 * N * K))))
        ws = [torch.empty(*((K, N) if epi == COLUMNS else (N, K)), device=device).normal_(0, 0.02).to(torch.bfloat16)
              for _ in range(many)]
        turn = itertools.cycle(ws)
        tiles = []
        for m, counts in rows.items():
            ratios = []
            for M in counts:
                x = torch.randn(M, K, device=device).to(torch.bfloat16)
                z = torch.empty(M, N, dtype=x.dtype, device=device)
                y = torch.empty(M, N // 2 if epi == 1 else N, dtype=x.dtype, device=device)

                def lib():
                    if epi == COLUMNS:
                        return torch.mm(x, next(turn), out=z)
                    torch.mm(x, next(turn).t(), out=z)
                    if epi == 1:
                        swiglu(z, out=y)
                    elif epi == 4:
                        hybrid.relu2(z, y)

                def tile():
                    kernel(x, next(turn), y, N, epi)

                def old():
                    _run(x, next(turn), y, N, epi)

                other = old if kernel is _run_mid and (few(M, N, K, epi) or chosen(M, N, K, epi)) else lib
                t = [min(v) for v in zip(*[(ms(other), ms(tile)) for _ in range(3)])]
                ratios.append(t[0] / t[1])
            if min(ratios) >= (0.97 if kernel is _run_mid else 1.0) and sum(ratios) / 3 >= (1.0 if kernel is _run_mid else 1.03):
                tiles.append(m)
        got[(N, K, epi)] = tiles
        if log:
            log(f"{_key((N, K, epi))}: {tiles}")
    return got


def save(path: str, got: Dict[Shape, list]) -> None:
    with open(path, "w") as f:
        f.write('{\n "arch": "gfx950",\n "tiles": {\n')
        f.write(",\n".join(f'  "{_key(s)}": {json.dumps(got[s])}' for s in sorted(got)))
        f.write("\n }\n}\n")
