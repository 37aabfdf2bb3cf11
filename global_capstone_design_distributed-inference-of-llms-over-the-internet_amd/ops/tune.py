"""Write the committed decode-kernel table (``ops.KERNEL_TABLE``) on an MI355X.

    python -m src.ops.tune                       # every preset the benches and tests run
    python -m src.ops.tune --models llama2-7b --batches 64 --out /tmp/t.json

For each model a full-depth stage with random-init weights is built with no table loaded
(``MPAMD_KERNEL_TABLE=0``), so its executor times every decode GEMM shape it uses (``autotune_gemm``
/ ``autotune_w8`` / ``autotune_qkv_fold``: M buckets 4..64), then ``warmup_serving`` runs the
end-to-end qkv-fold A/B of each decode batch in ``--batches``.  The resulting choices - one entry
per (row bucket, N, K, epilogue) and one fold decision per (graph batch bucket, N, K) - are
written as JSON.  Executors load that file by default, so every box running the tree runs the
same kernel mix (``ops.load_kernel_table``) and bench records carry its sha.

``--missing N`` adds what the table lacks, and changes nothing that it has: every decode product that some preset
(of ``--models``, default all, fp8 forms among them) would time at start-up, in N processes, and the folds of the Llama presets'
decode batches; the choice that won most often enters.  One such race is not enough: of 197 products, three processes
agreed on 139.  With every choice in the table, two processes give the same bits.

``--prompt`` writes the table of prompt products (``ops.prompt.TABLE``) instead: every projection of every preset, both
kernels timed over the row-tile counts of steps of 257 to 8192 rows, twice; a count enters where both sweeps agree.
"""
from __future__ import annotations

import argparse
import collections
import dataclasses
import gc
import os
import subprocess
import sys
import tempfile
import time


def every_spec() -> list:
    """Every preset that decodes with packed weights, and the fp8 form of those that have one."""
    from ..models.config import PRESETS

    names = [n for n, c in PRESETS.items() if c.model_type != "gpt2"]
    return names + [n + ":fp8" for n in names if not PRESETS[n].hybrid and not PRESETS[n].is_moe]


def stage(spec: str, whole: bool, batch: int = 4, device="cuda"):
    """An executor over the whole preset, or over one block of each kind that it has with its embedding and head: all its
    products."""
    from ..models.config import resolve_model
    from ..models.weights import random_stage_weights
    from ..runtime.executor import StageExecutor

    name, _, opt = spec.partition(":")
    cfg = resolve_model(name)
    n = cfg.num_hidden_layers
    if not whole:
        layers = tuple(dict.fromkeys(cfg.layers)) if cfg.hybrid else ()
        n = len(layers) or 1
        cfg = dataclasses.replace(cfg, layers=layers, num_hidden_layers=n) if cfg.hybrid else cfg
    w = random_stage_weights(cfg, 0, n, has_embed=True, has_head=True, device=device, seed=0, fp8=opt == "fp8")
    return StageExecutor(cfg, w, device, max_sessions=batch + 8, max_seq_len=512, kv_cache_bytes=8 << 30, graph_max_batch=64,
                         max_tokens_per_step=max(8192, 128 * batch), warmup=False)


def elect(sweeps) -> dict:
    """One table of several: each entry's most frequent value (of equals, the one that came first)."""
    out = {}
    for part in {p: None for t in sweeps for p in t if isinstance(t[p], dict)}:
        out[part] = {k: collections.Counter(t[part][k] for t in sweeps if k in t[part]).most_common(1)[0][0]
                     for k in sorted({k for t in sweeps for k in t.get(part, {})})}
    return out


def tune_missing(specs, batches, out=None) -> int:
    """This process' choices for the products that the table lacks, or (``batches``) for the folds of whole models."""
    import torch

    from .. import ops

    if not torch.cuda.is_available():
        print("tune: needs an MI355X", file=sys.stderr)
        return 2
    os.environ["MPAMD_GEMM_AUTOTUNE"] = "1"
    ops.load_kernel_table()
    ops.TUNE_ROUNDS = 24
    for spec in specs:
        ex = stage(spec, bool(batches), max(batches, default=4))
        for b in batches:
            ex.warmup_serving(b, 128)
        del ex
        gc.collect()
        torch.cuda.empty_cache()
    print(f"tune: {','.join(specs)}: {len(ops.kernel_table_report()['tuned_at_runtime'])} products timed", flush=True)
    ops.save_kernel_table(out)
    return 0


def tune_missing_often(specs, sweeps: int, batches, out=None) -> int:
    """``tune_missing`` in ``sweeps`` processes for each preset.  With the 3 rounds that a start takes its time for, what ran before
    decides: 4-row products of 16512 x 4096 went to 'lds42' in 9 of 9 fresh processes, at 30.4 us where 'pk' takes 28.1."""
    import json

    from .. import ops

    out = out or ops.KERNEL_TABLE
    ops.load_kernel_table()
    folds = [s for s in specs if s.split(":")[0] in ("llama2-7b", "llama3-8b", "llama3-70b")]
    with tempfile.TemporaryDirectory() as tmp:
        for todo, more in ((specs, []), (folds, ["--batches", ",".join(map(str, batches))])):
            base, got = ops.kernel_table(), []
            for spec in todo:
                for _ in range(sweeps):
                    path = os.path.join(tmp, "t.json")
                    subprocess.run([sys.executable, "-m", __spec__.name, "--missing", "1", "--models", spec, "--out", path, *more],
                                   check=True)
                    with open(path) as f:
                        t = json.load(f)
                    if t == base:
                        break  # nothing to time
                    got.append(t)
            t = elect([base] + got)
            for p in t:
                for k in t[p]:
                    votes = collections.Counter(g[p][k] for g in got if k in g[p])
                    if len(votes) > 1:
                        print(f"tune: {p} {k}: {dict(votes)}", flush=True)
            ops.set_kernel_table(t)
            sha = ops.save_kernel_table(out)
            os.environ["MPAMD_KERNEL_TABLE"] = out
    print(f"tune: wrote {out} (sha {sha})", flush=True)
    return 0


def tune_prompt(out=None) -> int:
    import torch

    from ..models.config import PRESETS
    from . import prompt

    if not torch.cuda.is_available():
        print("tune: needs an MI355X", file=sys.stderr)
        return 2
    todo = sorted({s for cfg in PRESETS.values() for f in (prompt.shapes, prompt.train_shapes) for s in f(cfg)})
    log = lambda m: print(f"tune: {m}", file=sys.stderr, flush=True)  # noqa: E731
    prompt.save(out or prompt.TABLE, prompt.tune(todo, log=log))
    few = (out + ".few") if out else prompt.FEW_TABLE
    prompt.save(few, prompt.tune(todo, log=log, rows=prompt.FEW_ROWS))
    return tune_mid(out)


def tune_mid(out=None) -> int:
    """What the 128 x 128 tiles make faster than what runs without them, by the tables of the others."""
    from ..models.config import PRESETS
    from . import prompt

    todo = sorted({s for cfg in PRESETS.values() for f in (prompt.shapes, prompt.train_shapes) for s in f(cfg)})
    prompt.save((out + ".mid") if out else prompt.MID_TABLE, prompt.tune(
        todo, log=lambda m: print(f"tune: {m}", file=sys.stderr, flush=True), rows=prompt.MID_ROWS, kernel=prompt._run_mid))
    return 0


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__.split("\n\n")[0])
    ap.add_argument("--models", default=None, help="comma-separated presets; ':fp8' = fp8 (W8A16) projection weights; "
                    "default: small-llama,tiny-llama,llama2-7b,llama3-8b,llama3-70b:fp8, or all with --missing")
    ap.add_argument("--batches", default=None, help="decode batches whose qkv-fold A/B is pinned (64; 24,32,48,64 with --missing)")
    ap.add_argument("--prompt-len", type=int, default=128)
    ap.add_argument("--out", default=None, help="default: the committed table path")
    ap.add_argument("--prompt", action="store_true", help="time the prompt products of every preset")
    ap.add_argument("--prompt-mid", action="store_true", help="time only those of few rows on the 128 x 128 tiles")
    ap.add_argument("--missing", type=int, default=0, metavar="N", help="add what the table lacks, by N processes")
    a = ap.parse_args(argv)
    if a.prompt:
        return tune_prompt(a.out)
    if a.prompt_mid:
        return tune_mid(a.out)
    batches = [int(b) for b in (a.batches or "").split(",") if b]
    if a.missing:
        specs = [m for m in (a.models or "").split(",") if m] or every_spec()
        return tune_missing(specs, batches, a.out) if a.missing == 1 else \
            tune_missing_often(specs, a.missing, batches or [24, 32, 48, 64], a.out)
    os.environ["MPAMD_KERNEL_TABLE"] = "0"   # time everything: nothing pre-loaded
    os.environ.setdefault("MPAMD_GEMM_AUTOTUNE", "1")
    import torch

    from .. import ops
    from ..models.config import resolve_model
    from ..models.weights import random_stage_weights
    from ..runtime.executor import StageExecutor

    if not torch.cuda.is_available():
        print("tune: needs an MI355X", file=sys.stderr)
        return 2
    batches = batches or [64]
    for spec in [m for m in (a.models or "small-llama,tiny-llama,llama2-7b,llama3-8b,llama3-70b:fp8").split(",") if m]:
        name, _, opt = spec.partition(":")
        cfg = resolve_model(name)
        t0 = time.time()
        w = random_stage_weights(cfg, 0, cfg.num_hidden_layers, has_embed=True, has_head=True, device="cuda",
                                 seed=0, fp8=opt == "fp8")
        B = max(batches)
        ex = StageExecutor(cfg, w, "cuda", max_sessions=B + 8, max_seq_len=512, kv_cache_bytes=8 << 30,
                           graph_max_batch=B, max_tokens_per_step=B * a.prompt_len, warmup=False)
        if cfg.model_type != "gpt2":
            for b in batches:
                ex.warmup_serving(b, a.prompt_len)
        print(f"tune: {spec} done in {time.time() - t0:.1f}s; fold {ex.qkv_fold_by_bucket} "
              f"ab {getattr(ex, 'qkv_fold_ab_ms', {})}", file=sys.stderr, flush=True)
        del ex, w
        gc.collect()
        torch.cuda.empty_cache()
    out = a.out or ops.KERNEL_TABLE
    sha = ops.save_kernel_table(out)
    print(f"tune: wrote {out} (sha {sha})", flush=True)
    return 0


if __name__ == "__main__":
    raise SystemExit(main())
