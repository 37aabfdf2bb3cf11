"""Products of few rows on 128 x 128 tiles (csrc/gemm_mid.hip) at the edges of tiles, parts and rings, which products take them, and
the wait states of their inline asm."""
import os
import re
import subprocess

import pytest
import torch

from src import ops
from src.models.config import PRESETS
from src.ops import build, prompt
from tests import test_tile_waits as waits
from tests.test_prompt_gemm import BF16, _want, gates_far_below_zero


# one stage, fewer than a ring's, a part of one; a few weight tiles and 65 to 130 of them, dealt in eights; a tile too few rows or
# columns, and one over; 3 row tiles of 88 weight tiles: more workgroups than CUs, the short ring
SHAPES = [(16, 64), (32, 128), (144, 192), (288, 320), (544, 2048), (2112, 4096), (4096, 1664), (8336, 640), (16640, 256), (11264, 512)]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 15, 64, 65, 128, 129, 300])
@pytest.mark.parametrize("N,K", SHAPES)
def test_products(M, N, K):
    """One sum of K exact products in 32 bits, in parts or whole and from any stage on, rounded to bf16 once."""
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    for epi, limit in ((0, 0.0), (1, 0.0), (1, 1.5), (4, 0.0), (prompt.COLUMNS, 0.0)):
        if epi == 1 and N % 32:
            continue
        v, want = (w.t().contiguous(), z) if epi == prompt.COLUMNS else (w, _want(z, epi, limit))
        cols = want.shape[1]
        room = torch.full((M + 130, cols), -3.0, dtype=torch.bfloat16, device="cuda")
        out = prompt._run_mid(x, v, room[:M], N, epi, limit)
        assert float((out.double() - want).norm() / want.norm()) < BF16
        assert bool((room[M:] == -3.0).all())
        assert torch.equal(out, prompt._run_mid(x, v, torch.empty_like(out), N, epi, limit))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(3, 64), (3, 4096)])  # (in one part and in several)
def test_gates_far_below_zero(M, K):
    ops.require_native()
    x, w, z = gates_far_below_zero("cuda")
    x, w = (torch.nn.functional.pad(t, (0, K - 64)) for t in (x, w))
    assert (torch.ops.mpamd.gemm_mid_ws(M, 32, K) > 0) == (K > 64)
    want = _want(z, 1, 0.0)
    got = prompt._run_mid(x, w, torch.empty(3, 16, dtype=torch.bfloat16, device="cuda"), 32, 1).double()
    assert float(((got - want) / want).abs().max()) < BF16 + 2e-5


@pytest.mark.gpu
def test_not_a_number_and_infinity_pass():
    ops.require_native()
    x = torch.ones(150, 4096, dtype=torch.bfloat16, device="cuda")
    x[3, 5], x[140, 600] = float("nan"), float("inf")
    w = torch.ones(32, 4096, dtype=torch.bfloat16, device="cuda")
    for epi in (0, 1, 4):
        y = prompt._run_mid(x, w, torch.empty(150, 16 if epi == 1 else 32, dtype=torch.bfloat16, device="cuda"), 32, epi)
        assert y[3].isnan().all() and y[140].isinf().all() and y[4:140].isfinite().all() and y[:3].isfinite().all()


@pytest.mark.gpu
def test_linear_takes_them(monkeypatch):
    """A row-major step where the table says so, ahead of the decode kernels that would pack it; a caller that does not ask, or whose
    packed weights are other ones, keeps what it had."""
    ops.require_native()
    monkeypatch.setitem(prompt._STATE, "mid", {(4096, 4096, 0): frozenset({4})})
    x, w = torch.randn(100, 4096, device="cuda").to(torch.bfloat16), torch.randn(4096, 4096, device="cuda").to(torch.bfloat16)
    calls, run = [], prompt._run_mid
    monkeypatch.setattr(prompt, "_run_mid", lambda *a: calls.append(a[0].shape[0]) or run(*a))
    want = x.double() @ w.double().t()
    for kw, n in (({"tiles": True}, 1), ({"tiles": True, "wp": ops.pack_weight(w)}, 1), ({}, 0), ({"wp": ops.pack_weight(w)}, 0),
                  ({"tiles": True, "policy": "hipblaslt"}, 0)):
        del calls[:]
        assert float((ops.linear(x, w, **kw).double() - want).norm() / want.norm()) < BF16 and len(calls) == n
    del calls[:]
    ops.linear(x[:90], w, tiles=True)
    assert not calls  # (another range of rows)
    ss = ops.norm_stats_buffer("cuda")[0]  # (rows of a fused norm: the decode kernels alone scale them)
    ss[0, :100] = (x.double().pow(2).sum(1) * 2 ** 20).long()
    kw = dict(wp=ops.pack_weight(w), ss_in=ss, eps=1e-5)
    assert torch.equal(ops.linear(x, w, tiles=True, **kw), ops.linear(x, w, **kw)) and not calls


def test_few_rows_of_large_packed_weights():
    """Where a step's weights are there packed as well: which rows leave the decode kernels."""
    for N, K, first in ((512, 512, 1), (6144, 4096, 1), (4096, 11008, 17), (28672, 4096, 17), (8192, 28672, 17), (57344, 8192, 33)):
        assert [prompt.ahead(M, N, K) for M in (first - 1, first)] == [first == 1, True], (N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,here", [(16, 0), (17, 1)])
def test_large_packed_weights(M, here, monkeypatch):
    ops.require_native()
    monkeypatch.setitem(prompt._STATE, "mid", {(4096, 11008, 0): frozenset({1})})
    x, w = torch.randn(M, 11008, device="cuda").to(torch.bfloat16), torch.randn(4096, 11008, device="cuda").to(torch.bfloat16)
    calls, run = [], prompt._run_mid
    monkeypatch.setattr(prompt, "_run_mid", lambda *a: calls.append(1) or run(*a))
    want = x.double() @ w.double().t()
    wp = ops.pack_weight(w)
    for kw, n in (({"wp": wp}, here), ({}, 1)):
        del calls[:]
        y = ops.linear(x, w, tiles=True, **kw)
        assert float((y.double() - want).norm() / want.norm()) < BF16 and len(calls) == n
    assert here or torch.equal(ops.linear(x, w, tiles=True, wp=wp), ops.linear(x, w, wp=wp))


def test_which_products(monkeypatch):
    monkeypatch.setitem(prompt._STATE, "mid", {(4096, 4096, 0): frozenset({1, 5})})
    for M, here in ((1, True), (32, True), (33, False), (128, False), (129, True), (192, True), (193, False), (385, False)):
        assert prompt.mid(M, 4096, 4096, 0) == here
    assert not prompt.mid(20, 4096, 4096, 1) and not prompt.mid(20, 4096, 8192, 0)  # (not timed)
    assert prompt.mid(8000, 512, 1024, 0) and not prompt.mid(8193, 512, 1024, 0) and not prompt.mid(100, 512, 1024 + 32, 0)
    # weights that no table holds: up to 8192 stages of tiles, or K 512; twice as much where the library needs a second pass
    for M, N, K, epi, here in ((2048, 1008, 4096, 0, True), (2049, 1008, 4096, 0, False), (8192, 768, 4096, 0, False),
                               (4096, 992, 4096, 1, True), (4097, 992, 4096, 1, False), (4096, 1024, 4032, 4, True), (8192, 1024, 4032, 4, False),
                               (8192, 4096, 512, 0, True), (8192, 4096, 512, 8, True), (8192, 4096, 576, 0, False), (8192, 4064, 1024, 1, True),
                               (8192, 2032, 1088, 1, False), (8192, 4096, 768, 8, False), (300, 4080, 1024, 0, True)):
        assert prompt.mid(M, N, K, epi) == here, (M, N, K, epi)
    x, w = torch.zeros(20, 512, dtype=torch.bfloat16), torch.zeros(512, 512, dtype=torch.bfloat16)
    assert not prompt.ok(x, w, 0) and torch.equal(prompt.gemm_columns(x, w), x @ w)  # the CPU
    monkeypatch.setenv("MPAMD_KERNEL_TABLE", "0")
    assert not prompt.mid(20, 512, 1024, 0)


def test_committed_tables():
    """Every preset's projections were timed; the other table of few rows holds no range that these tiles take whole."""
    mid, few = prompt._load(prompt.MID_TABLE), prompt._load(prompt.FEW_TABLE)
    for s in {s for c in PRESETS.values() for f in (prompt.shapes, prompt.train_shapes) for s in f(c)}:
        assert mid[s] <= set(range(1, len(prompt.MID) + 1))
        assert not any(parts <= mid[s] for r, parts in {1: {1}, 2: {2}, 3: {3, 4}, 4: {5, 6}}.items() if r in few[s])
    for r, rows in prompt.MID_ROWS.items():
        assert all((prompt.MID[r - 2] if r > 1 else 0) < M <= prompt.MID[r - 1] for M in rows)


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "mid.s")
    subprocess.run([build.HIPCC, "-O3", "-fPIC", "-std=c++17", f"--offload-arch={build.ARCH}", "-I" + build.CSRC, *build.DEVICE_FLAGS,
                    "-S", "--cuda-device-only", os.path.join(build.CSRC, "gemm_mid.hip"), "-o", out],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(out) as f:
        return list(waits._functions(f.read(), "gemm_mid_kernel"))


def test_wait_states(assembly):
    """As the 256 x 256 tiles': a product's operands are two wait states old, sums are read 16 states after their last product, loads in
    asm have their own m0 and waits, stores end with the buffer."""
    assert len(assembly) == 8
    waits.test_sums_are_made_before_they_are_read(assembly)
    loads = 0
    for name, code, before in assembly:
        assert sum(o.mfma for o in code) == 48, name  # 32 of a stage of a whole tile, 16 of a half one
        assert not any("m0" in o.writes for o in code if o.block), name
        for i, o in enumerate(code):
            if o.mfma:
                used = o.reads | o.writes
                assert waits._since(code, before, i, lambda p: p.valu and p.writes & used, 2) >= 2, (name, o.text)
            if o.block and o.name.startswith("buffer_load"):
                loads += 1
                first = next(k for k in range(i, -1, -1) if k == 0 or code[k - 1].block != o.block)
                assert sum(p.waits for p in code[first:i]) >= 5, name
                put = next(k for k in range(first - 1, -1, -1) if "m0" in code[k].writes)
                assert not any(p.name.startswith("buffer_load") for p in code[put:first]), name
            if o.name.startswith("buffer_store"):
                assert re.search(r"s\[\d+:\d+\], 0 offen", o.text), (name, o.text)
    assert loads == 48
