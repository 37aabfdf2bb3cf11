"""Prompt products (csrc/gemm_prompt.hip) at the edges of their tiles and parts, and which products take them."""
import os

import pytest
import torch

from src import ops
from src.ops import prompt

# bf16 has 7 stored bits: a value in [1, 2) is rounded by at most half a unit of 2^-7, so by 2^-8 of itself
BF16 = 2.0 ** -8


def _want(z, epi, limit):
    if epi == 4:
        return z.clamp_min(0) ** 2
    if epi == 0:
        return z
    v = z.view(z.shape[0], -1, 2, 16)
    g, u = v[:, :, 0].flatten(1), v[:, :, 1].flatten(1)
    if not limit:
        return torch.nn.functional.silu(g) * u
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1)


@pytest.fixture(params=[0, 8], ids=["estimate", "256rows"])
def height(request, monkeypatch):
    """Tiles as high as the estimate says, and of 256 rows, which the sizes below are made for."""
    run = prompt._run
    monkeypatch.setattr(prompt, "_run", lambda *a: run(*a, frags=request.param))
    return request.param


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 64, 65, 255, 256, 257, 640])
@pytest.mark.parametrize("N,K", [(16, 64), (32, 128), (256, 192), (288, 320), (544, 2048), (4096, 1664)])
def test_products(M, N, K, height):
    """One sum of K exact products in 32 bits (in parts or whole), rounded to bf16 once."""
    ops.require_native()
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g).to(torch.bfloat16)[:, :K]
    w = torch.randn(N, K, generator=g).div(K ** 0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    xd = torch.empty(M, K + 8, dtype=x.dtype, device="cuda")[:, :K].copy_(x)  # rows apart, as in a wider matrix
    for epi, limit in ((0, 0.0), (1, 0.0), (1, 1.5), (4, 0.0)):
        if epi == 1 and N % 32:
            continue
        out = torch.full((M, N // 2 if epi == 1 else N), float("nan"), dtype=torch.bfloat16, device="cuda")
        got = prompt.gemm(xd, w.cuda(), out, epi, limit)
        want = _want(z, epi, limit)
        assert got is out and float((out.double().cpu() - want).norm() / want.norm()) < BF16
        assert torch.equal(out, prompt.gemm(xd, w.cuda(), None, epi, limit))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4100, 4096, 2048), (300, 4096, 11008), (1030, 4096, 10240), (2049, 2304, 4096)])
@pytest.mark.parametrize("height", [8], indirect=True)
def test_left_over_tiles_in_parts(M, N, K, height):
    ops.require_native()
    assert torch.ops.mpamd.gemm_prompt_ws(M, N, K, height) > 0
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    for epi in (0, 1):
        r = _want(want, epi, 0.0)
        assert float((prompt.gemm(x, w, None, epi).double() - r).norm() / r.norm()) < BF16


# more tiles than workgroups (256): a ring of five slots runs on into the next tile, of 1, 3 and 32 stages; last tiles of 18 rows
# or of 3, whose other waves have none; whole tiles alone, and one with a part behind it
MANY = [(1554, 14352, 64), (1554, 14336, 192), (1554, 14336, 2048), (4100, 4096, 2048), (4099, 4112, 2048), (8195, 4096, 128)]
# last tiles of 64, 65, 128 rows, which workgroups make with half a wave's rows between whole ones, and of 129
MANY += [(1600, 14336, 192), (1601, 14336, 64), (1664, 14336, 128), (1665, 14336, 192)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", MANY)
def test_several_tiles_to_a_workgroup(M, N, K, height):
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    for epi in (0, 1, 4, prompt.COLUMNS):
        if epi == 1 and N % 32:
            continue
        out = torch.full((M, N // 2 if epi == 1 else N), float("nan"), dtype=torch.bfloat16, device="cuda")
        v = w.t().contiguous() if epi == prompt.COLUMNS else w
        prompt._run(x, v, out, N, epi)
        want = z if epi == prompt.COLUMNS else _want(z, epi, 0.0)
        assert float((out.double() - want).norm() / want.norm()) < BF16
        again = torch.empty_like(out)
        assert torch.equal(out, prompt._run(x, v, again, N, epi))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 40, 130])
def test_output_rows_of_many_columns(M, height):
    """A tile's 256 rows of the output are more than 2^31 bytes; K exact products in 32 bits, rounded once."""
    ops.require_native()
    N, K = (1 << 22) + 48, 64
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, device="cuda", generator=g).to(torch.bfloat16)
    out = prompt.gemm(x, w, torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"), 0)
    for n in range(0, N, 1 << 20):
        want = x.double() @ w[n:n + (1 << 20)].double().t()
        assert float((out[:, n:n + (1 << 20)].double() - want).norm() / want.norm()) < BF16


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 100, 129, 250, 300])
@pytest.mark.parametrize("N", [32, 144, 288])
def test_nothing_behind_the_output(M, N, height):
    """What lies behind the output, up to where a whole tile would end, stays as it was: rows and columns that are not there."""
    ops.require_native()
    K = 128
    g = torch.Generator().manual_seed(M + N)
    x, w = (torch.randn(n, K, generator=g).to(torch.bfloat16).cuda() for n in (M, N))
    for epi in (0, 1, 4, 8):
        cols = N // 2 if epi == 1 else N
        if epi == 1 and N % 32:
            continue
        room = torch.full((2 * prompt.TILE + M, cols), -3.0, dtype=torch.bfloat16, device="cuda")
        prompt._run(x, w.t().contiguous() if epi == 8 else w, room[:M], N, epi)
        assert bool((room[M:] == -3.0).all())
        want = _want(x.double() @ w.double().t(), 0 if epi == 8 else epi, 0.0)
        assert float((room[:M].double() - want).norm() / want.norm()) < BF16


def gates_far_below_zero(device):
    """(x [3, 64], w [32, 64], z): gates of -87 to -88.5, whose 1 + exp(88) lies above 2^126 (its reciprocal is no normal number of
    32 bits), beside up rows of 2^100, which bring the product back to 1e-6.  Every sum is one product."""
    x = torch.zeros(3, 64, dtype=torch.bfloat16, device=device)
    x[0, 0] = x[1, 1] = x[2, 2] = 1
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=device)
    w[:16, 0], w[:16, 1], w[:16, 2], w[16:, :3] = -87.0, -88.0, -88.5, 2.0 ** 100
    return x, w, x.double() @ w.double().t()


@pytest.mark.gpu
def test_gates_far_below_zero():
    """g / (1 + exp(-g)) u, rounded to bf16 once; the exponential of 88 is 1e-5 of itself off."""
    ops.require_native()
    x, w, z = gates_far_below_zero("cuda")
    want = _want(z, 1, 0.0)
    got = prompt.gemm(x, w, None, 1).double()
    assert float(want.abs().min()) > 1e-7 and float(((got - want) / want).abs().max()) < BF16 + 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (65, 272, 192), (257, 240, 64), (640, 528, 1664), (300, 4096, 11008), (2050, 2304, 4096)])
def test_products_with_columns(M, N, K, height):
    """x w, as a gradient goes back through a projection: ends of tiles and of a wave's columns, tiles in parts."""
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = torch.randn(K, N, device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    want = x.double() @ w.double()
    got = prompt.gemm_columns(x, w, always=True)
    assert float((got.double() - want).norm() / want.norm()) < BF16
    assert torch.equal(got, prompt.gemm_columns(x, w, always=True))


@pytest.mark.gpu
def test_not_a_number_and_infinity_pass():
    ops.require_native()
    x = torch.ones(260, 64, dtype=torch.bfloat16, device="cuda")
    x[3, 5], x[4, 6] = float("nan"), float("inf")
    w = torch.ones(32, 64, dtype=torch.bfloat16, device="cuda")
    for epi in (0, 1, 4):
        y = prompt.gemm(x, w, None, epi)
        assert y[3].isnan().all() and y[4].isinf().all() and y[5:].isfinite().all() and y[:3].isfinite().all()
    # a limit takes a number that is not one for itself, in the epilogue as in the pass over a product's rows
    y, z = prompt.gemm(x, w, None, 1, 1.5), torch.empty(260, 16, dtype=torch.bfloat16, device="cuda")
    ops.mixers.clamped_glu(prompt.gemm(x, w), z, 16, 1.5)
    assert torch.equal(y.isfinite(), z.isfinite()) and y[5:].isfinite().all() and y[:3].isfinite().all()


def test_table_and_rule(monkeypatch):
    """Tabled shapes by their row tiles, nothing else; never outside the kernel."""
    monkeypatch.setitem(prompt._STATE, "table", {(4096, 4096, 0): frozenset({3})})
    assert prompt.chosen(513, 4096, 4096, 0) and prompt.chosen(768, 4096, 4096, 0)
    assert not prompt.chosen(512, 4096, 4096, 0) and not prompt.chosen(769, 4096, 4096, 0)
    assert not prompt.chosen(768, 4096, 4096, 1)
    for M in (400, 1030, 1800, 4298):  # a shape that was not timed
        assert not prompt.chosen(M, 4096, 14336, 0)
    monkeypatch.setitem(prompt._STATE, "table", {(4096, 14336, 0): frozenset(range(1, 40)), (4096, 14336 + 32, 0): frozenset({2})})
    assert prompt.chosen(400, 4096, 14336, 0) and prompt.chosen(8192, 4096, 14336, 0)
    for M in (1, 256, 8193, 20000):
        assert not prompt.chosen(M, 4096, 14336, 0)
    assert not prompt.chosen(400, 4096 + 8, 14336, 0) and not prompt.chosen(400, 4096, 14336 + 32, 0)
    assert not prompt.chosen(400, 4096, 14336, 2) and not prompt.chosen(400, 4096, 14336, 3)
    x, w = torch.zeros(400, 14336, dtype=torch.bfloat16), torch.zeros(4096, 14336, dtype=torch.bfloat16)
    assert not prompt.ok(x, w, 0)  # the CPU
    assert prompt.shapes(__import__("src.models.config", fromlist=["PRESETS"]).PRESETS["llama2-7b"]) == \
        [(4096, 4096, 0), (4096, 11008, 0), (12288, 4096, 0), (22016, 4096, 1)]


def test_products_with_columns_elsewhere(monkeypatch):
    """What the kernel does not read, and shapes outside the table, keep the library's product."""
    monkeypatch.setitem(prompt._STATE, "table", {(64, 128, prompt.COLUMNS): frozenset({2})})
    monkeypatch.setattr(prompt, "_run", lambda *a: pytest.fail("not on the CPU"))
    x, w = torch.randn(300, 128), torch.randn(128, 64)
    assert prompt.chosen(300, 64, 128, prompt.COLUMNS) and not prompt.chosen(300, 128, 64, prompt.COLUMNS)
    for a, b in ((x, w), (x.bfloat16(), w.bfloat16()), (x.bfloat16(), w.t().contiguous().t().bfloat16())):
        assert torch.equal(prompt.gemm_columns(a, b), a @ b)
    with pytest.raises(RuntimeError):
        prompt.gemm_columns(x, w[:64])


def test_table_switched_off(monkeypatch):
    monkeypatch.setenv("MPAMD_KERNEL_TABLE", "0")
    monkeypatch.setitem(prompt._STATE, "table", None)
    assert prompt.table() == {} and not any(prompt.chosen(M, *s) for s in prompt._load(prompt.TABLE) for M in (400, 1800, 4298))


def test_committed_table_decides():
    """At every shape that was timed the choice is the table's."""
    for s, tiles in prompt._load(prompt.TABLE).items():
        for m in range(1, 34):
            assert prompt.chosen(256 * m, *s) == prompt.chosen(256 * m - 100, *s) == (m in tiles)


def test_sweeps_have_to_agree():
    a, b = {(64, 64, 0): [2, 3, 7], (32, 64, 1): []}, {(64, 64, 0): [3, 4, 7], (32, 64, 1): [5]}
    assert prompt.agreed([a, b]) == {(64, 64, 0): [3, 7], (32, 64, 1): []}


def test_committed_table_reads():
    t = prompt._load(prompt.TABLE)
    assert t and all(prompt.shape_ok(8192, *s) and all(2 <= m <= 32 for m in v) for s, v in t.items())


def test_few_rows(monkeypatch):
    """Up to 256 rows go by a table of their own, whose four ranges end at 32, 64, 128 and 256."""
    assert all(prompt.shape_ok(256, *s) and all(1 <= m <= 4 for m in v) for s, v in prompt._load(prompt.FEW_TABLE).items())
    for got, (lo, hi) in {1: (1, 32), 2: (33, 64), 3: (65, 128), 4: (129, 256)}.items():
        monkeypatch.setitem(prompt._STATE, "few", {(4096, 4096, 0): frozenset({got})})
        assert [M for M in range(1, 400) if prompt.few(M, 4096, 4096, 0)] == list(range(lo, hi + 1))
        assert set(prompt.FEW_ROWS[got]) <= set(range(lo, hi + 1))
    assert not prompt.few(200, 4096, 4096, 1) and not prompt.few(200, 4096, 8192, 0) and not prompt.chosen(200, 4096, 4096, 0)
    monkeypatch.setenv("MPAMD_KERNEL_TABLE", "0")
    monkeypatch.setitem(prompt._STATE, "few", None)
    assert prompt.table("few") == {}


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 33, 128, 129, 256])
@pytest.mark.parametrize("N,K,epi", [(4096, 28672, 8), (4096, 14336, 0)])
def test_products_of_few_rows(M, N, K, epi):
    """One row tile whose K is cut into as many parts as fill the CUs."""
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn(*((K, N) if epi == 8 else (N, K)), device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    want = x.double() @ (w.double() if epi == 8 else w.double().t())
    got = prompt._run(x, w, torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"), N, epi)
    assert float((got.double() - want).norm() / want.norm()) < BF16


def test_counts_that_were_timed_again():
    """Of the counts that sweeps did not agree on, the table holds those at which the record has the tile kernel no slower."""
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "prompt_products", "counts_timed_again.txt")
    if not os.path.exists(path):
        pytest.skip("no record")
    ratios = {}
    with open(path) as f:
        for line in f:
            p = line.split()
            if line.startswith("N") and len(p) == 7:
                ratios.setdefault((p[0], int(p[1])), []).append(float(p[6]))
    table = {prompt._key(s): v for s, v in prompt._load(prompt.TABLE).items()}
    assert len(ratios) == 56
    for (shape, m), r in ratios.items():
        assert (m in table[shape]) == (min(r) >= 1), (shape, m)
