"""Prompt products on tiles of 128 to 224 rows (csrc/gemm_prompt_low.hip): the edges of each height, several tiles to a workgroup, tiles
cut into parts; and the wait states of their inline asm, as tests/test_tile_waits.py reads them."""
import pytest
import torch

from src import ops
from src.ops import build, prompt
from tests import test_tile_waits as waits
from tests.test_prompt_gemm import BF16, _want

# fragments of a wave's rows (a tile has 32 times as many rows), then M, N, K: last tiles of 1 to 3 rows and others, of 16 columns and
# others; one stage and many; more tiles than CUs; the tiles past a round of CUs, or all of them, cut in K
CASES = [(4, 130, 2496, 64), (4, 2049, 2080, 2048), (4, 1101, 13632, 192), (4, 96, 12448, 8192), (4, 2433, 1520, 4096),
         (5, 1122, 7856, 64), (5, 1443, 5632, 512), (5, 1577, 10096, 192), (5, 2452, 7328, 1024), (5, 1603, 1216, 2048),
         (6, 1923, 5088, 320), (6, 1922, 10720, 64), (6, 2182, 9728, 192), (6, 174, 14240, 8192), (6, 2115, 1712, 8192),
         (7, 1345, 8768, 512), (7, 2508, 14384, 192), (7, 1795, 14080, 320), (7, 217, 7840, 8192), (7, 1345, 2944, 8192)]


@pytest.mark.gpu
@pytest.mark.parametrize("frags,M,N,K", CASES)
def test_heights(frags, M, N, K):
    """One sum of K exact products in 32 bits (in parts or whole), rounded to bf16 once; rows behind the output stay."""
    ops.require_native()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).div(K ** 0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    for epi in (0, 1, 4, prompt.COLUMNS):
        if epi == 1 and N % 32:
            continue
        cols = N // 2 if epi == 1 else N
        room = torch.full((M + 32, cols), -3.0, dtype=torch.bfloat16, device="cuda")
        v = w.t().contiguous() if epi == prompt.COLUMNS else w
        prompt._run(x, v, room[:M], N, epi, frags=frags)
        want = z if epi == prompt.COLUMNS else _want(z, epi, 0.0)
        assert float((room[:M].double() - want).norm() / want.norm()) < BF16
        assert bool((room[M:] == -3.0).all())
        assert torch.equal(room[:M], prompt._run(x, v, torch.empty_like(room[:M]), N, epi, frags=frags))


@pytest.mark.skipif(not ops.native_available(), reason="no kernel library")
@pytest.mark.parametrize("M,N,K,need", [(4100, 4096, 2048, False), (300, 4096, 11008, True), (8000, 4368, 10880, False), (1891, 18704, 28672, False)])
def test_workspace_is_the_height_s(M, N, K, need):
    """What the height that runs needs, and nothing where only tiles of 256 rows would be cut."""
    room = torch.ops.mpamd.gemm_prompt_ws
    assert room(M, N, K) == room(M, N, K, torch.ops.mpamd.gemm_prompt_frags(M, N, K))
    assert (room(M, N, K) > 0) == need and room(M, N, K, 8) > 0


@pytest.mark.gpu
def test_which_height():
    """Heights that a caller asks for, the estimate's without one, no others."""
    ops.require_native()
    x, w = torch.randn(300, 64, device="cuda").to(torch.bfloat16), torch.randn(512, 64, device="cuda").to(torch.bfloat16)
    y = torch.empty(300, 512, dtype=torch.bfloat16, device="cuda")
    own = torch.ops.mpamd.gemm_prompt_frags(300, 512, 64)
    assert 4 <= own <= 8 and torch.ops.mpamd.gemm_prompt_ws(300, 512, 64) == torch.ops.mpamd.gemm_prompt_ws(300, 512, 64, own)
    for frags in (-1, 1, 3, 9):
        with pytest.raises(RuntimeError, match="fragments"):
            prompt._run(x, w, y, 512, 0, frags=frags)


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    import os
    import subprocess

    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "low.s")
    subprocess.run([build.HIPCC, "-O3", "-fPIC", "-std=c++17", f"--offload-arch={build.ARCH}", "-I" + build.CSRC, *build.DEVICE_FLAGS,
                    "-S", "--cuda-device-only", os.path.join(build.CSRC, "gemm_prompt_low.hip"), "-o", out],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(out) as f:
        return list(waits._functions(f.read(), "gemm_prompt_kernel"))


def test_wait_states(assembly):
    assert len(assembly) == 16  # four heights, four ends
    for name, instrs, before in assembly:
        frags = int(name.split("Li")[2].split("E")[0])
        assert sum(o.mfma for o in instrs) == 16 * frags, name
    waits.test_sums_are_made_before_they_are_read(assembly)
    waits.test_stores_end_with_the_buffer(assembly)
    for name, instrs, before in assembly:
        for i, o in enumerate(instrs):
            if o.mfma:
                used = o.reads | o.writes
                assert waits._since(instrs, before, i, lambda p: p.valu and p.writes & used, 2) >= 2, (name, o.text)
            if o.block and o.name.startswith("buffer_load"):  # m0 set by the compiler for this load, five states ahead of it
                first = next(k for k in range(i, -1, -1) if k == 0 or instrs[k - 1].block != o.block)
                assert sum(p.waits for p in instrs[first:i]) >= 5, name
                put = next(k for k in range(first - 1, -1, -1) if "m0" in instrs[k].writes)
                assert not any(p.name.startswith("buffer_load") for p in instrs[put:first]), name
        assert not any("m0" in o.writes for o in instrs if o.block), name
