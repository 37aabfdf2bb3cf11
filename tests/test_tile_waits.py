"""Wait states and divisions in the 256 x 256 product tiles (csrc/wide_tile.h), whose MFMAs and column loads stand in inline asm: the
compiler counts none for them, so the assembly that it makes of the kernels is read here."""
import concurrent.futures as cf
import os
import re
import subprocess

import pytest

from src.ops import build

KERNELS = {"gemm_prompt.hip": "gemm_prompt_kernel", "moe.hip": "moe_gemm_wide_kernel"}
FREE = ("s_waitcnt", "s_barrier", "s_branch", "s_cbranch")  # (may cost nothing: no wait states counted)
REG = re.compile(r"\b([vas])(?:(\d+)|\[(\d+):(\d+)\])|\b(m0)\b")


def _regs(text):
    out = set()
    for kind, one, lo, hi, m0 in REG.findall(text):
        out |= {"m0"} if m0 else {kind + str(i) for i in range(int(one or lo), int(one or hi) + 1)}
    return out


class Op:
    def __init__(self, text, block):
        self.text, self.block = text, block  # block: the inline asm it stands in, 0: the compiler's own
        self.name, _, rest = text.partition(" ")
        ops = re.split(r",(?![^\[]*\])", rest)
        writes = 2 if "swap" in self.name else 1
        self.writes = _regs(",".join(ops[:writes])) if self.name[:2] in ("v_", "s_") and not self.name.startswith(FREE) else set()
        self.reads = _regs(",".join(ops[1:] if self.name[:2] in ("v_", "s_", "ds") else ops))
        self.mfma = self.name.startswith("v_mfma")
        self.valu = self.name.startswith("v_") and not self.mfma
        self.waits = 0 if self.name.startswith(FREE) else int(rest, 0) + 1 if self.name == "s_nop" else 1


def _functions(text, wanted):
    """(instructions, predecessors of each) of the wanted kernels."""
    for body in re.findall(r"^(_Z\w*%s\w*):.*?\n(.*?)^\.Lfunc_end" % wanted, text, re.S | re.M):
        ops, labels, block, inside, jumps = [], {}, 0, False, []
        for line in body[1].split("\n"):
            t = line.strip()
            if "#ASMSTART" in t:
                block, inside = block + 1, True
            elif "#ASMEND" in t:
                inside = False
            t = t.split(";")[0].split("//")[0].strip()
            if re.match(r"\.?\w+:", t):
                labels[t.split(":")[0]] = len(ops)
            elif t and not t.startswith("."):
                ops.append(Op(re.sub(r"\s+", " ", t), block if inside else 0))
        before = [[i - 1] if i and ops[i - 1].name not in ("s_branch", "s_endpgm") else [] for i in range(len(ops))]
        for i, o in enumerate(ops):
            m = re.match(r"s_c?branch\S* (\S+)", o.text)
            if m:
                before[labels[m.group(1)]].append(i)
        yield body[0], ops, before


def _since(ops, before, at, hit, far):
    """Fewest wait states of inline asm between an instruction for which ``hit`` holds and instruction ``at`` on any way there
    (``far``: as many or more).  What the compiler has placed there counts for none: it may place it elsewhere."""
    best, todo, seen = far, [(p, 0) for p in before[at]], {}
    while todo:
        i, n = todo.pop()
        if n >= best or seen.get(i, far) <= n:
            continue
        seen[i] = n
        if hit(ops[i]):
            best = n
        else:
            todo += [(p, n + (ops[i].waits if ops[i].block else 0)) for p in before[i]]
    return best


@pytest.fixture(scope="module")
def texts(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    at = tmp_path_factory.mktemp("asm")

    def make(src):
        out = str(at / (src + ".s"))
        subprocess.run([build.HIPCC, "-O3", "-fPIC", "-std=c++17", f"--offload-arch={build.ARCH}", "-I" + build.CSRC,
                        *build.DEVICE_FLAGS, "-S", "--cuda-device-only", os.path.join(build.CSRC, src), "-o", out],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        with open(out) as f:
            return f.read()
    with cf.ThreadPoolExecutor(2) as ex:
        return dict(zip(KERNELS, ex.map(make, KERNELS)))


@pytest.fixture(scope="module")
def assembly(texts):
    return [k for src, text in texts.items() for k in _functions(text, KERNELS[src])]


def test_operands_of_products_are_old_enough(assembly):
    """A vector instruction's result is read by an MFMA two wait states later or more, at a tile's first products above all."""
    assert len(assembly) == 7
    for name, ops, before in assembly:
        products = [i for i, o in enumerate(ops) if o.mfma]
        assert len(products) == 192, name  # 128 of a stage of a whole tile, 64 of a half one
        for i in products:
            used = ops[i].reads | ops[i].writes
            n = _since(ops, before, i, lambda o: o.valu and o.writes & used, 2)
            assert n >= 2, (name, ops[i].text)


def test_sums_are_made_before_they_are_read(assembly):
    """A sum is read or cleared by other instructions 16 wait states after its last product or more (a product of four passes
    needs fewer)."""
    for name, ops, before in assembly:
        for i, o in enumerate(ops):
            sums = {r for r in o.reads | o.writes if r[0] == "a"} if not o.mfma else None
            if sums:
                assert _since(ops, before, i, lambda p: p.mfma and p.writes & sums, 16) >= 16, (name, o.text)


def test_column_loads_know_their_place(assembly):
    """A load into LDS in asm takes m0 (where it goes) as an operand that the compiler sets, and waits five states in its own
    statement: the compiler may bring its other scalars back from lanes just ahead of it."""
    loads = 0
    for name, ops, before in assembly:
        assert not any("m0" in o.writes for o in ops if o.block), name
        for i, o in enumerate(ops):
            if o.block and o.name.startswith("buffer_load"):
                loads += 1
                first = next(k for k in range(i, -1, -1) if k == 0 or ops[k - 1].block != o.block)
                assert sum(p.waits for p in ops[first:i]) >= 5, name
                put = next(k for k in range(first - 1, -1, -1) if "m0" in ops[k].writes)
                assert not any(p.name.startswith("buffer_load") for p in ops[put:first]), name  # (set for this one)
    assert loads == 48  # two operands of a stage, of whole and of half tiles; of a loop's turn ahead of the first


def test_stores_end_with_the_buffer(assembly):
    """An output's stores have no scalar offset: those of rows that are not there go to a buffer of 0 bytes, whose end less such
    an offset is no number of bytes."""
    stores = 0
    for name, ops, _ in assembly:
        for o in ops:
            if o.name.startswith("buffer_store"):
                stores += 1
                assert re.search(r"s\[\d+:\d+\], 0 offen", o.text), (name, o.text)
    assert stores


def test_gates_are_divided(texts):
    """The gates' 1 / (1 + exp(-g)) is a division, correct to half a unit in 24 bits, and not the reciprocal instruction that a
    division begins with, which is a whole one off, and 0 where its result is below the normal numbers."""
    divided = 0
    for src, text in texts.items():
        for name, body in re.findall(r"^(_Z\w*gemm\w*):.*?\n(.*?)^\.Lfunc_end", text, re.S | re.M):
            n = len(re.findall(r"\bv_div_fixup_f32", body))
            assert len(re.findall(r"\bv_rcp_f32", body)) == n, name
            divided += n > 0
    assert divided == 2 + 7  # prompt products and their close; expert products of all forms
