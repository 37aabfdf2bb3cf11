"""The committed decode-kernel table holds every choice that a start would otherwise time: the kernel of a product decides the
order of its sums, so that a race at start-up gave an fp8 batch other logits, and an eighth of its tokens, from one process to
the next."""
import json

import pytest
import torch

from src import ops
from src.ops import tune


@pytest.mark.gpu
@pytest.mark.parametrize("spec", tune.every_spec())
def test_no_preset_times_a_product(spec, monkeypatch):
    monkeypatch.setenv("MPAMD_GEMM_AUTOTUNE", "1")
    before = set(ops._TABLE["runtime"])
    ex = tune.stage(spec, False)
    del ex
    torch.cuda.empty_cache()
    assert sorted(ops._TABLE["runtime"] - before) == []


def test_the_choice_that_won_most_often():
    a, b, c = ({"arch": "x", "gemm": g, "qkv_fold": {}} for g in ({"p": "pk", "q": "rw"}, {"p": "sk"}, {"p": "sk", "q": "pk"}))
    assert tune.elect([a, b, c]) == {"gemm": {"p": "sk", "q": "rw"}, "qkv_fold": {}}


def test_table_is_set_and_saved_as_it_is(tmp_path):
    with open(ops.KERNEL_TABLE) as f:
        want = json.load(f)
    saved = ops.kernel_table(), set(ops._TABLE["runtime"])
    try:
        ops.set_kernel_table(want)
        assert ops.kernel_table() == want
        ops.save_kernel_table(str(tmp_path / "t.json"))
        assert json.loads((tmp_path / "t.json").read_text()) == want
    finally:
        ops.set_kernel_table(saved[0])
        ops._TABLE["runtime"].update(saved[1])


def test_which_partial_slabs_are_turned():
    """Where the measured turn is the faster one or makes no difference: not at 2048 rows of 16384 columns."""
    assert [ops.partials_turned(N, K) for N, K in ((4096, 16384), (8192, 32768), (2048, 16384), (4096, 8192), (4096, 14336))] == \
        [True, True, False, False, False]
