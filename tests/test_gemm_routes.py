"""Which kernel W4Linear.forward takes past 16 rows: the ladders, a caller's own among them, and the rule on sizes."""

from __future__ import annotations

import copy
import pickle

import pytest

from tandem_amd.layers import awq, w4_plan
from tandem_amd.layers.w4_tables import GFX950_GEMM, OTHERS, RuleLadder

FIXED = ((64, ("mma", 8, 1, 1)), (1024, (4, 2, 4, 1, 2, 0)), (1 << 30, None))


def _layer(k=4096, n=6144, table=GFX950_GEMM):
    layer = awq.W4Linear(k, n, 128)
    layer.awq_layout = False
    layer.gemm_kernels = table
    return layer


def test_layers_without_a_table_take_the_fixed_ladder():
    """finalize(None): every shape takes the defaults."""
    assert awq.DEFAULT_GEMM == FIXED
    for k, n in ((4096, 6144), (256, 64)):
        layer = _layer(k, n, {})
        for m in (17, 64, 65, 1024, 1025, 1 << 18):
            assert layer.gemm_entry(m) == awq.pick_gemm(FIXED, m), m


def test_built_in_ladders_are_continued_by_the_rule():
    for ladder in GFX950_GEMM.values():
        assert isinstance(ladder, RuleLadder)
    layer, other = _layer(), _layer(2304, 4112)
    ladder = GFX950_GEMM[6144, 4096]
    assert layer.gemm_entry(17) == ladder[0][1] and layer.gemm_entry(ladder[-1][0]) == ladder[-1][1]
    for m in (ladder[-1][0] + 1, 700, 5000):
        assert layer.gemm_entry(m) == w4_plan.choose(m, 6144, 4096)
    assert not GFX950_GEMM[OTHERS]
    for m in (17, 700, 5000):
        assert other.gemm_entry(m) == w4_plan.choose(m, 4112, 2304)


@pytest.mark.parametrize("table", [{}, GFX950_GEMM])
def test_a_callers_ladder_is_continued_by_its_last_entry(table):
    cfg = (2, 1, 4, 2, 2, 4)
    layer = _layer(table={**table, (6144, 4096): ((64, cfg), (1024, None))})
    assert layer.gemm_entry(64) == cfg and layer.gemm_entry(65) is None and layer.gemm_entry(5000) is None
    assert layer.kernel_for(5000) == "dequant+matmul"
    layer.gemm_kernels = {**table, (6144, 4096): ((64, None), (128, cfg))}
    assert layer.gemm_entry(5000) == cfg and layer.kernel_for(5000) == f"gemm{cfg}"


def test_ladders_survive_a_copy_of_the_layer():
    for other in (copy.deepcopy(_layer()), pickle.loads(pickle.dumps(_layer()))):
        assert other.gemm_kernels == GFX950_GEMM
        for m in (17, 700, 5000):
            assert other.gemm_entry(m) == _layer().gemm_entry(m)
