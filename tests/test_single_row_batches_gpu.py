"""Batched and routed single rows whose problems take one part of each tile on the VALU kernel for parts: waves of one or two units up to
16 k steps, a wave for every fourth k step beyond, with four lookups per run, whatever the last k step or wave is short of, up to the
most k steps -- and always the bits of single launches."""
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY
from test_single_row_parts_gpu import batched_and_routed, plan_of

CASES = [
    # n_out, k, bits, quant_op, group, bias, element, parts, waves of the single launch
    (1020, 4320, 4, SCALE_AND_ZEROS, 96, True, "bf16", 4, 3),      # 9 k steps: waves of two units, the last of one
    (2048, 4896, 4, SCALE_ONLY, 96, False, "bf16", 2, 5),          # 10
    (1500, 7400, 4, PER_COLUMN, 0, True, "bf16", 2, 8),            # 15, the last one short
    (1000, 9312, 4, SCALE_AND_ZEROS, 96, True, "f16", 4, 5),       # 19, the last one short: waves of five and four units
    (2000, 9000, 4, PER_COLUMN, 0, True, "f16", 2, 3),             # 18
    (1024, 16640, 4, SCALE_ONLY, 64, False, "bf16", 4, 3),         # 33
    (1300, 4608, 8, SCALE_AND_ZEROS, 96, False, "f16", 2, 3),      # 18
    (1024, 32768, 8, SCALE_AND_ZEROS, 128, True, "f16", 4, 4),     # 128 k steps, the most
    (1004, 32640, 8, SCALE_AND_ZEROS, 96, False, "bf16", 4, 4),    # 128, the last one short
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_bits_of_single_launches(gpu, case):
    plan = plan_of(case)
    assert plan["split_k"] == case[8] and plan["workgroups"] == -(-(-(-case[0] // 16) * case[7]) // 8) * 8, plan
    batched_and_routed(gpu, case)
