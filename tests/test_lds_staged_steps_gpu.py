"""The LDS-staged matrix-core kernel's walk along k, which goes in pairs of steps with a single one behind them: every small
number of steps per wave, odd and even, last waves with one, two or more steps fewer than the others, stages shared by
several tiles and not, a workgroup with fewer tiles than the others, both element types and weight widths, 8 and 16 staged
rows.  Bars as everywhere: 2e-3 of the result (fp16: fp32 sums in another order, one rounding), the oracle's bf16 or its
neighbour."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, bf16_ulp_report, error_report

# k steps, k-split waves asked for, tiles per workgroup -> steps per wave, steps of the last wave
WALKS = [(1, 1, 1, 1, 1), (2, 1, 2, 2, 2), (3, 1, 1, 3, 3), (4, 1, 2, 4, 4), (5, 1, 4, 5, 5), (5, 2, 2, 3, 2), (7, 2, 1, 4, 3),
         (10, 4, 1, 3, 1), (13, 4, 2, 4, 1), (17, 4, 1, 5, 2), (9, 4, 1, 3, 3), (6, 4, 2, 2, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [5, 12])
@pytest.mark.parametrize("bits,qop,group", [(4, SCALE_AND_ZEROS, 128), (4, SCALE_ONLY, 96), (8, SCALE_ONLY, 64), (8, PER_COLUMN, 0)])
@pytest.mark.parametrize("element", ["f16", "bf16"])
def test_every_number_of_steps(gpu, element, bits, qop, group, rows):
    step = 512 if bits == 4 else 256
    mg.set_matrix_core_threshold(1)
    mg.set_matrix_core_variant(mg.MATRIX_CORE_LDS_STAGED)
    try:
        for ksteps, split, tiles, steps, last in WALKS:
            k = ksteps * step if qop == PER_COLUMN else (ksteps * step) // group * group
            mg.set_launch_override(split, tiles, 0, 0)
            prob = Problem(f"steps{ksteps}_{split}_{tiles}", 84, k, bits, qop, group, m_batch=rows, bias=True, element=element)
            plan = mg.query_launch(84, rows, k, bits, prob.group_size, element=element)
            assert plan["matrix_core"] == 2 and plan["steps_per_wave"] == steps, plan
            assert ksteps - (plan["split_k"] - 1) * steps == last, plan
            y = DeviceProblem(prob, gpu).run()
            ref = prob.oracle_gemv(threads=8)
            if element == "bf16":
                ulp, differing = bf16_ulp_report(y, ref)
                assert ulp <= 1.0 + 1e-6 and differing <= 0.02, (ksteps, split, tiles, ulp, differing)
            else:
                assert error_report(y, ref)[1] <= 2e-3 and np.isfinite(y.astype(np.float32)).all(), (ksteps, split, tiles)
    finally:
        mg.set_launch_override(0, 0, 0, 0)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_AUTO)
        mg.set_matrix_core_threshold(0)
