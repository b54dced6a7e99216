"""The builds of the VALU kernel for waves of one and of two units, at every row count, type and way of looking scales up, against
the loop (which the single-stage setting selects): the same bits."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem


@pytest.mark.gpu
@pytest.mark.parametrize("element", ["f16", "bf16"])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("bits, qop, group", [(4, SCALE_AND_ZEROS, 128), (4, SCALE_ONLY, 64), (4, SCALE_AND_ZEROS, 96), (4, PER_COLUMN, 0),
                                              (8, SCALE_AND_ZEROS, 128), (8, SCALE_ONLY, 96), (8, PER_COLUMN, 0)])
@pytest.mark.parametrize("split, steps, form", [(5, 1, mg.UNIT_FORM_ONE), (3, 2, mg.UNIT_FORM_TWO)])    # 1 + 1 + 1 + 1 + 1, 2 + 2 + 1
def test_bits_of_the_loop(gpu, split, steps, form, bits, qop, group, rows, element):
    step = 512 if bits == 4 else 256
    unit = 8 if qop == PER_COLUMN else group
    k = (5 * step - step // 2) // unit * unit                   # five k steps, the last a fragment
    prob = Problem("unit_builds", 16 * 20 + 4, k, bits, qop, group, m_batch=rows, bias=True, element=element)
    dev = DeviceProblem(prob, gpu)
    args = (prob.n_out, rows, k, bits, prob.group_size)
    try:
        mg.set_matrix_core_threshold(17)
        mg.set_launch_override(split, 1, 0, 0)
        plan = mg.query_launch(*args, element=element)
        assert plan["matrix_core"] == 0 and plan["steps_per_wave"] == steps, plan
        assert mg.probe_unit_form(*args, element=element) == form
        got = dev.run().copy()
        mg.set_prefetch_stages(1)
        assert mg.probe_unit_form(*args, element=element) == mg.UNIT_FORM_LOOP
        loop = dev.run().copy()
    finally:
        mg.set_prefetch_stages(0)
        mg.set_launch_override(0, 0, 0, 0)
        mg.set_matrix_core_threshold(0)
    assert np.array_equal(got.view(np.uint16), loop.view(np.uint16))
