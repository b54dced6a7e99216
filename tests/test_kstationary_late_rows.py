"""Activation rows 8-15 on the way into the operand of the k-stationary kernel where they are not requested with the first
eight (four groups per lane run, int8): in turns of four (int4) or eight rows, at the edges of a turn; and that the registers
this takes are there."""
import os
import re

import numpy as np
import pytest

import mixed_gemv_amd as mg
from mixed_gemv_amd import build as lib_build
from helpers import SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, error_report


def test_product_kernels_spill_hardly_any_registers():
    """Of the product's kernels one spills vector registers: the k-stationary one with four groups per run and zeros, 16."""
    files = [os.path.join(lib_build.OBJ_DIR, f) for f in (os.listdir(lib_build.OBJ_DIR) if os.path.isdir(lib_build.OBJ_DIR) else [])
             if f.endswith("-hip-amdgcn-amd-amdhsa-gfx950.s") and not f.startswith("probes")]
    if not files:
        pytest.skip("no device assembly: built elsewhere")
    seen, spilled = 0, {}
    for f in files:
        for name, count in re.findall(r"^ +\.symbol: +(\S+)\.kd\n(?:.*\n)*?^ +\.vgpr_spill_count: +(\d+)$", open(f).read(), re.M):
            seen += 1
            if int(count):
                spilled[name] = int(count)
    assert seen > 200
    assert [n for n in spilled if "gemv_mfma_kstat_kernelILi4ELi3ELi4ELi0ELi0E" not in n] == [], spilled
    assert all(count <= 20 for count in spilled.values()), spilled


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [8, 9, 11, 12, 13, 15, 16])
@pytest.mark.parametrize("n_out, k, bits, qop, group", [(1036, 2496, 4, SCALE_AND_ZEROS, 96),    # 5 k steps, the last one ragged
                                                        (520, 8064, 4, SCALE_ONLY, 192),         # 16 k steps
                                                        (1036, 1344, 8, SCALE_AND_ZEROS, 96)])   # int8, 6 k steps
def test_late_rows(gpu, n_out, k, bits, qop, group, rows):
    prob = Problem("late_rows", n_out, k, bits, qop, group, m_batch=rows, bias=True, x_dist="normal")
    dev = DeviceProblem(prob, gpu)
    try:
        mg.set_matrix_core_threshold(1)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_K_STATIONARY)
        mg.set_launch_override(0, 0, 0, 24)                                  # walks of 2 and 3 tiles
        assert mg.query_launch(n_out, rows, k, bits, group)["matrix_core"] == 3
        got = dev.run().copy()
        mg.set_launch_override(0, 0, 0, 0)
        assert np.array_equal(dev.run().view(np.uint16), got.view(np.uint16))
    finally:
        mg.set_launch_override(0, 0, 0, 0)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_AUTO)
        mg.set_matrix_core_threshold(0)
    _, rel, _ = error_report(got, prob.oracle_gemv(threads=8))
    assert rel <= 2e-3, rel   # the bound of the kernel's other tests: twice the half-ulp of the output type
