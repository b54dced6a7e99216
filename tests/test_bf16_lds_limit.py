"""The bf16 k-stationary kernel has 256 bytes of static LDS (zeros for the lanes of rows that do not exist) beside the dynamic LDS
that plans report: every plan leaves room for them, and one that fills the workgroup's 160 KiB to the last byte runs."""
import pytest

import mixed_gemv_amd as mg
from helpers import SCALE_AND_ZEROS, DeviceProblem, Problem, bf16_ulp_report

MOST_DYNAMIC = 160 * 1024 - 256


class k_stationary:
    def __init__(self, workgroups=0):
        self.workgroups = workgroups

    def __enter__(self):
        mg.set_matrix_core_threshold(1)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_K_STATIONARY)
        mg.set_launch_override(0, 0, 0, self.workgroups)

    def __exit__(self, *exc):
        mg.set_launch_override(0, 0, 0, 0)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_AUTO)
        mg.set_matrix_core_threshold(0)


def test_every_plan_leaves_room_for_the_static_part():
    most = 0
    for forced in (False, True):
        for bits, step in ((4, 512), (8, 256)):
            for ksteps in range(1, 17):
                for rows in range(1, 17):
                    for tiles in (64, 300, 770, 1500, 2816, 6103, 8016):
                        args = (16 * tiles, rows, ksteps * step, bits, 128)
                        if forced:
                            with k_stationary():
                                plan = mg.query_launch(*args, element="bf16", num_compute_units=256)
                        else:
                            plan = mg.query_launch(*args, element="bf16", num_compute_units=256)
                        if plan["matrix_core"] == 3:
                            most = max(most, plan["lds_bytes"])
    assert most == MOST_DYNAMIC


@pytest.mark.gpu
@pytest.mark.parametrize("tiles, rows, ksteps", [(12 * 8, 8, 14), (6 * 8, 16, 7)])   # walks of 12 and 6 tiles on 8 workgroups
def test_a_plan_at_the_limit(gpu, tiles, rows, ksteps):
    prob = Problem("lds_limit", 16 * tiles, 256 * ksteps, 8, SCALE_AND_ZEROS, 128, m_batch=rows, bias=True, element="bf16")
    dev = DeviceProblem(prob, gpu)
    with k_stationary(8):
        plan = mg.query_launch(16 * tiles, rows, 256 * ksteps, 8, 128, element="bf16", num_compute_units=256)
        assert plan["matrix_core"] == 3 and plan["lds_bytes"] == MOST_DYNAMIC, plan
        got = dev.run().copy()
    max_ulp, differing = bf16_ulp_report(got, prob.oracle_gemv(threads=8))
    assert max_ulp <= 1.0 + 1e-6 and differing <= 0.01, (max_ulp, differing)          # the bars of every bf16 launch
