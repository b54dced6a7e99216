"""bf16 launches of the VALU kernel on so many tiles that the wave budget stops at two waves per tile: four instead (three with
5 and 6 k steps), at the ends of the range, and results."""
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, error_report


def waves(tiles, ksteps, bits, rows=1, group=128):
    k = ksteps * (512 if bits == 4 else 256)
    k -= k % group
    args = (16 * tiles, rows, k, bits, group)
    plan = mg.query_launch(*args, element="bf16", num_compute_units=256)
    cov = mg.plan_coverage(*args, element="bf16", num_compute_units=256)
    assert cov["tiles_miscovered"] == 0 and cov["bad_waves"] == 0, args
    return plan["split_k"] if plan["matrix_core"] == 0 else None


@pytest.mark.parametrize("tiles, ksteps, bits, rows, group, want", [
    (2049, 17, 4, 1, 128, 4), (2400, 11, 4, 1, 96, 4), (2376, 17, 8, 1, 128, 4), (2392, 17, 4, 2, 64, 4), (4096, 20, 4, 1, 128, 4),
    (3000, 9, 4, 1, 96, 3), (8000, 5, 4, 1, 96, 3), (2909, 6, 8, 1, 128, 3), (3000, 8, 8, 2, 128, 4), (1500, 5, 8, 4, 128, 3),
    (4500, 10, 8, 1, 128, 4), (4500, 10, 8, 1, 96, 2), (4500, 10, 8, 2, 128, 2), (4500, 11, 8, 2, 128, 4),   # int8 with 9 and 10 k steps
    (4100, 17, 4, 1, 128, 1), (2048, 17, 4, 1, 128, 4)])                                                     # other budgets
def test_plans(tiles, ksteps, bits, rows, group, want):
    assert waves(tiles, ksteps, bits, rows, group) == want


@pytest.mark.gpu
@pytest.mark.parametrize("n_out, k, bits, qop, group, rows, bias", [
    (32788, 4896, 4, SCALE_AND_ZEROS, 96, 1, True),      # 2050 tiles, 10 k steps, the last a fragment
    (46548, 1456, 8, PER_COLUMN, 0, 2, False),           # 2910 tiles, int8, 6 k steps: three waves
    (33000, 8320, 4, SCALE_ONLY, 64, 2, True)])          # 17 k steps
def test_results(gpu, n_out, k, bits, qop, group, rows, bias):
    prob = Problem("bf16_budget", n_out, k, bits, qop, group, m_batch=rows, bias=bias, x_dist="normal", element="bf16")
    plan = mg.query_launch(n_out, rows, k, bits, prob.group_size, element="bf16")
    assert plan["matrix_core"] == 0 and plan["split_k"] in (3, 4) and plan["tiles_in_sequence"] == 1, plan
    _, rel, _ = error_report(DeviceProblem(prob, gpu).run(), prob.oracle_gemv(threads=16))
    assert rel <= 8e-3, rel                              # twice the half-ulp of the output type
