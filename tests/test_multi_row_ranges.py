"""The measured ranges of two and more rows (set_multi_row_ranges in gemv_kernels.hip): which launches they take, at the ends of
the ranges, that the plans they give cover the problem, and results through the new routes."""
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, error_report

VALU, LDS, KSTAT = 0, 2, 3


def plan_of(tiles, rows, ksteps, group=128, element="f16"):
    k = ksteps * 512
    args = (16 * tiles, rows, k - k % group, 4, group)
    got = mg.query_launch(*args, element=element, num_compute_units=256)
    cov = mg.plan_coverage(*args, element=element, num_compute_units=256)
    assert cov["tiles_miscovered"] == 0 and cov["bad_waves"] == 0, args
    mg.set_default_plans(False)
    try:
        rules = mg.query_launch(*args, element=element, num_compute_units=256)
        other = mg.query_launch(*args, element=element, num_compute_units=128)
    finally:
        mg.set_default_plans(True)
    assert mg.query_launch(*args, element=element, num_compute_units=128) == other      # 256 compute units only
    return got, rules


@pytest.mark.parametrize("tiles, rows, ksteps, group, taken", [
    (256, 9, 5, 128, True), (256, 16, 14, 128, True), (64, 12, 8, 128, True), (63, 12, 8, 128, False), (256, 16, 4, 128, False),
    (200, 14, 15, 64, True), (200, 15, 15, 64, False), (200, 9, 16, 128, False), (200, 12, 10, 96, False), (200, 8, 16, 128, False),
    (512, 13, 16, 64, True), (321, 16, 10, 128, True), (320, 16, 10, 128, False), (512, 16, 8, 128, False), (511, 16, 8, 128, True),
    (400, 14, 12, 128, False), (400, 14, 17, 128, False), (513, 16, 16, 128, False)])
def test_fp16_9_to_16_rows(tiles, rows, ksteps, group, taken):
    got, rules = plan_of(tiles, rows, ksteps, group)
    if taken:
        assert rules["matrix_core"] == LDS and got["matrix_core"] == KSTAT and got["workgroups"] == min(tiles, 256), got
    else:
        assert got == rules


@pytest.mark.parametrize("tiles, rows, ksteps, want", [
    (19 * 256 + 1, 2, 3, (KSTAT, 1024)), (19 * 256, 2, 3, None), (11 * 256 + 1, 2, 4, (KSTAT, 512)), (11 * 256, 2, 4, None),
    (26 * 256 + 1, 2, 8, (KSTAT, 512)), (26 * 256, 2, 8, None), (8016, 2, 8, (KSTAT, 512)), (8016, 3, 8, (KSTAT, 768)),
    (8016, 4, 8, (KSTAT, 1024)), (30 * 256, 4, 8, None), (41 * 256, 4, 8, None), (8016, 4, 7, None), (8016, 5, 8, None),
    (1854, 2, 9, (LDS, None)), (2275, 2, 9, None), (1536, 2, 5, None), (1792, 2, 16, None), (4096, 2, 17, None)])
def test_bf16_two_to_four_rows(tiles, rows, ksteps, want):
    got, rules = plan_of(tiles, rows, ksteps, element="bf16")
    if want is None:
        assert got == rules
    else:
        assert got != rules and got["matrix_core"] == want[0] and got["workgroups"] == (want[1] or got["workgroups"]), got


@pytest.mark.parametrize("tiles, ksteps, want", [(2049, 5, 5), (2500, 8, 8), (3500, 14, 7), (2048, 8, None), (3500, 15, None),
                                                 (3500, 4, None)])
def test_two_fp16_rows_int8(tiles, ksteps, want):
    args = (16 * tiles, 2, 256 * ksteps, 8, 128)
    got = mg.query_launch(*args, num_compute_units=256)
    cov = mg.plan_coverage(*args, num_compute_units=256)
    assert cov["tiles_miscovered"] == 0 and cov["bad_waves"] == 0
    mg.set_default_plans(False)
    try:
        rules = mg.query_launch(*args, num_compute_units=256)
    finally:
        mg.set_default_plans(True)
    if want is None:
        assert got == rules
    else:
        assert (got["matrix_core"], got["split_k"], got["tiles_per_wg"], got["tiles_in_sequence"]) == (VALU, want, 1, 1), got


@pytest.mark.gpu
def test_two_fp16_rows_int8_results(gpu):
    prob = Problem("ranges", 32788, 2568, 8, PER_COLUMN, 0, m_batch=2, bias=True, x_dist="normal")   # 2050 tiles, 11 k steps: 2 x 5 + 1
    assert mg.query_launch(32788, 2, 2568, 8, 2568, num_compute_units=256)["split_k"] == 6
    _, rel, _ = error_report(DeviceProblem(prob, gpu).run(), prob.oracle_gemv(threads=16))
    assert rel <= 2e-3, rel


@pytest.mark.gpu
@pytest.mark.parametrize("n_out, rows, k, qop, group, bias, element, kind", [
    (1028, 9, 2576, PER_COLUMN, 0, True, "f16", KSTAT),                 # 65 tiles, the last of four rows; the last k step of 16 elements
    (4092, 15, 6720, SCALE_AND_ZEROS, 64, False, "f16", KSTAT),         # 256 tiles, 14 k steps
    (5140, 13, 2560, SCALE_AND_ZEROS, 128, True, "f16", KSTAT),         # 322 tiles, walks of two, five waves
    (8180, 16, 7744, SCALE_ONLY, 64, True, "f16", KSTAT),               # 512 tiles, 16 waves
    (77844, 2, 1056, SCALE_AND_ZEROS, 96, True, "bf16", KSTAT),         # 4866 tiles, three k steps, four workgroups per compute unit
    (45072, 2, 2048, SCALE_AND_ZEROS, 128, False, "bf16", KSTAT),       # 2817 tiles, four
    (29652, 2, 4480, PER_COLUMN, 0, True, "bf16", LDS),                 # 1854 tiles, nine
    (122900, 4, 3592, PER_COLUMN, 0, True, "bf16", KSTAT)])             # 7682 tiles, eight, walks of 8 in 1024 workgroups
def test_results(gpu, n_out, rows, k, qop, group, bias, element, kind):
    plan = mg.query_launch(n_out, rows, k, 4, k if qop == PER_COLUMN else group, element=element, num_compute_units=256)
    assert plan["matrix_core"] == kind, plan
    prob = Problem("ranges", n_out, k, 4, qop, group, m_batch=rows, bias=bias, x_dist="normal", element=element)
    _, rel, _ = error_report(DeviceProblem(prob, gpu).run(), prob.oracle_gemv(threads=16))
    assert rel <= (2e-3 if element == "f16" else 8e-3), rel   # the bounds of the other tests: twice the half-ulp of the output type
