"""The measured ranges of single rows (single_row_split in gemv_kernels.hip): which launches they take, at the ends of the
ranges, and that the plans they give cover the problem."""
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, error_report


def waves(tiles, ksteps, bits=4, group=128, element="f16"):
    """(waves per tile, tiles per workgroup, tiles one after the other), or None where the rules decide."""
    k = ksteps * (512 if bits == 4 else 256)
    k -= k % group
    args = (16 * tiles, 1, k, bits, group)
    got = mg.query_launch(*args, element=element, num_compute_units=256)
    mg.set_default_plans(False)
    try:
        rules = mg.query_launch(*args, element=element, num_compute_units=256)
    finally:
        mg.set_default_plans(True)
    cov = mg.plan_coverage(*args, element=element, num_compute_units=256)
    assert cov["tiles_miscovered"] == 0 and cov["bad_waves"] == 0, args
    if got == rules:
        return None
    assert got["matrix_core"] == 0 and got["tiles_per_wg"] == 1 and got["tiles_in_sequence"] == 1, got
    return got["split_k"]


@pytest.mark.parametrize("tiles, ksteps, want", [
    # nothing up to one tile per compute unit, nor below five k steps
    (256, 12, None), (6000, 4, None),
    # 9-16 k steps: a wave per unit up to 512 tiles, two units a wave above
    (257, 12, 12), (500, 12, 12), (512, 14, None), (498, 14, None), (497, 14, 14), (400, 10, None), (513, 12, 6), (768, 13, 7), (768, 10, 5),
    (769, 10, None), (1024, 10, None), (1100, 16, 8), (1792, 12, None), (1791, 13, 7), (640, 16, None), (641, 16, 8),
    (3072, 16, 8), (9000, 12, 6),
    # 5-8 k steps: two units where there are many tiles, but for even fits
    (2049, 5, 3), (3073, 6, 3), (2050, 6, None), (1409, 8, 4), (1408, 8, None), (1536, 8, None), (2000, 7, None), (8000, 7, 4),
    # longer reductions: two units up to 768 tiles and 32 k steps, four waves above 1024
    (513, 17, 9), (768, 32, 16), (768, 33, 4), (769, 20, None), (1024, 20, None), (1100, 33, None), (512, 20, None), (2000, 30, 4)])
def test_fp16_int4(tiles, ksteps, want):
    assert waves(tiles, ksteps) == want


@pytest.mark.parametrize("tiles, ksteps, want", [
    (2049, 8, 8), (2048, 8, None), (1025, 10, 10), (1024, 10, None), (1025, 9, None), (2049, 13, 13), (2049, 14, None)])
def test_fp16_int8(tiles, ksteps, want):
    assert waves(tiles, ksteps, bits=8) == want


def test_groups_that_do_not_divide_the_k_step():
    assert waves(400, 10, group=96) == 10                                            # fp16: ten of them too
    assert [waves(400, ks, group=96, element="bf16") for ks in (8, 9, 16, 17)] == [None, 5, 8, None]
    assert waves(400, 12, element="bf16") is None and waves(513, 12, group=96, element="bf16") is None


def test_two_lookups_per_run_where_a_wave_per_tile_fills_the_simds():
    assert [waves(tiles, 12, group=64) for tiles in (993, 994, 995, 1024)] == [6, 6, None, None]
    assert waves(1024, 12) == 6


def test_other_devices_and_overrides_keep_the_rules():
    args = (16 * 3072, 1, 8192, 4, 128)
    mine = mg.query_launch(*args, num_compute_units=256)
    assert mine["split_k"] == 8
    mg.set_default_plans(False)
    try:
        rules = {cus: mg.query_launch(*args, num_compute_units=cus) for cus in (128, 256)}
    finally:
        mg.set_default_plans(True)
    assert mg.query_launch(*args, num_compute_units=128) == rules[128]
    mg.set_prefetch_stages(2)
    try:
        assert mg.query_launch(*args, num_compute_units=256) == rules[256]
    finally:
        mg.set_prefetch_stages(0)
    mg.set_launch_override(2, 1, 0, 0)
    try:
        assert mg.query_launch(*args, num_compute_units=256)["split_k"] == 2
    finally:
        mg.set_launch_override(0, 0, 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("n_out, k, bits, qop, group, bias, element, split, steps", [
    (4100, 4608, 4, SCALE_AND_ZEROS, 128, True, "f16", 9, 1),      # 257 tiles, the last of four rows: nine one-unit waves
    (8196, 6560, 4, PER_COLUMN, 0, False, "f16", 7, 2),            # 513 tiles, 13 k steps, the last a fragment: seven waves, the last of one unit
    (32788, 2496, 4, SCALE_ONLY, 96, True, "f16", 3, 2),           # 2050 tiles, five k steps: 2 + 2 + 1
    (8212, 8704, 4, SCALE_AND_ZEROS, 64, True, "f16", 9, 2),       # 514 tiles, 17 k steps: nine waves
    (16388, 2576, 8, PER_COLUMN, 0, True, "f16", 11, 1),           # 1025 tiles, int8, 11 k steps: eleven one-unit waves
    (5204, 4128, 4, SCALE_AND_ZEROS, 96, True, "bf16", 5, 2)])     # 326 tiles, bf16, a lookup per block: five waves of two units
def test_results(gpu, n_out, k, bits, qop, group, bias, element, split, steps):
    import torch
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    if cus != 256:
        pytest.skip("the ranges are for devices of 256 compute units")
    plan = mg.query_launch(n_out, 1, k, bits, k if qop == PER_COLUMN else group, element=element, num_compute_units=cus)
    assert (plan["split_k"], plan["steps_per_wave"], plan["tiles_per_wg"], plan["tiles_in_sequence"]) == (split, steps, 1, 1), plan
    prob = Problem("single_row", n_out, k, bits, qop, group, m_batch=1, bias=bias, x_dist="normal", element=element)
    _, rel, _ = error_report(DeviceProblem(prob, gpu).run(), prob.oracle_gemv(threads=16))
    assert rel <= (2e-3 if element == "f16" else 8e-3), rel   # the bounds of the other tests: twice the half-ulp of the output type
