"""The bf16 build of the k-stationary kernel (activation rows kept in LDS, one wave per k step, walks of tiles) against
the CPU oracle: the fewest and most k steps the rule takes, one and two rounds of rows, both weight widths, every quant
mode, four groups per lane run, ragged rows and reductions, LDS filled to within 5 KiB of its limit.

Bars as for every bf16 launch: the oracle's value or a neighbour of it, at most 1 % of the outputs differing (see
test_gemv_bf16_gpu.py)."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, bf16_ulp_report

MAX_ULP = 1.0 + 1e-6
MAX_DIFFERING = 0.01

CASES = [
    # tag, n_out, k, bits, quant_op, group, rows, bias, forced workgroups (0 = the built-in rule), k steps
    ("fewest_k_steps", 2048, 2304, 4, SCALE_AND_ZEROS, 128, 3, True, 0, 5),
    ("two_rows", 4100, 4096, 4, SCALE_AND_ZEROS, 64, 2, True, 0, 8),
    ("two_rows_16_k_steps", 2052, 8192, 4, SCALE_AND_ZEROS, 128, 2, True, 0, 16),
    ("two_rows_walk_of_4", 15312, 6104, 4, PER_COLUMN, 0, 2, False, 0, 12),
    ("two_rows_9_k_steps_generic_groups", 15316, 4512, 4, SCALE_AND_ZEROS, 96, 2, True, 0, 9),
    ("eight_rows_lds_nearly_full", 12288, 8192, 4, SCALE_AND_ZEROS, 128, 8, False, 0, 16),
    ("nine_rows_two_rounds", 8192, 2560, 4, SCALE_ONLY, 128, 9, True, 0, 5),
    ("sixteen_rows", 4096, 4096, 4, SCALE_AND_ZEROS, 128, 16, False, 0, 8),
    ("generic_groups_ragged", 5004, 5280, 4, SCALE_AND_ZEROS, 96, 3, True, 0, 11),
    ("generic_groups_16_k_steps", 2052, 8064, 4, SCALE_AND_ZEROS, 192, 7, False, 0, 16),
    ("per_column_k_not_a_multiple_of_8_words", 2056, 2504, 4, PER_COLUMN, 0, 5, True, 0, 5),
    ("int8_per_column", 4096, 4096, 8, PER_COLUMN, 0, 4, True, 0, 16),
    ("int8_groups_of_96_two_rows", 2080, 2304, 8, SCALE_AND_ZEROS, 96, 2, False, 0, 9),
    ("int8_sixteen_rows", 2048, 1280, 8, SCALE_ONLY, 64, 16, True, 0, 5),
    ("long_walk", 4096, 4096, 4, SCALE_AND_ZEROS, 128, 4, True, 16, 8),
    ("walk_longer_than_the_waves", 1040, 512, 4, SCALE_AND_ZEROS, 128, 3, False, 8, 1),
    ("one_row", 1000, 8192, 4, SCALE_AND_ZEROS, 128, 1, True, 8, 16),
]


class launch:
    """The k-stationary kernel by name with capped workgroups, or the built-in rule (cap 0)."""

    def __init__(self, cap):
        self.cap = cap

    def __enter__(self):
        if self.cap:
            mg.set_matrix_core_threshold(1)
            mg.set_matrix_core_variant(mg.MATRIX_CORE_K_STATIONARY)
            mg.set_launch_override(0, 0, 0, self.cap)

    def __exit__(self, *exc):
        mg.set_launch_override(0, 0, 0, 0)
        mg.set_matrix_core_variant(mg.MATRIX_CORE_AUTO)
        mg.set_matrix_core_threshold(0)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_plan_covers_the_problem(case):
    tag, n_out, k, bits, qop, group, rows, bias, cap, ksteps = case
    with launch(cap):
        plan = mg.query_launch(n_out, rows, k, bits, k if qop == PER_COLUMN else group, element="bf16")
        cover = mg.plan_coverage(n_out, rows, k, bits, k if qop == PER_COLUMN else group, element="bf16")
    assert plan["split_k"] == ksteps and plan["steps_per_wave"] == 1 and plan["tiles_per_wg"] == 1, plan
    assert plan["matrix_core"] == 3 and plan["tiles_in_sequence"] == -(-(-(-n_out // 16)) // (cap or 256)), plan
    assert cover["lds_bytes"] == ksteps * rows * ((1024 if bits == 4 else 512) + 16) + plan["tiles_in_sequence"] * 4 * rows * 17 * 16
    assert cover["lds_bytes"] <= 160 * 1024 and cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0, cover


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["auto", "general"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_parity_with_the_oracle(gpu, case, form):
    tag, n_out, k, bits, qop, group, rows, bias, cap, _ = case
    prob = Problem("ksb_" + tag, n_out, k, bits, qop, group, m_batch=rows, bias=bias, element="bf16")
    dev = DeviceProblem(prob, gpu)
    try:
        mg.set_dequant_form(mg.DEQUANT_EXACT_INTEGER if form == "general" else mg.DEQUANT_AUTO)
        with launch(cap):
            y = dev.run()
    finally:
        mg.set_dequant_form(mg.DEQUANT_AUTO)
    ulp, differing = bf16_ulp_report(y, prob.oracle_gemv(threads=16))
    assert ulp <= MAX_ULP and differing <= MAX_DIFFERING, (ulp, differing)


@pytest.mark.gpu
def test_batched_launch_matches_single_launches(gpu):
    """Three problems in one launch, strides in every operand: the bits of three launches."""
    import torch
    n_out, k, rows, count = 2048, 4096, 5, 3
    gen = torch.Generator(device=gpu).manual_seed(7)
    w_bytes = n_out * k // 2
    w = torch.randint(0, 256, (count, w_bytes), dtype=torch.uint8, device=gpu, generator=gen)
    s = (torch.rand((count, k // 128, n_out), device=gpu, generator=gen) * 0.019 + 0.001).to(torch.bfloat16)
    z = (torch.rand((count, k // 128, n_out), device=gpu, generator=gen) * 0.1 - 0.05).to(torch.bfloat16)
    x = torch.randn((count, rows, k), device=gpu, generator=gen).to(torch.bfloat16)
    bias = torch.randn((count, n_out), device=gpu, generator=gen).to(torch.bfloat16)
    y = torch.zeros((count, rows, n_out), dtype=torch.bfloat16, device=gpu)
    single = torch.zeros_like(y)
    assert mg.query_launch(n_out, rows, k, 4, 128, element="bf16")["matrix_core"] == 3
    mg.device_gemv(w, x, s, z, bias, y, count, n_out, rows, k, 128, SCALE_AND_ZEROS, 4,
                   batch_strides=(w_bytes, rows * k, k // 128 * n_out, n_out, rows * n_out))
    for b in range(count):
        mg.device_gemv(w[b], x[b], s[b], z[b], bias[b], single[b], 1, n_out, rows, k, 128, SCALE_AND_ZEROS, 4)
    torch.cuda.synchronize()
    assert np.array_equal(y.view(torch.int16).cpu().numpy(), single.view(torch.int16).cpu().numpy())
