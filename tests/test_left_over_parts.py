"""k-stationary launches whose left-over tiles are split into parts: which launches do (the plan's coverage replays the kernel's index
functions), and that the outputs have the bits of the same kernel on whole tiles -- one to three tiles a walk, one left-over tile and
the most that two and four parts reach, rows past the matrix, k steps that leave the last unit of a part short, every quant mode, batched
and routed launches, infinite scales in the last group."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, float64_bound_violations

CASES = [
    # tiles, k steps, k short of whole steps by, quant_op, group, rows, bias, element, tiles' parts
    (313, 11, 352, SCALE_ONLY, 96, 3, True, "bf16", 4),
    (257, 9, 0, SCALE_AND_ZEROS, 128, 4, False, "bf16", 4),
    (320, 6, 256, SCALE_AND_ZEROS, 64, 2, True, "bf16", 4),
    (576, 5, 8, PER_COLUMN, 0, 3, False, "bf16", 4),
    (384, 9, 128, SCALE_AND_ZEROS, 128, 8, True, "bf16", 2),
    (640, 13, 384, SCALE_ONLY, 128, 5, False, "bf16", 2),
    (800, 8, 0, SCALE_AND_ZEROS, 256, 3, True, "bf16", 4),
    (288, 16, 0, SCALE_AND_ZEROS, 128, 4, True, "f16", 4),
    (320, 15, 256, SCALE_ONLY, 64, 3, False, "f16", 4),
    (576, 10, 64, PER_COLUMN, 0, 3, True, "f16", 4),
    (600, 9, 128, SCALE_AND_ZEROS, 128, 8, False, "f16", 2),
    (896, 9, 256, SCALE_AND_ZEROS, 256, 8, True, "f16", 2),
]
# one unit of the busiest SIMD saved or none, too many left over, longer walks, int8
WHOLE = [(313, 7, 3, "bf16", 4), (384, 12, 4, "bf16", 4), (385, 9, 4, "bf16", 4), (1100, 9, 4, "bf16", 4), (313, 11, 3, "bf16", 8),
         (313, 8, 4, "f16", 4), (384, 16, 4, "f16", 4), (313, 16, 9, "f16", 4), (256, 9, 4, "bf16", 4)]


def shape(case):
    tiles, ksteps, short, qop, group, rows, bias, element, parts = case
    return 16 * tiles - 4, 512 * ksteps - short


def covered_in_parts(n_out, rows, k, bits, group, element):
    """The walks of whole tiles are then one shorter (a part is not counted as a unit of one)."""
    args = (n_out, rows, k, bits, group)
    plan = mg.query_launch(*args, element=element, num_compute_units=256)
    cover = mg.plan_coverage(*args, element=element, num_compute_units=256)
    assert plan["matrix_core"] == 3 and cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0, (plan, cover)
    assert cover["lds_bytes"] <= 160 * 1024 - 320
    tiles = -(-n_out // 16)
    return cover["max_units_per_wave"] < -(-tiles // 256) and tiles > 256


@pytest.mark.parametrize("case", CASES, ids=str)
def test_left_over_tiles_are_split(case):
    n_out, k = shape(case)
    assert covered_in_parts(n_out, case[5], k, 4, case[4] or k, case[7])
    mg.set_default_plans(False)
    try:
        assert not covered_in_parts(n_out, case[5], k, 4, case[4] or k, case[7])
    finally:
        mg.set_default_plans(True)


@pytest.mark.parametrize("tiles, ksteps, rows, element, bits", WHOLE)
def test_whole_tiles_where_parts_do_not_pay(tiles, ksteps, rows, element, bits):
    k = (512 if bits == 4 else 256) * ksteps
    plan = mg.query_launch(16 * tiles, rows, k, bits, 128, element=element, num_compute_units=256)
    cover = mg.plan_coverage(16 * tiles, rows, k, bits, 128, element=element, num_compute_units=256)
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0
    assert plan["matrix_core"] != 3 or cover["max_units_per_wave"] == -(-tiles // plan["workgroups"]), (plan, cover)


@pytest.mark.parametrize("tiles, ksteps, rows", [(607, 5, 7), (574, 5, 4), (312, 6, 4), (518, 6, 3), (816, 6, 4)])
def test_short_fp16_reductions_walk_whole_tiles(tiles, ksteps, rows):
    for k in (512 * ksteps, 512 * ksteps - 128):
        assert not covered_in_parts(16 * tiles, rows, k, 4, 128, "f16")


def problem(case, buffer=0):
    n_out, k = shape(case)
    tiles, ksteps, short, qop, group, rows, bias, element, parts = case
    return Problem(f"left over {case}", n_out, k, 4, qop, group, m_batch=rows, bias=bias, element=element, buffer=buffer)


def on_whole_tiles(call):
    mg.set_default_plans(False)
    try:
        return call()
    finally:
        mg.set_default_plans(True)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["auto", "general", "infinite"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_bits_of_whole_tiles(gpu, case, form):
    prob = problem(case)
    if form == "infinite":
        prob.scale[-1, ::7] = 0x7F80 if prob.element == "bf16" else np.inf
    dev = DeviceProblem(prob, gpu)
    mg.set_dequant_form(mg.DEQUANT_EXACT_INTEGER if form == "general" else mg.DEQUANT_AUTO)
    try:
        got = dev.run().copy().view(np.uint16)
        want = on_whole_tiles(lambda: dev.run().copy().view(np.uint16))
    finally:
        mg.set_dequant_form(mg.DEQUANT_AUTO)
    if form == "infinite":   # any NaN will do, and past the reduction a whole tile makes one of an infinity
        inf = 0x7F80 if prob.element == "bf16" else 0x7C00
        special = (got & 0x7FFF) >= inf
        assert np.array_equal(special, (want & 0x7FFF) >= inf) and special.any() and not special.all()
        assert np.array_equal(got[~special], want[~special])
    else:
        assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[10]], ids=str)
def test_batched_and_routed_launches_have_the_bits_of_single_ones(gpu, case):
    import torch
    n_out, k = shape(case)
    tiles, ksteps, short, qop, group, rows, bias, element, parts = case
    devs = [DeviceProblem(problem(case, b), gpu) for b in range(2)]
    single = [d.run().copy().view(np.uint16) for d in devs]
    cat = lambda name: None if getattr(devs[0], name) is None else torch.stack([getattr(d, name) for d in devs])  # noqa: E731
    w, scale, zero, b = (cat(n) for n in ("w", "scale", "zero", "bias"))
    x = torch.stack([devs[0].x] * 2)
    strides = (w[0].numel(), rows * k, scale[0].numel(), n_out if b is not None else 0, rows * n_out)
    y = torch.full((2, rows, n_out), 0x7E00, dtype=torch.int16, device=gpu)
    mg.device_gemv(w, x, scale, zero, b, y, 2, n_out, rows, k, group, qop, 4, batch_strides=strides, element=element)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), np.stack(single))     # the activations are the same in every buffer
    route = torch.tensor([1, 1], dtype=torch.int32, device=gpu)
    y.fill_(0x7E00)
    mg.device_gemv_routed(w, x, scale, zero, b, y, route, 2, 2, n_out, rows, k, group, strides, qop, 4, element=element)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), np.stack([single[1]] * 2))


@pytest.mark.gpu
@pytest.mark.parametrize("qop", [SCALE_ONLY, SCALE_AND_ZEROS])
@pytest.mark.parametrize("n_out, k, rows", [(5004, 4640, 4), (9596, 4640, 8)])
def test_one_group_as_long_as_the_reduction(gpu, n_out, k, rows, qop):
    """Plans take such a group for the per-column mode, whose left-over tiles go in parts; by group the fp16 launch looks four scales
    up per run, for which no such build exists: every output is there all the same."""
    assert covered_in_parts(n_out, rows, k, 4, k, "f16")
    prob = Problem("one group", n_out, k, 4, qop, k, m_batch=rows, bias=True)
    y = DeviceProblem(prob, gpu).run()
    assert float64_bound_violations(prob, y)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[1], (288, 8, 0, SCALE_AND_ZEROS, 128, 4, True, "f16", 0), (266, 16, 128, SCALE_ONLY, 128, 4, False, "f16", 4)], ids=str)
def test_batched_launches_with_few_tiles_left_over_have_the_bits_of_single_ones(gpu, case):
    """A single launch may take them in parts, a batched one takes whole tiles."""
    test_batched_and_routed_launches_have_the_bits_of_single_ones(gpu, case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[2], CASES[8], CASES[10], (576, 6, 128, PER_COLUMN, 0, 3, True, "bf16", 4),
                                  (257, 9, 0, PER_COLUMN, 0, 4, False, "bf16", 4), (288, 16, 256, PER_COLUMN, 0, 4, False, "f16", 4)], ids=str)
def test_infinities_are_those_of_whole_tiles(gpu, case):
    """Infinite scales of the last group (of the column): an output is infinite or not a number in a part where it is in a whole tile,
    the oracle's where the last k step is whole."""
    prob = problem(case)
    prob.q[:] = np.abs(prob.q.astype(np.int16)).clip(1, 7)
    from oracle import pack_int4
    prob.w_raw = pack_int4(prob.q)
    prob.scale[-1, ::5] = 0x7F80 if prob.element == "bf16" else np.inf
    prob.x[:] = 0x3F80 if prob.element == "bf16" else 1.0
    inf = 0x7F80 if prob.element == "bf16" else 0x7C00
    special = lambda y: np.where((y.view(np.uint16) & 0x7FFF) > inf, 2, np.where((y.view(np.uint16) & 0x7FFF) == inf, 1, 0))  # noqa: E731
    dev = DeviceProblem(prob, gpu)
    got = dev.run().copy()
    whole = on_whole_tiles(lambda: dev.run().copy())
    assert (special(got)[:, ::5] > 0).all() and np.array_equal(special(whole), special(got))
    if prob.k % 512 == 0:
        assert np.array_equal(special(got), special(prob.oracle_gemv(threads=16).reshape(got.shape)))
