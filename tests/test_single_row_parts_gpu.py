"""The VALU kernel for parts of tiles (one activation row, a workgroup per 4, 8 or 16 rows of a tile, four, two or one k steps at a
time): which launches take it, and its results against the CPU oracle where it can go wrong -- the last unit of a reduction shorter
than the others, whole parts past the matrix, one to eight waves and one or more units each, both orders of the sums (up to
16 k steps and beyond), both weight widths, every quant mode, four lookups per run, both dequantiser forms.

Bars: fp16 outputs within what the mathematics allows any fp32 accumulation of the dequantised weights
(helpers.float64_bound_violations), bf16 outputs the oracle's or a neighbour, at most 1 % of them differing."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, bf16_ulp_report, float64_bound_violations

CASES = [
    # n_out, k, bits, quant_op, group, bias, element, parts, waves
    (4, 4608, 4, SCALE_AND_ZEROS, 128, True, "f16", 4, 3),          # one part of one tile, 9 k steps: a last unit of one
    (1008, 8192, 4, SCALE_AND_ZEROS, 64, False, "f16", 4, 4),       # 16 k steps, as many as one order of the sums has
    (1000, 8448, 4, SCALE_AND_ZEROS, 256, True, "f16", 4, 5),       # 17: the other order; parts past n_out
    (1000, 17000, 4, PER_COLUMN, 0, True, "f16", 4, 3),             # 34, the last one short, 9 units of three waves
    (516, 31200, 4, SCALE_ONLY, 96, False, "f16", 4, 4),            # 61 k steps, four lookups per run
    (1000, 2560, 8, SCALE_AND_ZEROS, 128, True, "f16", 4, 3),
    (1024, 32768, 8, PER_COLUMN, 0, False, "f16", 4, 4),            # 128 k steps, the most
    (2000, 8704, 4, SCALE_AND_ZEROS, 128, True, "f16", 2, 3),       # 17: 9 units of two k steps
    (1300, 4608, 8, SCALE_AND_ZEROS, 96, False, "f16", 2, 3),       # 18
    (1020, 2400, 4, SCALE_AND_ZEROS, 96, True, "bf16", 4, 2),       # 5 k steps
    (24, 6144, 4, SCALE_ONLY, 128, False, "bf16", 4, 3),
    (1024, 16640, 4, SCALE_AND_ZEROS, 64, True, "bf16", 4, 3),      # 33
    (1024, 4416, 8, SCALE_AND_ZEROS, 64, True, "bf16", 4, 5),       # 18
    (1024, 8192, 4, SCALE_AND_ZEROS, 128, True, "bf16", 2, 8),      # eight waves
    (2048, 4096, 4, SCALE_AND_ZEROS, 128, False, "bf16", 2, 4),     # exactly half as many tiles as compute units
    (1500, 9000, 4, PER_COLUMN, 0, True, "bf16", 2, 3),             # 18
    (2044, 4800, 8, SCALE_ONLY, 96, False, "bf16", 2, 4),           # 19
]


def plan_of(case):
    n_out, k, bits, qop, group, bias, element, parts, waves = case
    return mg.query_launch(n_out, 1, k, bits, k if qop == PER_COLUMN else group, element=element, num_compute_units=256)


@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_launch_takes_the_kernel(case):
    plan, tiles, parts = plan_of(case), -(-case[0] // 16), case[7]
    ksteps = -(-case[1] // (512 if case[2] == 4 else 256))
    assert plan["matrix_core"] == 0 and plan["tiles_per_wg"] == 1 and plan["split_k"] == case[8], plan
    assert plan["workgroups"] == -(-tiles * parts // 8) * 8 and plan["steps_per_wave"] % parts == 0, plan
    cover = mg.plan_coverage(case[0], 1, case[1], case[2], case[4] or case[1], element=case[6], num_compute_units=256)
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0 and cover["lds_bytes_used"] <= cover["lds_bytes"], cover
    assert cover["lds_bytes"] >= 256 * max(16, -(-ksteps // parts)) and cover["lds_bytes"] % 4096 == 0   # whole turns of 16 units
    mg.set_default_plans(False)
    try:
        assert plan_of(case) != plan
    finally:
        mg.set_default_plans(True)


def test_where_the_kernel_ends():
    parts = lambda n_out, k, bits=4, el="f16": mg.query_launch(n_out, 1, k, bits, 128, element=el, num_compute_units=256)["workgroups"] // (n_out // 16)  # noqa: E731
    assert [parts(1024, 512 * ks) for ks in (8, 9, 128, 129)] == [1, 4, 4, 1]
    assert [parts(1152, 512 * ks) for ks in (16, 17)] == [1, 2] and parts(2048, 512 * 20) == 2 and parts(2064, 512 * 20) == 1
    assert [parts(1024, 512 * ks, el="bf16") for ks in (4, 5)] == [1, 4] and [parts(2048, 512 * ks, el="bf16") for ks in (4, 5)] == [1, 2]
    assert parts(2176, 512 * 20, el="bf16") == 1 and [parts(1024, 256 * ks, 8, "bf16") for ks in (16, 17)] == [1, 4]


def problem(case, **more):
    n_out, k, bits, qop, group, bias, element, parts, waves = case
    return Problem(f"row parts{case}", n_out, k, bits, qop, group, m_batch=1, bias=bias, element=element, **more)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["auto", "general"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_parity_with_the_oracle(gpu, case, form):
    prob = problem(case)
    dev = DeviceProblem(prob, gpu)
    mg.set_dequant_form(mg.DEQUANT_EXACT_INTEGER if form == "general" else mg.DEQUANT_AUTO)
    try:
        y = dev.run()
    finally:
        mg.set_dequant_form(mg.DEQUANT_AUTO)
    if prob.element == "bf16":
        ulp, differing = bf16_ulp_report(y, prob.oracle_gemv(threads=16))
        assert ulp <= 1.0 + 1e-6 and differing <= 0.01
    else:
        assert float64_bound_violations(prob, y)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[3], CASES[5], CASES[7], CASES[9], CASES[-1]], ids=str)
def test_one_hot_rows_give_the_dequantised_columns(gpu, case):
    """One k at a time, in every slice and k step of a unit: each lane meets its own activations."""
    prob = problem(case[:5] + (False,) + case[6:])
    dequantised, dev = prob.oracle_dequant().view(np.uint16), None
    rng = np.random.default_rng(5)
    for at in [0, prob.k - 1, *rng.choice(prob.k, 40, replace=False)]:
        prob.x[:] = 0
        prob.x[0, at] = 0x3F80 if prob.element == "bf16" else 1.0
        got = DeviceProblem(prob, gpu).run().view(np.uint16).reshape(-1)
        want = dequantised[:, at]
        zero = (want & 0x7FFF) == 0   # a zero weight's sign is lost in the sum
        assert np.array_equal(np.where(zero, got & 0x7FFF, got), np.where(zero, 0, want)), at


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[2], CASES[7], CASES[9], CASES[11], CASES[-1]], ids=str)
def test_infinite_scales_stay_with_their_rows(gpu, case):
    """The last group's scales (or the columns') are infinite in some rows: those outputs are infinite as the oracle's, although the last
    unit reaches past the reduction, and the other rows are untouched."""
    prob = problem(case)
    prob.q[:] = np.abs(prob.q.astype(np.int16)).clip(1, 7)
    from oracle import pack_int4
    prob.w_raw = pack_int4(prob.q) if prob.bits == 4 else prob.q.view(np.uint8).copy()
    prob.scale[-1, ::5] = 0x7F80 if prob.element == "bf16" else np.inf
    prob.x[:] = 0x3F80 if prob.element == "bf16" else 1.0
    f32 = (lambda a: (a.astype(np.uint32) << 16).view(np.float32)) if prob.element == "bf16" else (lambda a: a.astype(np.float32))
    g, w = f32(DeviceProblem(prob, gpu).run()).reshape(-1), f32(prob.oracle_gemv(threads=16)).reshape(-1)
    assert np.isposinf(w[::5]).all() and np.array_equal(np.isposinf(g), np.isposinf(w)) and np.isfinite(g[w != np.inf]).all()
    ok = np.isfinite(w)
    assert not ok.any() or np.abs(g[ok] - w[ok]).max() <= (2.0 ** -7 if prob.element == "bf16" else 2e-3) * np.abs(w[ok]).max()


@pytest.mark.gpu
@pytest.mark.parametrize("default_plans", [True, False])
@pytest.mark.parametrize("case", [CASES[1], CASES[2], CASES[7], CASES[9], CASES[11], CASES[13]], ids=str)
def test_batched_and_routed_launches_have_the_bits_of_single_ones(gpu, case, default_plans):
    """However many problems: four parts, two, one, or whole tiles on the other kernel (all of them there without the measured plans)."""
    mg.set_default_plans(default_plans)
    try:
        batched_and_routed(gpu, case)
    finally:
        mg.set_default_plans(True)


def batched_and_routed(gpu, case):
    import torch
    n_out, k, bits, qop, group, bias, element = case[:7]
    most = 5
    probs = [problem(case, buffer=b) for b in range(most)]
    devs = [DeviceProblem(p, gpu) for p in probs]
    single = np.stack([d.run().copy().view(np.uint16) for d in devs])
    cat = lambda name: None if getattr(devs[0], name) is None else torch.stack([getattr(d, name) for d in devs])  # noqa: E731
    w, scale, zero, b, x = (cat(n) for n in ("w", "scale", "zero", "bias", "x"))
    strides = (w[0].numel(), k, scale[0].numel(), n_out if b is not None else 0, n_out)
    for count in range(1, most + 1):
        y = torch.full((most, 1, n_out), 0x7E00, dtype=torch.int16, device=gpu)
        mg.device_gemv(w, x, scale, zero, b, y, count, n_out, 1, k, group, qop, bits, batch_strides=strides, element=element)
        torch.cuda.synchronize()
        got = y.cpu().numpy().view(np.uint16)
        assert np.array_equal(got[:count], single[:count]) and (got[count:] == 0x7E00).all(), count
    x0 = torch.stack([devs[0].x] * most)
    ref = [DeviceProblem(probs[i], gpu) for i in (3, 0)]
    for r in ref:
        r.x.copy_(devs[0].x)
    want = [r.run().copy().view(np.uint16) for r in ref]
    route = torch.tensor([3, 0], dtype=torch.int32, device=gpu)
    y.fill_(0x7E00)
    mg.device_gemv_routed(w, x0, scale, zero, b, y, route, most, 2, n_out, 1, k, group, strides, qop, bits, element=element)
    torch.cuda.synchronize()
    got = y.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and (got[2:] == 0x7E00).all()
