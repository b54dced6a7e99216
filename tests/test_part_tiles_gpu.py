"""The part-tile matrix-core kernel (a workgroup per 16, 8 or 4 rows of a tile, one, two or four k steps at a time): which launches
take it, and its results against the CPU oracle where it can go wrong -- the last unit of a reduction shorter than the others, rows
and whole parts past the matrix, the most rows each split has columns for, one to eight waves and units per wave, both weight
widths, every quant mode, four lookups per run, both dequantiser forms.

Bars: fp16 outputs within what the mathematics allows any fp32 accumulation of the dequantised weights
(helpers.float64_bound_violations), bf16 outputs the oracle's or a neighbour, at most 1 % of them differing."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem, bf16_ulp_report, float64_bound_violations

CASES = [
    # n_out, k, bits, quant_op, group, rows, bias, element, parts, waves
    (40, 2560, 4, SCALE_AND_ZEROS, 128, 2, True, "f16", 4, 2),          # 5 k steps: a last unit of one; parts past n_out
    (1024, 3584, 4, SCALE_AND_ZEROS, 64, 4, False, "f16", 4, 2),        # 7: a last unit of three
    (1020, 6144, 4, PER_COLUMN, 0, 3, True, "bf16", 4, 3),
    (996, 17000, 4, PER_COLUMN, 0, 4, False, "f16", 4, 3),              # 34 k steps, the last one short, in 9 units of 3 waves
    (24, 8448, 8, SCALE_ONLY, 96, 4, True, "bf16", 4, 3),
    (1028, 2592, 4, SCALE_ONLY, 96, 2, False, "f16", 2, 3),             # 6
    (2044, 8320, 4, SCALE_AND_ZEROS, 128, 4, True, "bf16", 2, 3),       # 17: one k step in the last unit
    (36, 4608, 4, SCALE_AND_ZEROS, 256, 8, True, "f16", 2, 5),          # 16 columns: 8 rows of two k steps
    (2048, 4096, 4, SCALE_AND_ZEROS, 64, 5, False, "f16", 2, 4),
    (1000, 5088, 4, SCALE_AND_ZEROS, 96, 7, True, "bf16", 2, 5),
    (1800, 16640, 8, SCALE_AND_ZEROS, 128, 6, False, "f16", 2, 4),      # 65: 33 units of 4 waves, the last one short
    (1000, 5120, 8, PER_COLUMN, 0, 8, True, "bf16", 2, 4),
    (100, 4864, 4, SCALE_AND_ZEROS, 128, 16, True, "f16", 1, 4),        # 10 k steps, four waves
    (1900, 2560, 4, SCALE_ONLY, 64, 9, False, "bf16", 1, 5),
    (4096, 8704, 4, SCALE_AND_ZEROS, 128, 3, True, "f16", 1, 4),        # 17
    (4092, 2048, 8, SCALE_AND_ZEROS, 64, 16, True, "f16", 1, 8),
    (6000, 8960, 4, SCALE_AND_ZEROS, 128, 3, False, "bf16", 2, 3),      # more workgroups than compute units
    (9000, 8928, 4, SCALE_ONLY, 96, 4, True, "f16", 1, 4),
]


def plan_of(case):
    n_out, k, bits, qop, group, rows, bias, element, parts, waves = case
    return mg.query_launch(n_out, rows, k, bits, k if qop == PER_COLUMN else group, element=element, num_compute_units=256)


@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_launch_takes_the_kernel(case):
    plan, tiles = plan_of(case), -(-case[0] // 16)
    assert plan["matrix_core"] == 2 and plan["tiles_per_wg"] == 1 and plan["split_k"] == case[9], plan
    assert plan["workgroups"] == -(-tiles * case[8] // 8) * 8 and plan["steps_per_wave"] % case[8] == 0, plan
    cover = mg.plan_coverage(case[0], case[5], case[1], case[2], case[4] or case[1], element=case[7], num_compute_units=256)
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0, cover
    mg.set_default_plans(False)
    try:
        assert plan_of(case) != plan
    finally:
        mg.set_default_plans(True)


def problem(case, **more):
    n_out, k, bits, qop, group, rows, bias, element, parts, waves = case
    return Problem(f"parts{case}", n_out, k, bits, qop, group, m_batch=rows, bias=bias, element=element, **more)


def within_bars(prob, y):
    if prob.element == "bf16":
        ulp, differing = bf16_ulp_report(y, prob.oracle_gemv(threads=16))
        return ulp <= 1.0 + 1e-6 and differing <= 0.01
    return float64_bound_violations(prob, y)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["auto", "general"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_parity_with_the_oracle(gpu, case, form):
    prob = problem(case)
    dev = DeviceProblem(prob, gpu)
    mg.set_dequant_form(mg.DEQUANT_EXACT_INTEGER if form == "general" else mg.DEQUANT_AUTO)
    try:
        assert within_bars(prob, dev.run())
    finally:
        mg.set_dequant_form(mg.DEQUANT_AUTO)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[3], CASES[6], CASES[10], CASES[12]], ids=str)
def test_one_hot_rows_give_the_dequantised_columns(gpu, case):
    """Each activation row picks a k of its own: the lanes of every k step of a unit meet their own activations."""
    prob = problem(case[:6] + (False,) + case[7:])
    rng = np.random.default_rng(5)
    at = rng.choice(prob.k, prob.m_batch, replace=False)
    at[0] = prob.k - 1
    prob.x[:] = 0
    prob.x[np.arange(prob.m_batch), at] = 0x3F80 if prob.element == "bf16" else 1.0
    got = DeviceProblem(prob, gpu).run().view(np.uint16)
    want = prob.oracle_dequant().view(np.uint16)[:, at].T
    zero = (want & 0x7FFF) == 0   # a zero weight's sign is lost in the sum
    assert np.array_equal(np.where(zero, got & 0x7FFF, got), np.where(zero, 0, want))


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[2], CASES[6], CASES[10]], ids=str)
def test_infinite_scales_stay_with_their_rows_and_groups(gpu, case):
    """The last group's scales (or the columns') are infinite in some rows: those outputs are what the oracle gives, infinite or not
    a number, although the last unit reaches past the reduction; the other rows are untouched, and so are the activation rows beside
    one of infinities."""
    prob = problem(case)
    prob.q[:] = np.abs(prob.q.astype(np.int16)).clip(1, 7)
    from oracle import pack_int4
    prob.w_raw = pack_int4(prob.q) if prob.bits == 4 else prob.q.view(np.uint8).copy()
    inf = 0x7F80 if prob.element == "bf16" else np.inf
    prob.scale[-1, ::5] = inf
    prob.x[:, -1] = 0x3F80 if prob.element == "bf16" else 1.0
    prob.x[0] = 0x3F80 if prob.element == "bf16" else 1.0
    if prob.m_batch > 2:
        prob.x[2, 8] = inf
    got, want = DeviceProblem(prob, gpu).run(), prob.oracle_gemv(threads=16)
    f32 = (lambda a: (a.astype(np.uint32) << 16).view(np.float32)) if prob.element == "bf16" else (lambda a: a.astype(np.float32))
    g, w = f32(got), f32(want.reshape(got.shape))
    assert np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(np.isposinf(g), np.isposinf(w)) and np.array_equal(np.isneginf(g), np.isneginf(w))
    assert np.isposinf(w[0, ::5]).all() and np.isfinite(w[1]).any()
    ok = np.isfinite(w)
    rms = np.sqrt(np.mean(w[ok] ** 2))
    assert np.abs(g[ok] - w[ok]).max() <= (2.0 ** -7 if prob.element == "bf16" else 2e-3) * max(rms, np.abs(w[ok]).max())


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[1], CASES[8], CASES[13]], ids=str)
def test_batched_and_routed_launches_have_the_bits_of_single_ones(gpu, case):
    import torch
    n_out, k, bits, qop, group, rows, bias, element = case[:8]
    probs = [problem(case, buffer=b) for b in range(3)]
    devs = [DeviceProblem(p, gpu) for p in probs]
    single = [d.run().copy().view(np.uint16) for d in devs]
    cat = lambda name: None if getattr(devs[0], name) is None else torch.stack([getattr(d, name) for d in devs])  # noqa: E731
    w, scale, zero, b = (cat(n) for n in ("w", "scale", "zero", "bias"))
    x = torch.stack([devs[0].x] * 3)
    strides = (w[0].numel(), rows * k, scale[0].numel(), n_out if b is not None else 0, rows * n_out)
    y = torch.full((3, rows, n_out), 0x7E00, dtype=torch.int16, device=gpu)
    mg.device_gemv(w, x, scale, zero, b, y, 3, n_out, rows, k, group, qop, bits, batch_strides=strides, element=element)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), np.stack(single))     # the activations are the same in every buffer
    route = torch.tensor([2, 0], dtype=torch.int32, device=gpu)
    y.fill_(0x7E00)
    mg.device_gemv_routed(w, x, scale, zero, b, y, route, 3, 2, n_out, rows, k, group, strides, qop, bits, element=element)
    torch.cuda.synchronize()
    got = y.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[0], single[2]) and np.array_equal(got[1], single[0]) and (got[2] == 0x7E00).all()
