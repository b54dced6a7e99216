"""Batched and routed single rows whose problems take one part of each tile on the VALU kernel for parts: waves of one or two units up to
16 k steps, a wave for every fourth k step beyond, with four lookups per run, whatever the last k step or wave is short of, up to the
most k steps -- and always the bits of single launches."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem
from test_single_row_parts_gpu import batched_and_routed, plan_of, problem

CASES = [
    # n_out, k, bits, quant_op, group, bias, element, parts, waves of the single launch
    (1020, 4320, 4, SCALE_AND_ZEROS, 96, True, "bf16", 4, 3),      # 9 k steps: waves of two units, the last of one
    (2048, 4896, 4, SCALE_ONLY, 96, False, "bf16", 2, 5),          # 10
    (1500, 7400, 4, PER_COLUMN, 0, True, "bf16", 2, 8),            # 15, the last one short
    (1000, 9312, 4, SCALE_AND_ZEROS, 96, True, "f16", 4, 5),       # 19, the last one short: waves of five and four units
    (2000, 9000, 4, PER_COLUMN, 0, True, "f16", 2, 3),             # 18
    (1024, 16640, 4, SCALE_ONLY, 64, False, "bf16", 4, 3),         # 33
    (1300, 4608, 8, SCALE_AND_ZEROS, 96, False, "f16", 2, 3),      # 18
    (1024, 32768, 8, SCALE_AND_ZEROS, 128, True, "f16", 4, 4),     # 128 k steps, the most
    (1004, 32640, 8, SCALE_AND_ZEROS, 96, False, "bf16", 4, 4),    # 128, the last one short
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_bits_of_single_launches(gpu, case):
    plan = plan_of(case)
    assert plan["split_k"] == case[8] and plan["workgroups"] == -(-(-(-case[0] // 16) * case[7]) // 8) * 8, plan
    batched_and_routed(gpu, case)


INFINITE = [
    (1000, 4704, 4, SCALE_AND_ZEROS, 96, False, "f16", 4, 3),      # 10 k steps; many problems take whole tiles, a wave per k step
    (1000, 4736, 4, PER_COLUMN, 0, True, "f16", 4, 3),
    (1020, 2400, 4, SCALE_ONLY, 96, True, "bf16", 4, 2),           # 5
    (1020, 3712, 4, PER_COLUMN, 0, False, "bf16", 4, 2),           # 8
    (1020, 2464, 8, SCALE_ONLY, 0, False, "f16", 4, 3),            # 10, one group as long as the reduction
    (1020, 4320, 4, SCALE_AND_ZEROS, 96, True, "bf16", 4, 3),      # 9: one part
    (1000, 9312, 4, SCALE_AND_ZEROS, 96, True, "f16", 4, 5),       # 19: a wave for every fourth k step
    (1000, 17000, 4, PER_COLUMN, 0, True, "f16", 4, 3),            # a run that lies partly past the reduction
    (1500, 9000, 4, PER_COLUMN, 0, True, "bf16", 2, 3),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", INFINITE, ids=str)
def test_infinities_of_single_and_batched_launches(gpu, case):
    """Infinite scales of the last group (of the column), and a last k step that is short: the outputs that are infinite or not a number
    are the same however many problems a launch has, and where no lane's run lies partly past the reduction they are the oracle's."""
    import torch
    n_out, k, bits, qop, group, bias, element = case[:7]
    case = (*case[:4], group or k, *case[5:])
    prob = problem(case)
    prob.q[:] = np.abs(prob.q.astype(np.int16)).clip(1, 7)
    from oracle import pack_int4
    prob.w_raw = pack_int4(prob.q) if bits == 4 else prob.q.view(np.uint8).copy()
    prob.scale[-1, ::5] = 0x7F80 if element == "bf16" else np.inf
    prob.x[:] = 0x3F80 if element == "bf16" else 1.0
    inf = 0x7F80 if element == "bf16" else 0x7C00
    special = lambda y: np.where((y & 0x7FFF) > inf, 2, np.where((y & 0x7FFF) == inf, 1, 0))  # noqa: E731
    dev = DeviceProblem(prob, gpu)
    single = dev.run().copy().view(np.uint16).reshape(-1)
    assert (special(single)[::5] > 0).all() and (np.delete(special(single), np.s_[::5]) == 0).all()
    if k % 128 == 0 or qop != PER_COLUMN:
        assert np.array_equal(special(single), special(prob.oracle_gemv(threads=16).view(np.uint16).reshape(-1)))
    most = 6
    cat = lambda t: None if t is None else torch.stack([t] * most)  # noqa: E731
    w, scale, zero, b, x = (cat(getattr(dev, name)) for name in ("w", "scale", "zero", "bias", "x"))
    strides = (w[0].numel(), k, scale[0].numel(), n_out if bias else 0, n_out)
    for count in (2, 3, 6):
        y = torch.full((most, 1, n_out), 0x7E01, dtype=torch.int16, device=gpu)
        mg.device_gemv(w, x, scale, zero, b, y, count, n_out, 1, k, group or k, qop, bits, batch_strides=strides, element=element)
        torch.cuda.synchronize()
        for got in y.cpu().numpy().view(np.uint16)[:count, 0]:
            assert np.array_equal(special(got), special(single)), count
            assert np.array_equal(got[special(got) < 2], single[special(got) < 2]), count
