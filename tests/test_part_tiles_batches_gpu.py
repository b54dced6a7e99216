"""Batched and routed launches of two and more rows on the part-tile matrix-core kernel: the more problems, the fewer parts of each
tile, down to one, and always the bits of single launches -- both numbers of chains, one to eight waves, chains that the reduction ends
in, waves without a unit, four and eight staged rows, both weight widths and types, every quant mode."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem

CASES = [
    # n_out, k, bits, quant_op, group, rows, bias, element, parts of a single launch, numbers of problems
    (996, 2560, 4, SCALE_AND_ZEROS, 128, 2, True, "f16", 4, (2, 3, 5)),      # 5 k steps in two ranges: the second has one
    (1024, 9984, 4, SCALE_AND_ZEROS, 64, 4, False, "f16", 4, (2, 4, 6)),     # 20, four rows staged
    (512, 17000, 4, PER_COLUMN, 0, 3, True, "bf16", 4, (2, 3, 8, 9)),        # 34, the last one short; waves of several chains
    (640, 8448, 8, SCALE_ONLY, 96, 4, True, "bf16", 4, (2, 3, 4, 7)),        # 33, four lookups per run
    (2044, 8320, 4, SCALE_AND_ZEROS, 128, 4, True, "bf16", 2, (2, 3)),       # 17: ranges of six, the last of five
    (1028, 2592, 4, SCALE_ONLY, 96, 2, False, "f16", 2, (2, 3, 5)),
    (1300, 4608, 4, SCALE_AND_ZEROS, 256, 8, True, "f16", 2, (2, 4)),        # eight rows staged
    (1000, 5088, 4, SCALE_AND_ZEROS, 96, 7, True, "bf16", 2, (2, 3, 5)),     # 10 k steps, five waves
    (328, 7168, 4, SCALE_ONLY, 256, 8, False, "f16", 2, (6,)),               # 42 parts six times: more than an XCD's compute units
    (1800, 16640, 8, SCALE_AND_ZEROS, 128, 6, False, "f16", 2, (2, 3)),      # 65
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_bits_of_single_launches(gpu, case):
    import torch
    n_out, k, bits, qop, group, rows, bias, element, parts, counts = case
    plan = mg.query_launch(n_out, rows, k, bits, group or k, element=element, num_compute_units=256)
    assert plan["matrix_core"] == 2 and plan["workgroups"] == -(-(-(-n_out // 16) * parts) // 8) * 8, plan
    most = max(counts)
    probs = [Problem(f"parts batch {case}", n_out, k, bits, qop, group, m_batch=rows, bias=bias, element=element, buffer=b) for b in range(3)]
    devs = [DeviceProblem(probs[b % 3], gpu) for b in range(3)]
    xs = [torch.roll(devs[0].x, shifts=8 * b, dims=1).contiguous() for b in range(most)]
    single = np.empty((3, most, rows, n_out), np.uint16)     # every matrix with every problem's rows
    for b, d in enumerate(devs):
        for i in range(most):
            d.x.copy_(xs[i])
            single[b, i] = d.run().view(np.uint16).reshape(rows, n_out)
    cat = lambda name: None if getattr(devs[0], name) is None else torch.stack([getattr(devs[b % 3], name) for b in range(most)])  # noqa: E731
    w, scale, zero, b_ = (cat(n) for n in ("w", "scale", "zero", "bias"))
    x = torch.stack(xs)
    strides = (w[0].numel(), rows * k, scale[0].numel(), n_out if bias else 0, rows * n_out)
    for count in counts:
        y = torch.full((most, rows, n_out), 0x7E00, dtype=torch.int16, device=gpu)
        mg.device_gemv(w, x, scale, zero, b_, y, count, n_out, rows, k, group or k, qop, bits, batch_strides=strides, element=element)
        torch.cuda.synchronize()
        got = y.cpu().numpy().view(np.uint16)
        for i in range(count):
            assert np.array_equal(got[i], single[i % 3, i]), (count, i)
        assert (got[count:] == 0x7E00).all()
        route = torch.tensor([(2 * i + 1) % 3 for i in range(count - 1)] + [most], dtype=torch.int32, device=gpu)   # the last: outside the stack
        y.fill_(0x7E00)
        mg.device_gemv_routed(w, x, scale, zero, b_, y, route, most, count, n_out, rows, k, group or k, strides, qop, bits, element=element)
        torch.cuda.synchronize()
        got = y.cpu().numpy().view(np.uint16)
        for i in range(count - 1):
            assert np.array_equal(got[i], single[(2 * i + 1) % 3, i]), (count, i)
        assert (got[count - 1:] == 0x7E00).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n_out, k, rows, element", [(996, 17000, 4, "f16"), (1020, 9000, 3, "bf16"), (2000, 9000, 6, "f16")])
def test_infinite_columns_where_a_run_lies_partly_past_the_reduction(gpu, n_out, k, rows, element):
    """Per-column scales: those rows' outputs are infinite or not a number, the same ones however many problems, the others finite."""
    import torch
    assert mg.query_launch(n_out, rows, k, 4, k, element=element, num_compute_units=256)["workgroups"] > 2 * (n_out // 16) - 8
    prob = Problem("infinite columns", n_out, k, 4, PER_COLUMN, 0, m_batch=rows, element=element)
    prob.scale[0, ::5] = 0x7F80 if element == "bf16" else np.inf
    inf = 0x7F80 if element == "bf16" else 0x7C00
    special = lambda y: np.where((y & 0x7FFF) > inf, 2, np.where((y & 0x7FFF) == inf, 1, 0))  # noqa: E731
    dev = DeviceProblem(prob, gpu)
    single = dev.run().copy().view(np.uint16).reshape(rows, n_out)
    assert (special(single)[:, ::5] > 0).all() and (np.delete(special(single), np.s_[::5], axis=1) == 0).all()
    w, scale, x = (torch.stack([t] * 6) for t in (dev.w, dev.scale, dev.x))
    strides = (w[0].numel(), rows * k, n_out, 0, rows * n_out)
    for count in (2, 3, 6):
        y = torch.full((6, rows, n_out), 0x7E01, dtype=torch.int16, device=gpu)
        mg.device_gemv(w, x, scale, None, None, y, count, n_out, rows, k, k, PER_COLUMN, 4, batch_strides=strides, element=element)
        torch.cuda.synchronize()
        for got in y.cpu().numpy().view(np.uint16)[:count]:
            assert np.array_equal(special(got), special(single)), count
            assert np.array_equal(got[special(got) < 2], single[special(got) < 2]), count
