"""The bf16 dequantisers' short forms at the edges of the scales they take: int4 products go through fp16, so their scales
span 12 binades at most, moved by a power of two per four rows; everything else takes the general form.  One-hot activation rows
make every output a single dequantised weight, so the comparison with the CPU oracle is bit for bit."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem

pytestmark = pytest.mark.gpu


def _bits(power, mantissa=0):
    return ((127 + power) << 7) | mantissa


SCALES = {
    # every scale inside the unmoved range, its first and last value among them
    "unmoved_edges": [_bits(-17), _bits(-17, 127), _bits(-6, 127), _bits(-10, 3)],
    "one_past_the_top": [_bits(-5), _bits(-6, 127), _bits(-8, 1), _bits(-5, 127)],
    "one_below_the_bottom": [_bits(-18, 127), _bits(-17), _bits(-12, 5), _bits(-18)],
    "moved_up_as_far_as_it_goes": [_bits(4, 9), _bits(4, 127), _bits(9, 127), _bits(-2)],
    "too_large_to_move": [_bits(20), _bits(20, 1), _bits(21, 127), _bits(25, 64)],
    "moved_down": [_bits(-25, 77), _bits(-25, 1), _bits(-31), _bits(-20, 127)],
    "too_small_to_move": [_bits(-60), _bits(-61, 5), _bits(-60, 127), _bits(-62)],
    "wider_than_four_rows_can_take": [_bits(-10, 1), _bits(3, 9), _bits(-30, 3), _bits(-5)],
    "signs_and_zeros": [0x0000, 0x8000, _bits(-9, 7) | 0x8000, _bits(-9, 7)],
}


# magnitudes of the four rows that share a range, by the first row's number / 4; the ranges reach from 2^-31 to 2^10
BY_FOUR_ROWS = {
    "ranges_of_their_own": lambda q, g: [-17 + 4 * (q % 5), -17 + 4 * (q % 5) + 11, -14 + 4 * (q % 5), -8 + 4 * (q % 5)],
    "smallest_first_and_last": lambda q, g: ([-31, -20, -25, -31], [-20, -31, -31, -28])[(q + g) % 2],
    "largest": lambda q, g: ([9, -2, 3, 8], [9, 9, 9, 9])[(q + g) % 2],
    "another_range_per_group": lambda q, g: [-30 + 9 * (g % 4) + r for r in (0, 11, 5, 2)],
    "one_binade_too_many": lambda q, g: [-20, -8 if (q, g) == (3, 0) else -9, -15, -12],
    "one_below_the_smallest": lambda q, g: [-32 if (q, g) == (18, 1) else -31, -25, -30, -21],
    "one_past_the_largest": lambda q, g: [10 if (q, g) == (0, 2) else 9, 0, 4, 9],
}


@pytest.mark.parametrize("name", sorted(SCALES) + sorted(BY_FOUR_ROWS))
@pytest.mark.parametrize("bits,qop,rows", [(4, SCALE_AND_ZEROS, 1), (4, SCALE_ONLY, 5), (4, SCALE_AND_ZEROS, 16),
                                           (8, SCALE_AND_ZEROS, 3), (4, PER_COLUMN, 2)])
def test_one_hot_rows_are_bit_exact_for_scales_at_the_edges(gpu, name, bits, qop, rows):
    import torch
    k = 1152 if bits == 4 else 640
    prob = Problem(f"bsf_{name}", 76, k, bits, qop, 64, m_batch=rows, element="bf16")
    if name in SCALES:
        values = np.array(SCALES[name], dtype=np.uint16)
        prob.scale = values[np.arange(prob.scale.size) % values.size].reshape(prob.scale.shape).copy()
    else:
        table = [[_bits(p, (37 * n + 11 * g) % 128) for n, p in enumerate(sum((BY_FOUR_ROWS[name](q, g) for q in range(19)), []))]
                 for g in range(prob.scale.size // 76)]
        prob.scale = np.array(table, dtype=np.uint16).reshape(prob.scale.shape)
    if prob.zero_add is not None:
        prob.zero_add[1::3, ::2] = 0x0001                      # subnormal
        prob.zero_add[::3, 1::2] = np.uint16(0x8000)
    dq = prob.oracle_dequant()
    dev = DeviceProblem(prob, gpu)
    assert np.array_equal(dev.dequant(), dq)
    for trial in range(3):
        hot = [(b * 131 + trial * 257) % k for b in range(rows)]
        x = np.zeros((rows, k), dtype=np.uint16)
        x[np.arange(rows), hot] = 0x3F80
        dev.x = torch.from_numpy(x.view(np.int16)).to(gpu)
        got = dev.run()
        for b in range(rows):
            want = dq[:, hot[b]]
            nz = (want & 0x7FFF) >= 0x0080                     # outputs below the normal range may lose bits in the sum
            assert np.array_equal(got[b][nz], want[nz]), (trial, b)
            assert np.all((got[b][~nz] & 0x7FFF) < 0x0080)
