"""The kernels' group lookup (group_of, csrc/kernel_common.h) for group sizes that are no power of two, in its arithmetic:
    floor((q + 1/2) * rcp(d)) in fp32,  q = reduction position / 32,  d = group size / 32,
with a reciprocal that may be one unit in the last place off either way (v_rcp_f32), must be q / d.  For one d and one
reciprocal the product grows with q, so the two positions beside every group border stand for all q.  The kernels' limit
is 65 535 k steps of 512, q < 2^20; checked here twice as far, for every d below 4096 and a sample of those above."""
import numpy as np
import pytest


def border_errors(divisors, q_limit, unit):
    wrong = 0
    for d in divisors:
        exact = np.float32(1.0) / np.float32(d)                  # correctly rounded
        rcp = exact if unit == 0 else np.nextafter(exact, np.float32(2.0 * unit), dtype=np.float32)
        first = np.arange(0, q_limit, d, dtype=np.int64)         # the first position of every group
        for q, want in ((first, first // d), (first[1:] - 1, first[1:] // d - 1)):
            got = ((q.astype(np.float32) + np.float32(0.5)) * rcp).astype(np.int64)
            wrong += int((got != want).sum())
        last = q_limit - 1
        wrong += int(int((np.float32(last) + np.float32(0.5)) * rcp) != last // d)
    return wrong


@pytest.mark.parametrize("unit", [-1, 0, 1])
def test_every_group_border(unit):
    small = [d for d in range(2, 4096) if d & (d - 1)]
    assert border_errors(small, 1 << 21, unit) == 0
    rng = np.random.default_rng(5)
    large = sorted(set(rng.integers(4096, 1 << 21, 20000).tolist()) | {(1 << 21) - 1, (1 << 20) + 1, (1 << 20) - 16, 4097})
    assert border_errors(large, 1 << 21, unit) == 0


def test_the_check_sees_an_error():
    """Eight times the limit, where the quotient's error passes half a position, must fail."""
    assert border_errors([d for d in range(3, 64) if d & (d - 1)], 1 << 24, 1) > 0
