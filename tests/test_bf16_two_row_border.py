"""Two bf16 rows with a lookup per block: the LDS-staged kernel takes over from the k-stationary one at a border of their own."""
import pytest

import mixed_gemv_amd as mg

LDS, KSTAT = 2, 3


@pytest.mark.parametrize("tiles, ksteps, group, taken", [
    (1793, 10, 96, False), (1793, 10, 128, True), (2817, 10, 96, True),     # 1.2 times as many units on the busiest SIMD; walks of 8 and 12
    (3589, 13, 96, False), (3589, 13, 64, True),                            # 1.15
    (1600, 6, 96, False), (3585, 9, 96, True), (1793, 9, 96, True), (2000, 5, 96, True)])   # 1.17 twice, 1.33, 1.6
def test_two_bf16_rows(tiles, ksteps, group, taken):
    k = ksteps * 512
    args = (16 * tiles, 2, k - k % group, 4, group)
    got = mg.query_launch(*args, element="bf16", num_compute_units=256)
    mg.set_default_plans(False)
    try:
        rules = mg.query_launch(*args, element="bf16", num_compute_units=256)
    finally:
        mg.set_default_plans(True)
    assert rules["matrix_core"] == KSTAT and got["matrix_core"] == (LDS if taken else KSTAT), (got, rules)
