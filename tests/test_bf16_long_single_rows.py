"""A single bf16 row on 1.5 to 2 tiles per compute unit with a long reduction: four waves per tile where pairs of tiles had two each."""
import pytest

import mixed_gemv_amd as mg


@pytest.mark.parametrize("tiles, ksteps, bits, group, four", [
    (385, 25, 4, 128, True), (384, 25, 4, 128, False), (512, 56, 4, 64, True), (400, 24, 4, 128, False),
    (400, 18, 4, 96, True), (400, 17, 4, 96, False), (512, 40, 8, 96, True), (512, 40, 8, 128, False), (500, 30, 4, 0, True)])
def test_waves_per_tile(tiles, ksteps, bits, group, four):
    step = 512 if bits == 4 else 256
    k = ksteps * step // (group or 8) * (group or 8)
    plan = mg.query_launch(16 * tiles, 1, k, bits, group or k, element="bf16", num_compute_units=256)
    assert (plan["split_k"] == 4 and plan["tiles_per_wg"] == 1 and plan["workgroups"] == -(-tiles // 8) * 8) == four, plan
    cover = mg.plan_coverage(16 * tiles, 1, k, bits, group or k, element="bf16", num_compute_units=256)
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0 and cover["lds_bytes_used"] <= cover["lds_bytes"], cover
