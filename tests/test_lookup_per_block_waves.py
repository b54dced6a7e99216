"""A single row with a scale lookup per block on half a tile to one tile per compute unit: eight waves per tile with 9-16 k steps."""
import pytest

import mixed_gemv_amd as mg


@pytest.mark.parametrize("element", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tiles, ksteps, waves", [(129, 9, 5), (256, 16, 8), (200, 12, 6), (256, 15, 8), (200, 17, 4), (129, 4, 4), (257, 17, None)])
def test_waves_per_tile(tiles, ksteps, waves, bits, element):
    step = 512 if bits == 4 else 256
    k = ksteps * step // 96 * 96
    plan = mg.query_launch(16 * tiles, 1, k, bits, 96, element=element, num_compute_units=256)
    assert -(-k // step) == ksteps and (waves is None or plan["split_k"] == waves) and plan["matrix_core"] == 0, plan
    cover = mg.plan_coverage(16 * tiles, 1, k, bits, 96, element=element, num_compute_units=256)
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0 and cover["lds_bytes_used"] <= cover["lds_bytes"], cover
