"""Launch rules of a single bf16 row on many tiles: 3 or 4 waves per tile, and every plan covers its problem."""
import pytest

import mixed_gemv_amd as mg


@pytest.mark.parametrize("bits,group", [(4, 128), (4, 96), (8, 64), (8, 96)])
@pytest.mark.parametrize("ksteps", [3, 4, 5, 6, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("tiles", [256, 703, 704, 705, 2000, 4097, 8016])
def test_plans_cover_the_problem(bits, group, ksteps, tiles):
    step = 512 if bits == 4 else 256
    k = ksteps * step // group * group
    plan = mg.query_launch(16 * tiles, 1, k, bits, group, element="bf16")
    cover = mg.plan_coverage(16 * tiles, 1, k, bits, group, element="bf16")
    assert cover["tiles_miscovered"] == 0 and cover["bad_waves"] == 0 and cover["lds_bytes_used"] <= cover["lds_bytes"]
    assert plan["threads"] <= 512 and plan["matrix_core"] == 0


def test_waves_per_tile():
    waves = lambda tiles, k, bits=4, group=128: mg.query_launch(16 * tiles, 1, k, bits, group, element="bf16")["split_k"]  # noqa: E731
    assert [waves(1200, 512 * ks) for ks in (3, 4, 5, 6, 7, 8)] == [3, 4, 3, 3, 4, 8]
    assert [waves(600, 512 * ks) for ks in (5, 6, 7, 8)] == [5, 6, 7, 8]                 # fewer tiles: a wave per k step
    assert waves(1400, 4096) == 8 and waves(1200, 4032, group=96) == 4             # 8 k steps: only with four groups per run
    assert waves(8016, 4096) == 4 and waves(8016, 4608, group=96) == 1 and waves(8016, 2048) == 4
    assert waves(1200, 256 * 6, bits=8) == 6 and waves(8016, 256 * 8, bits=8) == 4
