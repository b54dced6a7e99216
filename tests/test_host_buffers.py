"""Host utilities on the buffers callers have: operands that share memory, with more elements than one thread takes."""
import ctypes

import numpy as np
import pytest

import oracle as orc
from mixed_gemv_amd import _lib

# above 65536 the work is dealt out over threads; an odd count of bytes leaves a remainder behind the vectors
COUNTS = [2, 62, 65536 * 2 + 66, 1 << 24]


def _at(array, offset=0):
    return ctypes.c_void_p(array.ctypes.data + offset)


@pytest.mark.parametrize("n", COUNTS)
@pytest.mark.parametrize("ahead", [0, 1, 5])
def test_packing_in_place_or_downwards(n, ahead):
    """The packed bytes may start at the unpacked ones, or in front of them: every byte is written behind its reads."""
    q = orc.fill_int8(n, 11, -8, 7)
    want = orc.pack_int4(q)
    for _ in range(5):
        buf = np.concatenate([np.zeros(ahead, np.int8), q])
        assert _lib.lib().mgemv_pack_int4(_at(buf), _at(buf, ahead), n) == 0
        assert np.array_equal(buf[:n // 2].view(np.uint8), want)


@pytest.mark.parametrize("n", COUNTS)
def test_unpacking_over_the_packed_upper_half(n):
    packed = orc.pack_int4(orc.fill_int8(n, 12, -8, 7))
    want = orc.unpack_int4(packed)
    for _ in range(5):
        buf = np.concatenate([np.zeros(n - n // 2, np.uint8), packed])
        assert _lib.lib().mgemv_unpack_int4(_at(buf), _at(buf, n - n // 2), n // 2) == 0
        assert np.array_equal(buf.view(np.int8), want)


@pytest.mark.parametrize("element", ["f16", "bf16"])
@pytest.mark.parametrize("n", [2, 30, 100003])
def test_folding_over_its_own_operands(element, n):
    """The result over the scales, in front of them, and over zero points kept in the upper half of its room."""
    rng = np.random.default_rng(n)
    scales = (rng.random(n) * 0.02 + 0.001).astype(np.float16).view(np.uint16)
    zeros = rng.integers(-8, 8, n).astype(np.int8)
    fold = _lib.lib().mgemv_fold_zero_points if element == "f16" else _lib.lib().mgemv_fold_zero_points_bf16
    want = np.empty(n, np.uint16)
    assert fold(_at(want), _at(scales), _at(zeros), n) == 0
    for ahead in (0, 1, 3):
        for _ in range(5):
            buf = np.concatenate([np.zeros(ahead, np.uint16), scales])
            assert fold(_at(buf), _at(buf, 2 * ahead), _at(zeros), n) == 0
            assert np.array_equal(buf[:n], want)
    for _ in range(5):
        buf = np.concatenate([np.zeros(n, np.int8), zeros])
        assert fold(_at(buf), _at(scales), _at(buf, n), n) == 0
        assert np.array_equal(buf.view(np.uint16), want)
