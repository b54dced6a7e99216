"""Host utilities on the buffers callers have: operands that share memory, with more elements than one thread takes, and
byte buffers at any address."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as orc
from mixed_gemv_amd import _lib, build

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


ODD_ADDRESSES = """
import ctypes, sys
import numpy as np
lib = ctypes.CDLL(sys.argv[1])
vp = ctypes.c_void_p
rng = np.random.default_rng(3)
at = lambda a, off=0: vp(a.ctypes.data + off)
for bits, n_out, k in ((4, 36, 1048), (4, 16, 512), (8, 20, 528), (8, 48, 8)):
    shape = (ctypes.c_size_t * 2)(k, n_out)
    qt = 1 if bits == 4 else 0
    lib.mgemv_preprocessed_size.restype = ctypes.c_size_t
    size = lib.mgemv_preprocessed_size(shape, 2, qt)
    raw = rng.integers(0, 256, n_out * k * bits // 8, dtype=np.uint8)
    want = np.zeros(size, np.uint8)
    for off in (0, 1, 2, 7):
        src, dst, back = (np.zeros(n + 16, np.uint8) for n in (raw.size, size, raw.size))
        src[off:off + raw.size] = raw
        for layout in (1, 0):
            assert lib.mgemv_preprocess_weights(at(dst, off), at(src, off), shape, 2, layout, qt) == 0
        assert lib.mgemv_preprocess_weights(at(dst, off), at(src, off), shape, 2, 1, qt) == 0
        if off == 0:
            want[:] = dst[:size]
        assert np.array_equal(dst[off:off + size], want)
        assert lib.mgemv_unpreprocess_weights(at(back, off), at(dst, off), shape, 2, qt) == 0
        assert np.array_equal(back[off:off + raw.size], raw) and not back[off + raw.size:].any() and not dst[off + size:].any()
        wide, tight = np.zeros(2 * raw.size + 16, np.int8), np.zeros(raw.size + 16, np.uint8)
        assert lib.mgemv_unpack_int4(at(wide, off), at(src, off), ctypes.c_size_t(raw.size)) == 0
        assert lib.mgemv_pack_int4(at(tight, off), at(wide, off), ctypes.c_size_t(2 * raw.size)) == 0
        assert np.array_equal(tight[off:off + raw.size], raw)
print("ok")
"""


def test_byte_buffers_may_begin_at_any_address(tmp_path):
    """The host code built with a trap in front of every access at less than its type's alignment."""
    so = str(tmp_path / "host_utils.so")
    subprocess.run([build.hipcc(), "-x", "c++", "-std=c++17", "-O1", "-fPIC", "-shared", "-fvisibility=hidden", "-DMGEMV_BUILDING_LIBRARY",
                    "-fsanitize=alignment", "-fsanitize-trap=alignment", "-I", os.path.join(build.REPO_DIR, "include"), "-I", build.CSRC,
                    os.path.join(build.CSRC, "host_utils.cpp"), "-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", ODD_ADDRESSES, so], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
