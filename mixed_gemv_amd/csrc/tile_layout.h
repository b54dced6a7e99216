// Weight tile layout for 64-lane wavefronts and 128-bit loads on gfx950.
//
// This is the layout descriptor that takes the place of the reference's
// RowMajorTileInterleave<8,4> tag (layout/tile_interleaved_layout.h:42-47) and of the
// interleave arithmetic in utils/preprocess.h:292-348, 365-455.  It is shared by the host
// preprocessor and the device kernels so that the two cannot disagree.
//
// The n_out x k weight matrix is cut into UNITS of 16 rows x kStepK reduction elements.
// A unit is 4096 contiguous bytes = 4 BLOCKS of 1024 bytes; one block is exactly what one
// wavefront fetches with a single 128-bit-per-lane load (64 lanes x 16 bytes), so every wave
// load is one contiguous KiB and a wave that walks consecutive units streams one contiguous
// range.  Units are stored tile-major: unit (t, s) of row tile t and k step s starts at byte
// (t * ksteps + s) * 4096.
//
// Inside a unit, lane l of block i holds the 16-byte CHUNK of
//     row  16 t + (l % 16)
//     k    s*kStepK + (l / 16)*kRunK + i*kChunkK ... + kChunkK
// so lane l owns one row and, over the 4 blocks, one contiguous RUN of kRunK reduction
// elements of that row (128 for int4, 64 for int8): with a group size of 128 a lane needs a
// single scale/zero pair per unit.  The 16 lanes of a DPP row own 16 different rows at the
// SAME k range, so the activations of that range are held one piece per lane and handed
// round with DPP row broadcasts instead of being loaded 16 times.  The same arrangement
// (lane % 16 = row, lane / 16 = k slice) is the operand shape of the 16x16 matrix-core
// instructions, so the small-batch path consumes the identical buffer.
//
// A chunk is four 32-bit words in ascending k.  int4: a word holds 8 consecutive elements,
// each stored biased (value + 8) as a 4-bit field at these bits of the word (the field of element 5
// wraps round from bit 31 to bits 0-2):
//     e      0   1   2   3   4   5   6   7
//     bits  7-10 23-26 3-6 19-22 15-18 31,0-2 11-14 27-30
// The k-adjacent pair (2h, 2h+1) always lands at the SAME position of the two 16-bit halves,
// either at bits 7-10 or at bits 3-6 of the half, directly (h = 0, 1) or after rotating the
// word right by 8 (h = 2, 3).  Read as fp16, a half-word that is zero outside bits 0-10 has
// the value (bits) * 2^-24 -- exponent fields 0 and 1 continue each other linearly -- so one
// AND yields the packed pair (u * 2^-17, u' * 2^-17) or (u * 2^-21, u' * 2^-21) with no
// integer-to-float conversion at all; the kernels fold the missing power of two into the scale.
// int8: a word holds 4 consecutive elements in natural byte order, stored biased (value + 128).
//
// Rows are padded to a multiple of 16 and k to a multiple of kStepK with zero bytes; padded
// positions are never multiplied by a non-zero activation.
#ifndef MIXED_GEMV_AMD_TILE_LAYOUT_H_
#define MIXED_GEMV_AMD_TILE_LAYOUT_H_

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define MGEMV_HD __host__ __device__ inline
#else
#define MGEMV_HD inline
#endif

namespace mgemv {

constexpr int kTileRows = 16;       // rows per tile = lanes per DPP row
constexpr int kKSlices = 4;         // k slices per unit = DPP rows per wave
constexpr int kBlocksPerUnit = 4;   // wave loads per unit
constexpr int kChunkBytes = 16;     // one lane, one load
constexpr int kBlockBytes = 1024;   // one wave, one load
constexpr int kUnitBytes = kBlocksPerUnit * kBlockBytes;

template <int BITS>
struct Geometry {
  static_assert(BITS == 4 || BITS == 8, "int4 or int8 weights");
  static constexpr int kChunkK = kChunkBytes * 8 / BITS;        // 32 | 16
  static constexpr int kRunK = kBlocksPerUnit * kChunkK;        // 128 | 64
  static constexpr int kStepK = kKSlices * kRunK;               // 512 | 256
};

MGEMV_HD int chunk_k(int bits) { return kChunkBytes * 8 / bits; }
MGEMV_HD int run_k(int bits) { return kBlocksPerUnit * chunk_k(bits); }
MGEMV_HD int step_k(int bits) { return kKSlices * run_k(bits); }
MGEMV_HD int num_tiles(int n_out) { return (n_out + kTileRows - 1) / kTileRows; }
MGEMV_HD int num_ksteps(int k, int bits) { return (k + step_k(bits) - 1) / step_k(bits); }
MGEMV_HD size_t preprocessed_bytes(size_t n_out, size_t k, int bits) {
  size_t t = (n_out + kTileRows - 1) / kTileRows;
  size_t s = (k + (size_t)step_k(bits) - 1) / (size_t)step_k(bits);
  return t * s * (size_t)kUnitBytes;
}

// 32-bit words (W: one, or a vector of them) in natural order -- int4: element e in bits 4e..4e+3, two's complement --
// to stored order and back.  (In place: a wide vector as an argument or a result has no agreed place without the instructions for it.)
template <typename W>
MGEMV_HD void encode_int4(W& w) {
  const W b = w ^ 0x88888888u;  // +8 on each two's-complement nibble
  const W f5 = b & 0x00f00000u;
  w = ((b & 0x0000000fu) << 7) | ((b & 0x000000f0u) << 19) | ((b & 0x00000f00u) >> 5) | ((b & 0x0000f000u) << 7) |
      ((b & 0x000f0000u) >> 1) | (f5 << 11) | (f5 >> 21) | ((b & 0x0f000000u) >> 13) | ((b & 0xf0000000u) >> 1);
}
template <typename W>
MGEMV_HD void decode_int4(W& w) {
  const W f5 = ((w >> 11) | (w << 21)) & 0x00f00000u;
  w = (((w >> 7) & 0x0000000fu) | ((w >> 19) & 0x000000f0u) | ((w << 5) & 0x00000f00u) | ((w >> 7) & 0x0000f000u) |
       ((w << 1) & 0x000f0000u) | f5 | ((w << 13) & 0x0f000000u) | ((w << 1) & 0xf0000000u)) ^ 0x88888888u;
}
// (its own inverse)
template <typename W>
MGEMV_HD void recode_int8(W& w) { w = w ^ 0x80808080u; }

}  // namespace mgemv

#endif  // MIXED_GEMV_AMD_TILE_LAYOUT_H_
