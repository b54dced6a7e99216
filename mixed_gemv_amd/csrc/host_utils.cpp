// Host-side utilities of the library: int4 packing, zero-point folding and the weight
// preprocessor that produces the gfx950 tile layout.  They stand in for
// utils/preprocess.h:41-84 (SubBytePacker), :94-101 (ZeroPointPreprocessor) and :482-522
// (MixedGemvWeightPreprocessor::run) of the reference: same inputs, same meaning, new layout.
#include <cstring>
#include <vector>

#include "mixed_gemv.h"
#include "tile_layout.h"

namespace {

// The loops below are written on vectors and compiled three times: for any x86-64 (SSE2), for AVX2 and for AVX-512; the
// processor says which one runs.  Called from Python on 16 threads of an EPYC, SSE2 / AVX-512: a 4096x4096 int4 matrix laid out
// 54 us / 24, packed 27 / 17, 131072 zero points folded 15.5 / 11 (most of it the call and the threads); the three together 113 / 63.
// (New inputs with every result kept, as loading a model has it: 515-645 us / 475-535, most of it page faults of the results.)
// A loop is a class whose run<W> takes the variant's vector of 32-bit words and is inlined into a function of that variant.
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define MGEMV_FOR(isa) __attribute__((target(isa)))
#define MGEMV_VARIANTS 1
#else
#define MGEMV_FOR(isa)
#define MGEMV_VARIANTS 0
#endif
#define MGEMV_INLINE inline __attribute__((always_inline))
typedef uint32_t word4 __attribute__((vector_size(16)));
typedef uint32_t word8 __attribute__((vector_size(32)));
typedef uint32_t word16 __attribute__((vector_size(64)));

template <typename Loop, typename... Args>
void run_plain(Args... args) { Loop::template run<word4>(args...); }
template <typename Loop, typename... Args>
MGEMV_FOR("avx2") void run_avx2(Args... args) { Loop::template run<word8>(args...); }
template <typename Loop, typename... Args>
MGEMV_FOR("avx512f,avx512bw,avx512vl") void run_avx512(Args... args) { Loop::template run<word16>(args...); }

int vector_variant() {
#if MGEMV_VARIANTS
  static const int variant = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512vl") ? 2
                             : __builtin_cpu_supports("avx2")                                                                         ? 1
                                                                                                                                       : 0;
  return variant;
#else
  return 0;
#endif
}
template <typename Loop, typename... Args>
void run_loop(Args... args) {
  switch (vector_variant()) {
    case 2: return run_avx512<Loop, Args...>(args...);
    case 1: return run_avx2<Loop, Args...>(args...);
    default: return run_plain<Loop, Args...>(args...);
  }
}

// ---- binary16 helpers (host): eight values at a time, selects instead of branches -----------

typedef uint16_t u16x8 __attribute__((vector_size(16)));
typedef int8_t i8x8 __attribute__((vector_size(8)));
typedef uint32_t u32x8 __attribute__((vector_size(32)));
typedef float f32x8 __attribute__((vector_size(32)));

// (by reference: a 32-byte vector argument has no agreed place without AVX)
MGEMV_INLINE void half_bits_to_float(const u16x8& h16, f32x8& f) {
  // Place exponent+mantissa in the binary32 fields, then multiply by 2^(127-15) = 2^112:
  // exact for normals, and it normalises subnormals for free.
  const u32x8 h = __builtin_convertvector(h16, u32x8);
  const u32x8 sign = (h & 0x8000u) << 16, body = h & 0x7fffu;
  const u32x8 scaled = (u32x8)((f32x8)(body << 13) * 0x1p112f);
  const u32x8 special = 0x7f800000u | ((body & 0x3ffu) << 13);
  f = (f32x8)(sign | (body >= 0x7c00u ? special : scaled));
}

// binary32 -> binary16, round-to-nearest-even.
MGEMV_INLINE void float_to_half_bits(const f32x8& f, u16x8& h) {
  const u32x8 sign = ((u32x8)f >> 16) & 0x8000u, x = (u32x8)f & 0x7fffffffu;
  const u32x8 nan = (u32x8){} + 0x7e00u, inf = (u32x8){} + 0x7c00u;
  const u32x8 big = x > 0x7f800000u ? nan : inf;  // |f| >= 65536, inf or nan
  // |f| < 2^-14: the result is subnormal (or zero).  Adding 0.5 shifts the value so that the binary32 unit in the last
  // place is 2^-24, the subnormal half spacing; the hardware's RNE does the rounding.
  const u32x8 small = (u32x8)((f32x8)x + 0.5f) - 0x3f000000u;
  // rebias the exponent by (15 - 127) and add the rounding bias 0xfff, and one more where ties have to go up to even
  const u32x8 normal = (x + 0xc8000fffu + ((x >> 13) & 1u)) >> 13;
  const u32x8 body = x < 0x38800000u ? small : normal;
  h = __builtin_convertvector(sign | (x >= 0x47800000u ? big : body), u16x8);
}

// Elements a thread should have at least (a few microseconds' work: what starting the others costs).
constexpr size_t kGrain = (size_t)1 << 15;

bool share_memory(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
  const uintptr_t a0 = (uintptr_t)a, b0 = (uintptr_t)b;
  return a0 < b0 + b_bytes && b0 < a0 + a_bytes;
}

// fn(first, last) over pieces of `grain` elements of [0, n), side by side where there is enough to do.  in_order: one
// ascending piece, for a result that lies over its operands -- a thread would write what another has yet to read.
template <typename Fn>
void in_pieces(size_t n, size_t grain, bool in_order, Fn fn) {
  const size_t pieces = in_order ? 1 : (n + grain - 1) / grain;
  if (pieces <= 1) {
    fn((size_t)0, n);
    return;
  }
#pragma omp parallel for schedule(static)
  for (long long i = 0; i < (long long)pieces; ++i) {
    const size_t first = (size_t)i * grain;
    fn(first, first + grain < n ? first + grain : n);
  }
}

bool shape_ok(const size_t* shape, int rank, size_t& experts, size_t& k, size_t& n_out) {
  if (shape == nullptr || (rank != 2 && rank != 3)) return false;
  experts = rank == 2 ? 1 : shape[0];
  k = rank == 2 ? shape[0] : shape[1];
  n_out = rank == 2 ? shape[1] : shape[2];
  return true;
}

int bits_of_quant_type(int quant_type) {
  if (quant_type == MGEMV_W4_A16) return 4;
  if (quant_type == MGEMV_W8_A16) return 8;
  return 0;
}

// Transpose a [k][n_out] matrix of `bits`-wide elements into [n_out][k] (both densely packed,
// low nibble = even index).  Blocked so that both sides are walked in cache-sized tiles.
void transpose_quantised(uint8_t* dst, const uint8_t* src, size_t k, size_t n_out, int bits) {
  constexpr size_t kBlock = 64;
  const long long n_blocks = (long long)((n_out + kBlock - 1) / kBlock);
  // one thread per block of 64 output rows: no two threads write the same byte (k is even)
#pragma omp parallel for schedule(static)
  for (long long nb = 0; nb < n_blocks; ++nb) {
    const size_t n0 = (size_t)nb * kBlock;
    const size_t n1 = n0 + kBlock < n_out ? n0 + kBlock : n_out;
    if (bits == 4) std::memset(dst + n0 * k / 2, 0, (n1 - n0) * k / 2);
    for (size_t k0 = 0; k0 < k; k0 += kBlock) {
      const size_t k1 = k0 + kBlock < k ? k0 + kBlock : k;
      if (bits == 8) {
        for (size_t n = n0; n < n1; ++n)
          for (size_t kk = k0; kk < k1; ++kk) dst[n * k + kk] = src[kk * n_out + n];
      } else {
        for (size_t n = n0; n < n1; ++n)
          for (size_t kk = k0; kk < k1; ++kk) {
            const size_t si = kk * n_out + n;
            const uint8_t v = (uint8_t)((src[si >> 1] >> (4 * (si & 1))) & 0xfu);
            const size_t di = n * k + kk;
            dst[di >> 1] = (uint8_t)(dst[di >> 1] | (v << (4 * (di & 1))));
          }
      }
    }
  }
}

template <int BITS, bool DECODE, typename W>
MGEMV_INLINE void recode_words(W& w) {
  if constexpr (BITS == 8) mgemv::recode_int8(w);
  else if constexpr (DECODE) mgemv::decode_int4(w);
  else mgemv::encode_int4(w);
}

// One 16-row tile between rows (row_bytes apart, `rows` of them) and its units.  A lane's run -- 64 bytes of one row, whose
// four chunks go to the four blocks of a unit -- is a cache line of the row, and the unit's 4 KiB stay in the first-level
// cache while the runs of 16 rows x 4 slices fill them, so that both sides are walked line by line.  (A row at a time,
// as the first version of this loop had it, comes back to each line of the tiled side four times.)
template <int BITS, bool DECODE>
struct RecodeTile {
  template <typename W>
  static MGEMV_INLINE void run(uint8_t* units, uint8_t* rows_base, size_t rows, size_t row_bytes, size_t ksteps);
};
template <int BITS, bool DECODE>
template <typename W>
MGEMV_INLINE void RecodeTile<BITS, DECODE>::run(uint8_t* units, uint8_t* rows_base, size_t rows, size_t row_bytes, size_t ksteps) {
  constexpr size_t kRunBytes = (size_t)mgemv::kBlocksPerUnit * mgemv::kChunkBytes;
  for (size_t s = 0; s < ksteps; ++s) {
    uint8_t* const unit = units + s * (size_t)mgemv::kUnitBytes;
    for (size_t slice = 0; slice < (size_t)mgemv::kKSlices; ++slice) {
      const size_t off = (s * mgemv::kKSlices + slice) * kRunBytes;
      if (off >= row_bytes) break;  // a run past k: left as it is (zero)
      const size_t here = row_bytes - off < kRunBytes ? row_bytes - off : kRunBytes;
      for (size_t r = 0; r < rows; ++r) {
        uint8_t* const row = rows_base + r * row_bytes + off;
        uint8_t* const lane = unit + (slice * mgemv::kTileRows + r) * mgemv::kChunkBytes;
        if (here == kRunBytes) {
          constexpr int kChunks = (int)sizeof(W) / mgemv::kChunkBytes;
          for (int blk = 0; blk < mgemv::kBlocksPerUnit; blk += kChunks) {
            W w;
            uint8_t* const in_row = row + blk * mgemv::kChunkBytes;
            uint8_t* const in_unit = lane + blk * mgemv::kBlockBytes;
            if (DECODE)
              for (int c = 0; c < kChunks; ++c)
                std::memcpy(reinterpret_cast<uint8_t*>(&w) + c * mgemv::kChunkBytes, in_unit + c * mgemv::kBlockBytes, mgemv::kChunkBytes);
            else
              std::memcpy(&w, in_row, sizeof(W));
            recode_words<BITS, DECODE>(w);
            if (DECODE)
              std::memcpy(in_row, &w, sizeof(W));
            else
              for (int c = 0; c < kChunks; ++c)
                std::memcpy(in_unit + c * mgemv::kBlockBytes, reinterpret_cast<uint8_t*>(&w) + c * mgemv::kChunkBytes, mgemv::kChunkBytes);
          }
          continue;
        }
        for (size_t blk = 0; blk * mgemv::kChunkBytes < here; ++blk) {
          const size_t valid = here - blk * mgemv::kChunkBytes < (size_t)mgemv::kChunkBytes ? here - blk * mgemv::kChunkBytes
                                                                                           : (size_t)mgemv::kChunkBytes;
          word4 w = {0, 0, 0, 0};  // positions past k inside a chunk: any value, they only ever meet zero activations
          uint8_t* const in_unit = lane + blk * mgemv::kBlockBytes;
          std::memcpy(&w, DECODE ? in_unit : row + blk * mgemv::kChunkBytes, DECODE ? (size_t)mgemv::kChunkBytes : valid);
          recode_words<BITS, DECODE>(w);
          std::memcpy(DECODE ? row + blk * mgemv::kChunkBytes : in_unit, &w, DECODE ? valid : (size_t)mgemv::kChunkBytes);
        }
      }
    }
  }
}

// One matrix between rows of k elements (n_out rows) and the tile layout.
template <int BITS, bool DECODE>
void recode_matrix(uint8_t* tiled, uint8_t* rows, size_t n_out, size_t k) {
  const size_t ksteps = (size_t)mgemv::num_ksteps((int)k, BITS), tiles = (size_t)mgemv::num_tiles((int)n_out);
  const size_t row_bytes = k * (size_t)BITS / 8, tile_bytes = ksteps * (size_t)mgemv::kUnitBytes;
  const bool padded = k % (size_t)mgemv::step_k(BITS) != 0;
#pragma omp parallel for schedule(static) if (tiles * tile_bytes >= 4 * kGrain)
  for (long long t = 0; t < (long long)tiles; ++t) {
    const size_t row0 = (size_t)t * mgemv::kTileRows;
    const size_t here = n_out - row0 < (size_t)mgemv::kTileRows ? n_out - row0 : (size_t)mgemv::kTileRows;
    uint8_t* const tile = tiled + (size_t)t * tile_bytes;
    // zero bytes only where the layout pads: rows past n_out, reduction positions past k
    if (!DECODE && (padded || here < (size_t)mgemv::kTileRows)) std::memset(tile, 0, tile_bytes);
    run_loop<RecodeTile<BITS, DECODE>>(tile, rows + row0 * row_bytes, here, row_bytes, ksteps);
  }
}

void tile_one_matrix(uint8_t* dst, const uint8_t* src, size_t n_out, size_t k, int bits) {
  uint8_t* const rows = const_cast<uint8_t*>(src);  // only read
  if (bits == 4) recode_matrix<4, false>(dst, rows, n_out, k); else recode_matrix<8, false>(dst, rows, n_out, k);
}

void untile_one_matrix(uint8_t* dst, const uint8_t* src, size_t n_out, size_t k, int bits) {
  uint8_t* const tiled = const_cast<uint8_t*>(src);  // only read
  if (bits == 4) recode_matrix<4, true>(tiled, dst, n_out, k); else recode_matrix<8, true>(tiled, dst, n_out, k);
}

// Two elements a byte.  A 16-bit pair holds element 2i in its low byte and 2i + 1 in its high one.
struct PackInt4 {
  template <typename W>
  static MGEMV_INLINE void run(uint8_t* packed, const int8_t* unpacked, size_t first, size_t last) {
    constexpr size_t kBytes = sizeof(W);  // packed at a time
    typedef uint16_t pairs __attribute__((vector_size(2 * kBytes)));
    typedef uint8_t bytes __attribute__((vector_size(kBytes)));
    size_t i = first;
    for (; i + kBytes <= last; i += kBytes) {
      pairs v;
      std::memcpy(&v, unpacked + 2 * i, sizeof(v));
      const bytes b = __builtin_convertvector((v & 0x000f) | ((v >> 4) & 0x00f0), bytes);
      std::memcpy(packed + i, &b, sizeof(b));
    }
    for (; i < last; ++i)
      packed[i] = (uint8_t)(((unsigned)unpacked[2 * i] & 0xfu) | (((unsigned)unpacked[2 * i + 1] & 0xfu) << 4));
  }
};

struct UnpackInt4 {
  template <typename W>
  static MGEMV_INLINE void run(int8_t* unpacked, const uint8_t* packed, size_t first, size_t last) {
    typedef int8_t bytes16 __attribute__((vector_size(16), aligned(1), may_alias));
    size_t i = first;
    for (; i + 16 <= last; i += 16) {
      const bytes16 v = *reinterpret_cast<const bytes16*>(packed + i);
      const bytes16 lo = ((v & 0xf) ^ 8) - 8, hi = (((v >> 4) & 0xf) ^ 8) - 8;
      bytes16* const to = reinterpret_cast<bytes16*>(unpacked + 2 * i);
      to[0] = __builtin_shufflevector(lo, hi, 0, 16, 1, 17, 2, 18, 3, 19, 4, 20, 5, 21, 6, 22, 7, 23);
      to[1] = __builtin_shufflevector(lo, hi, 8, 24, 9, 25, 10, 26, 11, 27, 12, 28, 13, 29, 14, 30, 15, 31);
    }
    for (; i < last; ++i) {
      unpacked[2 * i] = (int8_t)(((packed[i] & 0xf) ^ 8) - 8);
      unpacked[2 * i + 1] = (int8_t)(((packed[i] >> 4) ^ 8) - 8);
    }
  }
};

// -z is an integer of magnitude <= 128: exact in binary16.  The binary32 product of two halves is exact, so one rounding to
// binary16 is the correctly rounded fp16 multiply.
struct FoldZeroPoints {
  template <typename W>
  static MGEMV_INLINE void run(uint16_t* out, const uint16_t* scales, const int8_t* zeros, size_t first, size_t last) {
    for (size_t i = first; i < last; i += 8) {
      const size_t here = last - i < 8 ? last - i : 8;
      u16x8 s = {}, r;
      i8x8 z = {};
      std::memcpy(&s, scales + i, here == 8 ? 16 : here * 2);
      std::memcpy(&z, zeros + i, here == 8 ? 8 : here);
      f32x8 f;
      half_bits_to_float(s, f);
      typedef int32_t i32x8 __attribute__((vector_size(32)));
      float_to_half_bits(__builtin_convertvector(-__builtin_convertvector(z, i32x8), f32x8) * f, r);
      std::memcpy(out + i, &r, here == 8 ? 16 : here * 2);
    }
  }
};

int check_dims(size_t n_out, size_t k, int bits) {
  if (n_out == 0 || k == 0) return MGEMV_ERR_SIZE;
  if (n_out % 4) return MGEMV_ERR_ROWS;                          // utils/preprocess.h:319-322
  if (k % 8) return MGEMV_ERR_COLS;                              // utils/preprocess.h:324-327
  if (n_out > 0x7fffffffull || k > 0x7fffffffull) return MGEMV_ERR_SIZE;
  return MGEMV_OK;
}

}  // namespace

extern "C" {

int mgemv_pack_int4(uint8_t* packed, const int8_t* unpacked, size_t n_unpacked) {
  if (n_unpacked == 0) return MGEMV_OK;
  if (packed == nullptr || unpacked == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (n_unpacked % 2) return MGEMV_ERR_SIZE;  // two elements per byte
  const bool in_order = share_memory(packed, n_unpacked / 2, unpacked, n_unpacked);
  in_pieces(n_unpacked / 2, kGrain, in_order, [=](size_t first, size_t last) { run_loop<PackInt4>(packed, unpacked, first, last); });
  return MGEMV_OK;
}

int mgemv_unpack_int4(int8_t* unpacked, const uint8_t* packed, size_t n_packed) {
  if (n_packed == 0) return MGEMV_OK;
  if (packed == nullptr || unpacked == nullptr) return MGEMV_ERR_NULL_POINTER;
  const bool in_order = share_memory(unpacked, 2 * n_packed, packed, n_packed);
  in_pieces(n_packed, kGrain, in_order, [=](size_t first, size_t last) { run_loop<UnpackInt4>(unpacked, packed, first, last); });
  return MGEMV_OK;
}

int mgemv_fold_zero_points(uint16_t* out, const uint16_t* scales, const int8_t* zeros, size_t n) {
  if (n == 0) return MGEMV_OK;
  if (out == nullptr || scales == nullptr || zeros == nullptr) return MGEMV_ERR_NULL_POINTER;
  const bool in_order = share_memory(out, 2 * n, scales, 2 * n) || share_memory(out, 2 * n, zeros, n);
  in_pieces(n, kGrain / 4, in_order, [=](size_t first, size_t last) { run_loop<FoldZeroPoints>(out, scales, zeros, first, last); });
  return MGEMV_OK;
}

int mgemv_fold_zero_points_bf16(uint16_t* out, const uint16_t* scales, const int8_t* zeros, size_t n) {
  if (n == 0) return MGEMV_OK;
  if (out == nullptr || scales == nullptr || zeros == nullptr) return MGEMV_ERR_NULL_POINTER;
  const bool in_order = share_memory(out, 2 * n, scales, 2 * n) || share_memory(out, 2 * n, zeros, n);
  in_pieces(n, kGrain / 4, in_order, [=](size_t first, size_t last) {
    for (size_t i = first; i < last; ++i) {
      // -z has at most 8 significant bits: exact in bfloat16.  The binary32 product of two
      // bfloat16 values is exact, so one rounding (nearest even) is the correctly rounded multiply.
      const uint32_t s_bits = (uint32_t)scales[i] << 16;
      float s;
      std::memcpy(&s, &s_bits, 4);
      const float prod = (float)(-(int)zeros[i]) * s;
      uint32_t bits;
      std::memcpy(&bits, &prod, 4);
      if ((bits & 0x7fffffffu) > 0x7f800000u) {
        out[i] = (uint16_t)((bits >> 16) | 0x0040u);  // NaN stays NaN
      } else {
        out[i] = (uint16_t)((bits + 0x7fffu + ((bits >> 16) & 1u)) >> 16);
      }
    }
  });
  return MGEMV_OK;
}

size_t mgemv_preprocessed_size(const size_t* shape, int rank, int quant_type) {
  size_t experts, k, n_out;
  const int bits = bits_of_quant_type(quant_type);
  if (bits == 0 || !shape_ok(shape, rank, experts, k, n_out)) return 0;
  return experts * mgemv::preprocessed_bytes(n_out, k, bits);
}

int mgemv_preprocess_weights(uint8_t* dst, const uint8_t* src, const size_t* shape, int rank, int layout,
                             int quant_type) {
  if (dst == nullptr || src == nullptr || shape == nullptr) return MGEMV_ERR_NULL_POINTER;
  size_t experts, k, n_out;
  if (!shape_ok(shape, rank, experts, k, n_out)) return MGEMV_ERR_RANK;
  const int bits = bits_of_quant_type(quant_type);
  if (bits == 0) return MGEMV_ERR_QUANT_TYPE;
  if (layout != MGEMV_ROW_MAJOR && layout != MGEMV_COLUMN_MAJOR) return MGEMV_ERR_LAYOUT;
  if (const int st = check_dims(n_out, k, bits)) return st;

  const size_t src_bytes = n_out * k * (size_t)bits / 8;
  const size_t dst_bytes = mgemv::preprocessed_bytes(n_out, k, bits);
  std::vector<uint8_t> transposed;
  if (layout == MGEMV_ROW_MAJOR) transposed.resize(src_bytes);
  for (size_t e = 0; e < experts; ++e) {
    const uint8_t* matrix = src + e * src_bytes;
    if (layout == MGEMV_ROW_MAJOR) {
      transpose_quantised(transposed.data(), matrix, k, n_out, bits);
      matrix = transposed.data();
    }
    tile_one_matrix(dst + e * dst_bytes, matrix, n_out, k, bits);
  }
  return MGEMV_OK;
}

int mgemv_unpreprocess_weights(uint8_t* dst, const uint8_t* src_preprocessed, const size_t* shape, int rank,
                               int quant_type) {
  if (dst == nullptr || src_preprocessed == nullptr || shape == nullptr) return MGEMV_ERR_NULL_POINTER;
  size_t experts, k, n_out;
  if (!shape_ok(shape, rank, experts, k, n_out)) return MGEMV_ERR_RANK;
  const int bits = bits_of_quant_type(quant_type);
  if (bits == 0) return MGEMV_ERR_QUANT_TYPE;
  if (const int st = check_dims(n_out, k, bits)) return st;
  const size_t raw_bytes = n_out * k * (size_t)bits / 8;
  const size_t tiled_bytes = mgemv::preprocessed_bytes(n_out, k, bits);
  for (size_t e = 0; e < experts; ++e)
    untile_one_matrix(dst + e * raw_bytes, src_preprocessed + e * tiled_bytes, n_out, k, bits);
  return MGEMV_OK;
}

const char* mgemv_status_string(int status) {
  switch (status) {
    case MGEMV_OK: return "ok";
    case MGEMV_ERR_NULL_POINTER: return "a required pointer is NULL";
    case MGEMV_ERR_RANK: return "weight shape must be 2-D {k, n_out} or 3-D {experts, k, n_out}";
    case MGEMV_ERR_ROWS: return "n_out must be a multiple of 4";
    case MGEMV_ERR_COLS: return "k must be a multiple of 8";
    case MGEMV_ERR_GROUP_SIZE: return "group_size must be >= 64, a multiple of 32 and divide k";
    case MGEMV_ERR_QUANT_OP: return "quant_op must be 1 (per-column scale), 2 (group scale) or 3 (group scale + zero)";
    case MGEMV_ERR_QUANT_TYPE: return "weights must be int8 (W8_A16) or int4 (W4_A16)";
    case MGEMV_ERR_BATCH: return "batch_count must be >= 1 and m_batch in [1, 16]";
    case MGEMV_ERR_LAYOUT: return "layout must be 0 (row major) or 1 (column major)";
    case MGEMV_ERR_LEADING_DIMENSION: return "a leading dimension or batch stride describes an operand this library does not take (only the reference's dense operands)";
    case MGEMV_ERR_ALLOCATION: return "device memory could not be allocated (host-pointer entry point)";
    case MGEMV_ERR_SCRATCH_SIZE: return "the problem does not fit the static scratch arrays of the allocation-free host-pointer entry point";
    case MGEMV_ERR_SIZE: return "a dimension is zero, negative or exceeds the 32-bit index range of the kernels";
    case MGEMV_ERR_LAUNCH: return "HIP launch failed";
    case MGEMV_ERR_NO_DEVICE: return "no usable gfx950 device";
    case MGEMV_ERR_ALIGNMENT: return "device pointer alignment: weights and activations 16 bytes, scales / zeros / bias / outputs 2 bytes, dequantised output 4 bytes";
    default: return "unknown status";
  }
}

int mgemv_version(void) { return 212; }  // 2xx: int4 fields at bits 7-10 / 3-6 of each half-word

}  // extern "C"
