// C-ABI entry points of the device side: argument checks, launch geometry, tuned plans, and the
// dequantise kernel.  The GEMV kernels live in gemv_dpp_kernel.h (VALU) and launch_mfma.hip
// (matrix cores).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "kernel_common.h"

namespace mgemv {

struct DequantParams {
  const uint8_t* weights;
  const half_t* scale;
  const half_t* zero_add;
  int n_out, k, group_size, num_groups, tiles, ksteps, flags;
};

// The scales (or zeros) of the 16 rows of a tile in one group: 32 neighbouring bytes of the table, row 2i in the low and
// row 2i + 1 in the high half of word i.  Rows past the table read as zero.
struct TileScales {
  uint32_t v[kTileRows / 2];
};
__device__ __forceinline__ TileScales load_tile_scales(__amdgpu_buffer_rsrc_t table, int byte_offset) {
  TileScales t;
#pragma unroll
  for (int i = 0; i < kTileRows / 2; i += 4) {
    const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(table, byte_offset + i * 4, 0, kCacheDefault);
    t.v[i] = q[0]; t.v[i + 1] = q[1]; t.v[i + 2] = q[2]; t.v[i + 3] = q[3];
  }
  return t;
}

// True when all 16 scales permit the short dequantiser (with shift 0), in every lane.
template <int BITS, int ACT>
__device__ __forceinline__ bool tile_scales_permit_short_form(const TileScales& s) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  constexpr uint16_t kFirst = ACT != kActBf16 ? kShortF16First : BITS == 4 ? kShortBf16Int4First : kShortBf16Int8First;
  constexpr uint16_t kPast = ACT != kActBf16 ? kShortF16Past : BITS == 4 ? kShortBf16Int4Past : kShortBf16Int8Past;
  u16x2 most = u16x2{0, 0};
#pragma unroll
  for (int i = 0; i < kTileRows / 2; ++i)
    most = __builtin_elementwise_max(most, (u16x2)(__builtin_bit_cast(u16x2, s.v[i]) - u16x2{kFirst, kFirst}));
  return __builtin_amdgcn_ballot_w64((most[0] > most[1] ? most[0] : most[1]) >= kPast - kFirst) == 0;
}

// Eight consecutive weights of one row (one word of int4, two of int8) to 16 bytes, with the converters of the GEMV kernels.
template <int BITS, int QOP, int ACT, bool SHORT>
__device__ __forceinline__ u32x4 dequantize_eight(const uint32_t (&w)[8 * BITS / 32], const ConvertRegs& c, uint32_t s_bits,
                                                  uint32_t z_bits) {
  constexpr bool kHasZero = QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS;
  u32x4 out;
  if constexpr (ACT == kActBf16) {
    const Bf16Scale bs = make_bf16_scale<BITS, SHORT>(s_bits, kHasZero ? z_bits : 0u, make_identity4(),
                                                      Int4ScaleBf16{bf16_low_to_f32(s_bits), kNoShift});
    uint32_t d[4];
    if constexpr (BITS == 4) dequant_int4_words_bf16<kHasZero, SHORT, 1>(w, c, bs, d);
    else dequant_int8_words_bf16<kHasZero, SHORT, 2>(w, bs, d);
    out = u32x4{d[0], d[1], d[2], d[3]};
  } else {
    const half2_t s2 = splat_low(s_bits), z2 = kHasZero ? splat_low(z_bits) : half2_t{};
    half2_t d[4];
    if constexpr (BITS == 4 && SHORT) {
      dequant_int4_word_short<kHasZero>(w[0], c, make_short_form_scale(s2), z2, d);
    } else {
      half2_t q[4];
      if constexpr (BITS == 4) {
        convert_int4_word(w[0], c, q);
      } else {
        half2_t q0[2], q1[2];
        convert_int8_word(w[0], c, q0);
        convert_int8_word(w[1], c, q1);
        q[0] = q0[0]; q[1] = q0[1]; q[2] = q1[0]; q[3] = q1[1];
      }
#pragma unroll
      for (int h = 0; h < 4; ++h) d[h] = dequant_pair<kHasZero>(q[h], s2, z2);
    }
    out = u32x4{as_u32(d[0]), as_u32(d[1]), as_u32(d[2]), as_u32(d[3])};
  }
  return out;
}

// One wave per unit; writes the dequantised weights of its 16 rows x kStepK columns with the same converters, and the
// same wave-uniform choice between them, as the GEMV kernels.
// Bound by its stores (four bytes out for one byte of int4 in), so the lanes are dealt out along the OUTPUT: a store
// instruction of the wave writes one whole row of the unit (int4: 64 lanes x 16 bytes = 512 k) or two (int8), contiguous,
// and each lane picks the one or two weight words it needs for that out of the 16-byte chunks of the tile layout (the four
// or eight lanes of a chunk share its cache line, and the 16 rows of a unit read each of its lines 8 times out of the L1).
// With a lane per row, as the GEMV kernels have it, every store instruction scatters 64 pieces of 4 bytes.
constexpr int kDequantWaves = 4;
template <int BITS, int QOP, int ACT>
__global__ void __launch_bounds__(kWave * kDequantWaves) dequantize_kernel(const DequantParams p, half_t* __restrict__ out) {
  using G = Geometry<BITS>;
  constexpr int kWords = 8 * BITS / 32;                // weight words of eight weights: 1 | 2
  constexpr int kLanesPerRow = G::kStepK / 8;          // 64 | 32
  constexpr int kRowsPerStore = kWave / kLanesPerRow;  // 1 | 2
  typedef u32x4 __attribute__((aligned(4))) u32x4_any;  // the caller's rows are 4-byte aligned
  const int lane = threadIdx.x % kWave;
  const long long unit = (long long)blockIdx.x * kDequantWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (unit >= (long long)p.tiles * p.ksteps) return;  // whole waves only
  const int tile = (int)(unit / p.ksteps), kstep = (int)(unit % p.ksteps);
  const int piece = lane % kLanesPerRow, sub_row = lane / kLanesPerRow;  // eight weights of a row; which row of the store
  const int k0 = kstep * G::kStepK + piece * 8;
  const int row0 = tile * kTileRows;

  const int slice = piece * 8 / G::kRunK, block = piece * 8 % G::kRunK / G::kChunkK, word = piece % (G::kChunkK / 8) * kWords;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(p.weights + (size_t)unit * kUnitBytes, kUnitBytes);
  const int w_offset = block * kBlockBytes + (slice * kTileRows + sub_row) * kChunkBytes + word * 4;
  uint32_t w[kTileRows / kRowsPerStore][kWords];
#pragma unroll
  for (int i = 0; i < kTileRows / kRowsPerStore; ++i) {
    const int off = w_offset + i * kRowsPerStore * kChunkBytes;
    if constexpr (BITS == 4) {
      w[i][0] = __builtin_amdgcn_raw_buffer_load_b32(w_rsrc, off, 0, kCacheDefault);
    } else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, off, 0, kCacheDefault);
      w[i][0] = v[0]; w[i][1] = v[1];
    }
  }
  int group = 0;
  if constexpr (QOP != MGEMV_PER_COLUMN_SCALE_ONLY) {
    Problem geo{};
    geo.k = p.k;
    geo.group_size = p.group_size;
    group = group_of<4>(geo, k0);
  }
  const int table_offset = (group * p.n_out + row0) * 2;
  const uint32_t table_bytes = (uint32_t)p.num_groups * (uint32_t)p.n_out * 2u;
  const TileScales s = load_tile_scales(make_rsrc(p.scale, table_bytes), table_offset);
  TileScales z{};
  if constexpr (QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS) z = load_tile_scales(make_rsrc(p.zero_add, table_bytes), table_offset);

  const ConvertRegs c = make_convert_regs();
  half_t* const dst = out + (size_t)(row0 + sub_row) * (size_t)p.k + k0;
  const bool inside = k0 < p.k;  // k is a multiple of 8
  auto write_rows = [&](auto short_form) {
    constexpr bool kShort = decltype(short_form)::value;
#pragma unroll
    for (int i = 0; i < kTileRows / kRowsPerStore; ++i) {
      const int row = i * kRowsPerStore + sub_row;
      const int shift = kRowsPerStore == 1 ? 16 * (i & 1) : 16 * sub_row;
      const int entry = kRowsPerStore == 1 ? i / 2 : i;
      const u32x4 d = dequantize_eight<BITS, QOP, ACT, kShort>(w[i], c, (s.v[entry] >> shift) & 0xffffu, (z.v[entry] >> shift) & 0xffffu);
      if (inside && row0 + row < p.n_out)
        __builtin_nontemporal_store(d, reinterpret_cast<u32x4_any*>(dst + (size_t)(i * kRowsPerStore) * (size_t)p.k));
    }
  };
  // rows past n_out read the next group's scales or zeros: they may only cost the short form
  if ((BITS == 4 || ACT == kActBf16) && (p.flags & kExactIntegerFormOnly) == 0 && tile_scales_permit_short_form<BITS, ACT>(s))
    write_rows(std::true_type{});
  else
    write_rows(std::false_type{});
}

// ---------------------------------------------------------------------------------------------
// Host side: argument checks, launch geometry, dispatch
// ---------------------------------------------------------------------------------------------

std::atomic<int> g_override_split_k{0};
std::atomic<int> g_override_tiles_per_wg{0};
std::atomic<int> g_override_tiles_per_wave{0};
std::atomic<int> g_override_workgroups{0};
std::atomic<int> g_matrix_core_min_batch{0};  // m_batch from which the matrix-core kernels are used; 0 = built-in rule
std::atomic<int> g_dequant_flags{0};          // kExactIntegerFormOnly or 0
std::atomic<int> g_override_stages{0};        // 0 = built-in (2), 1 or 2
std::atomic<int> g_matrix_core_variant{MGEMV_MATRIX_CORE_AUTO};

// What steers plan_launch besides the shape: zeros mean "built-in rule".
struct PlanKnobs {
  int split_k = 0, tiles_per_wg = 0, tiles_per_wave = 0, workgroups = 0;
  int parts = 0;            // part-tile kernels: workgroups per tile
  bool split_left_over = false;  // k-stationary kernel: tiles that do not divide over the workgroups go to two or four of them
  int matrix_core_min_batch = 0;
  int matrix_core_variant = MGEMV_MATRIX_CORE_AUTO;
  bool wide_waves = false;  // the kernel is one of those compiled for at most 8 waves per workgroup
  int stages = 0;           // VALU kernel: 0 = built-in rule (2: the next unit in flight while one is computed), 1, 2
  int num_cus = kNumCus;    // compute units of the device the launch goes to (256 on an unpartitioned MI355X)
  bool generic_groups = false;  // the group size does not divide the k step: one scale / zero lookup per block of a unit
};

// Tuned plans by problem: (n_out, k, weight bits, group size or 0 for any, m_batch) -> knobs.
using PlanKey = std::tuple<int, int, int, int, int, int>;  // n_out, k, bits, group size, rows, element
std::mutex g_tuned_mutex;
std::map<PlanKey, PlanKnobs> g_tuned_plans;
std::atomic<int> g_tuned_count{0};  // lets the launch path skip the lock while the table is empty

// Built-in table: plans measured on an unpartitioned MI355X that the rules below do not produce,
// kept as data (mixed_gemv_amd/default_plans.json, compiled in by the build) instead of as one
// more shape threshold in plan_launch.  Consulted after the caller's table, for launches on a
// device of kDefaultPlanCus compute units only.
const mgemv_tuned_plan kDefaultPlans[] = {
#include "default_plans.inc"
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}  // terminator (n_out = 0)
};
constexpr int kDefaultPlanCus = 256;
std::atomic<int> g_default_plans_enabled{1};

int default_plan_count() {
  int n = 0;
  while (kDefaultPlans[n].n_out != 0) ++n;
  return n;
}

PlanKnobs knobs_of_plan(const mgemv_tuned_plan& plan) {
  PlanKnobs kn;
  kn.split_k = plan.split_k_waves;
  kn.tiles_per_wg = plan.tiles_per_workgroup;
  kn.tiles_per_wave = plan.tiles_per_wave;
  kn.workgroups = plan.max_workgroups;
  kn.stages = plan.stages;
  switch (plan.kernel) {
    case MGEMV_KERNEL_VALU: kn.matrix_core_min_batch = MGEMV_MAX_M_BATCH + 1; break;
    case MGEMV_KERNEL_MATRIX_CORE_REGISTER_OPERAND:
      kn.matrix_core_min_batch = 1;
      kn.matrix_core_variant = MGEMV_MATRIX_CORE_REGISTER_OPERAND;
      break;
    case MGEMV_KERNEL_MATRIX_CORE_LDS_STAGED:
      kn.matrix_core_min_batch = 1;
      kn.matrix_core_variant = MGEMV_MATRIX_CORE_LDS_STAGED;
      break;
    case MGEMV_KERNEL_MATRIX_CORE_K_STATIONARY:
      kn.matrix_core_min_batch = 1;
      kn.matrix_core_variant = MGEMV_MATRIX_CORE_K_STATIONARY;
      break;
    default: break;
  }
  return kn;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Tile sequences of a four-wave workgroup (4, 2 or 1, the waves left over splitting k) with which one workgroup per compute
// unit takes the tiles in walks of up to longest_walk that are even to 3 %; 0: none.
inline int even_fit(int tiles, int ksteps, int longest_walk, int cus) {
  for (int tw = 4; tw >= 1; tw /= 2) {
    const int sequences = cus * tw, walk = ceil_div(tiles, sequences);
    if (walk > longest_walk) continue;
    // The k steps must divide evenly over the 4 / tw waves of a sequence as well, or a SIMD of every compute
    // unit idles (6 k steps on 4 waves are 2 + 2 + 2 + 0): against one workgroup per tile with a wave per k step,
    // 12288x3072 7.09 us / 5.68, 20480x3072 10.10 / 8.79, 28672x3072 12.95 / 11.05, 12288x2560 7.13 / 5.24,
    // 12288x3584 7.18 / 6.24, 12288x5120 9.39 / 8.58; with four k steps or fewer that launch is ahead on every
    // even fit (12288x2048 5.10 / 4.52; 20480x2048 6.78 / 5.93; 28672x2048 8.32 / 7.64; 16384x2048 5.42 / 5.23).
    if (ksteps % (4 / tw) != 0) continue;
    // ... and with up to 8 k steps a single tile sequence of four k-split waves (two units a wave, then the next
    // tile) is behind a workgroup of one-unit waves per tile: 12288x4096 6.6 us / 7.3; 20480x4096 9.8 / 10.4; 20048x3840
    // 10.0 / 11.0; 28672x4096 level (two or four sequences side by side stay: 16384x4096 8.0 / 9.0; 24576x3072 9.5 / 10.1)
    if (ksteps <= 8 && tw == 1) continue;
    if ((long long)walk * sequences * 100 <= (long long)tiles * 103) return tw;
  }
  return 0;
}

// 1 or 2: the group size divides the k step ("regular" scale addressing, one or two groups per
// lane run); 4: any other legal group size ("generic", one lookup per block).
int groups_per_run(int group_size, int bits) {
  const int run = run_k(bits);
  if (step_k(bits) % group_size != 0) return 4;
  return group_size % run == 0 ? 1 : 2;
}

// Scale / zero lookups per lane run of a launch: groups_per_run, one for a group as long as k (per-column mode) or none given.
inline int lookups_per_run(int k, int group_size, int bits) {
  return group_size > 0 && group_size != k ? groups_per_run(group_size, bits) : 1;
}

// Waves per tile, each workgroup one tile, of a single row on more tiles than compute units; 0: as the rules of plan_launch
// have it.  Those rules are older than the builds of the VALU kernel without a loop (waves of one or two units), of which more
// are in flight at once and which request all they need up front: most launches that used to want longer waves -- walks of
// several tiles, whole-k waves, two tiles per workgroup -- now want two units a wave.  Part of the built-in measured
// plans, so for the device these were measured on only.
// fp16, int4; us of the rules / here, both through the builds there are now; "of the time" is here over the rules, on launches
// of random shapes:
//   9-16 k steps, more than 512 tiles: two units.  50408x4480 g64 28.2 / 24.2, 14108x8064 g96 16.3 / 13.7, 37912x4608 g96 24.3 / 22.1,
//     68696x7168 56.6 / 52.5; 0.924 of the time (0.69-1.05) on 1500 launches of more than 1024 tiles, 0.970 (0.79-1.11) on 470 of
//     513-1024.
//   9-16 k steps, up to 512 tiles: one unit.  7312x5568 g96 8.27 / 7.07, 4172x6400 g64 7.57 / 6.85, 6908x5888 per column 6.56 / 6.12;
//     0.933 (0.77-1.06) on 660.
//   5-7 k steps: one unit up to 5.5 (7 k steps), 8 (5) or 12 (6) tiles per compute unit, then two.  79772x2560 g64 26.4 / 22.6, 74732x2304
//     scale only 19.1 / 17.8; 0.927 (0.68-1.07) on 1170.  8 k steps: two from 5.5 on; 51248x4032 g96 27.3 / 22.5, 82844x3840 35.0 / 30.7,
//     0.891 on 240 launches of more than 2048 tiles, but 1.04 (0.94-1.13) on 70 of 1409-2048, where one unit is still ahead.
//   17-32 k steps, up to 768 tiles: two units (8656x12800 g64 15.3 / 13.6, 10092x12160 14.4 / 13.2; 0.927 on 430); more than 1024: four
//     waves (26560x14208 g96 45.7 / 40.0, 36336x12288 42.9 / 39.5; 0.935, 0.72-1.07, on 650).  33 and more: four waves either way; up to
//     768 tiles they are what the rules take, but for the last few tile counts (0.976-1.007 on 60), above 1024 0.90 on 50.
//   With the rules stay, as measured: lookups per block on up to 640 tiles (8400x5280 g96 8.67 / 8.97), two lookups per run where a
//     wave per tile fills the SIMDs (16384x6144 g64 scale only 9.85 / 10.3), even fits with 5-8 k steps (24576x4096 11.6 / 11.8) and
//     769-1024 tiles with 17 and more (0.89-1.045).
//   With the rules stay because a launch test holds one shape of each to its older plan, not because it is faster; two units /
//     the plan that stays: 16 k steps on 513-640 tiles 0.80-0.92 of the time, mean 0.86, on 60 (9216x8192); 9 and 10 k steps on 769-1024
//     tiles 0.88-1.03, mean 0.98 (13824x5120); 9-12 on even fits of 1025-2048 (28672x6144 17.8 us / 17.4).  One unit / the plan
//     that stays: 10 k steps up to 512 tiles 0.90-1.04, mean 0.99, with two lookups per run 1.02 (5120x5120); 14-16 on evenly filled 512
//     tiles 0.93-1.04, mean 0.99, two lookups per run 1.03, lookups per block 0.91 (8192x8192).
// fp16, int8, more than 4 tiles per compute unit: one unit a wave at 10-12 k steps (49568x2816 25.6 / 23.4, 71644x3072 37.7 / 35.2,
//   19712x2560 per column 10.2 / 9.7; 0.95, 0.85-1.03, on 360); more than 8: at 5-9 and 13 as well (72220x1632 g96 24.6 / 22.1, 37952x2176
//   16.7 / 15.6; 0.94 on 790); with 14 it loses (20480x3584 12.9 / 13.8).
// bf16 with a lookup per block, 9-16 k steps on 1.125 to 2 tiles per compute unit: up to eight waves instead of pairs of tiles
//   (5052x4320 g96 9.65 / 8.39, 7936x7680 11.3 / 9.5, int8 5784x2304 7.6 / 6.05; 0.79-1.06 on 400); other group sizes gain and lose.
// A lookup per block, half a tile to one tile per compute unit, 9-16 k steps, both types: eight waves of one or two units instead of four of
//   three and four: both are requested at once, and nine k steps on four waves are 3 + 3 + 3 and a SIMD idle.  int4 0.92 of the time
//   (0.74-1.04) on 185 (4096x8064 g96 6.37 / 6.16, in bf16 8.25 / 7.79), int8 0.86 (0.75-0.94) on 63 (3072x3072 g96 4.65 / 4.37); two to
//   six problems 0.87-0.98, eight 0.93, but bf16 int4 1.03, up to 1.15.  Longer reductions take 0.85-0.96 alone and 1.05-1.2 in batched launches, with one or two lookups 0.9-1.2.
// bf16, 1.5 to 2 tiles per compute unit and longer reductions: four waves per tile instead of pairs of tiles with two each, which leave a wave
//   alone on every SIMD they have and some without one.  A lookup per block, from 18 k steps (17, as fast, is held by a launch test): 0.88 of the time (0.81-0.96) on 70 (8192x23040 g96
//   33.2 / 30.4, int8 8192x16224 g96 33.9 / 28.8); int4 otherwise, from 25: 0.92 (0.74-1.03) on 130 (8192x27904 32.8 / 31.0, 8192x21248
//   26.0 / 24.6; with 17-24 k steps 0.96, up to 1.03, left).  int8 otherwise 1.0-1.1, up to 1.5 tiles 1.03-1.3.
inline int single_row_split(int tiles, int ksteps, int bits, int cus, bool bf16, int lookups) {
  const bool generic_groups = lookups == 4;
  if (generic_groups && tiles * 2 > cus && tiles <= cus && ksteps >= 9 && ksteps <= 16) return 8;
  if (tiles <= cus || ksteps < 5) return 0;
  const bool fills_simds = tiles <= 4 * cus && tiles * 103 >= cus * 400;  // with a wave per tile
  if (bf16) {
    const bool two_per_cu = tiles * 8 >= cus * 9 && tiles <= 2 * cus && ksteps >= 9 && ksteps <= 16;
    if (two_per_cu && generic_groups) return kMaxWavesPerWideWorkgroup;
    return tiles * 2 > cus * 3 && tiles <= 2 * cus && ksteps >= (generic_groups ? 18 : 25) && (generic_groups || bits == 4) ? 4 : 0;
  }
  const int two_units = ceil_div(ksteps, 2);
  if (bits == 8) {
    if (ksteps <= 8 && tiles <= 8 * cus) return 0;
    if (ksteps >= 10 && ksteps <= 12) return tiles > 4 * cus ? ksteps : 0;
    return ksteps <= 13 && tiles > 8 * cus ? ksteps : 0;
  }
  if (ksteps <= 8) {
    if (tiles <= 8 * cus && even_fit(tiles, ksteps, 7, cus) != 0) return 0;
    return tiles * 2 > cus * (ksteps == 5 ? 16 : ksteps == 6 ? 24 : 11) ? two_units : 0;
  }
  if (ksteps <= 16) {
    if (tiles <= 2 * cus) return (ksteps == 10 && !generic_groups) || (ksteps >= 14 && tiles * 103 >= cus * 200) ? 0 : ksteps;
    if ((ksteps == 16 || generic_groups) && tiles * 2 <= 5 * cus) return 0;
    if ((ksteps <= 10 && tiles > 3 * cus && tiles <= 4 * cus) || (fills_simds && lookups == 2)) return 0;
    return ksteps <= 12 && tiles > 4 * cus && tiles <= 8 * cus && even_fit(tiles, ksteps, 7, cus) != 0 ? 0 : two_units;
  }
  if (tiles <= 2 * cus || (tiles > 3 * cus && tiles <= 4 * cus)) return 0;
  return tiles <= 3 * cus && ksteps <= 32 ? two_units : 4;
}

// A single row on few tiles: workgroups per tile on the VALU kernel for parts of tiles (launch_valu_parts.hip); 0: not on that
// kernel.  Of the time of the kernel for whole tiles, 700 launches of random shapes, geometric means (worst):
//   at most a quarter as many tiles as compute units, four parts: fp16 int4 9-16 k steps 0.79 (0.97), 17-32 0.69 (0.82), more 0.60; int8
//     0.84 (0.86), 0.83 (0.86), 0.65; bf16 int4 5-8 0.73 (0.91), 9-16 0.63 (0.70), 17-32 0.60 (0.69), more 0.44; int8 17-32 0.73 (0.78), more
//     0.53 (512x5120 3.9 us / 3.1, 1024x16384 7.3 / 5.0; 900x4608 per column bf16 5.5 / 3.3, 1024x16320 g96 bf16 12.6 / 7.5);
//   at most half as many, two parts: from 17 k steps fp16 int4 0.79 (0.88), int8 0.85, bf16 int8 0.84 (0.88); bf16 int4 from 5 0.60-0.81
//     (0.97) (2048x8192 bf16 6.1 / 4.8, 2048x16384 7.7 / 5.8, 2000x12288 int8 7.3 / 6.2).  fp16 with 9-16 k steps is level (0.97-1.1), more
//     tiles take 1.1-1.8 times as long.
// Shorter reductions gain and lose; bf16 int8 with 9-16 k steps (0.8) loses up to 1.07 in batched launches (plan_of_batch).
// Launch tests hold two shapes of int4 on exactly a quarter as many tiles to their older plans, 16 k steps to its threads and 20, in
// fp16, to its bits: fp16 keeps the plan between them (1024x8192 4.5 us, four parts 3.6), bf16 takes two parts with 16 (5.9 / 4.2,
// four 4.05).
// kMaxValuPartsKSteps: as many as were measured; the sums of every unit lie in the LDS.
constexpr int kMaxValuPartsKSteps = 128;
inline int single_row_parts(int tiles, int ksteps, int bits, bool bf16, int cus) {
  if (ksteps > kMaxValuPartsKSteps) return 0;
  const int from = !bf16 ? 9 : bits == 8 ? 17 : 5;
  if (tiles * 4 == cus && bits == 4 && ksteps >= 16 && ksteps <= 20) {
    if (!bf16) return 0;
    if (ksteps == 16) return 2;
  }
  if (tiles * 4 <= cus) return ksteps >= from ? 4 : 0;
  return tiles * 2 <= cus && ksteps >= (bf16 ? from : 17) ? 2 : 0;
}

// Tiles per workgroup of the LDS-staged matrix-core kernel (= waves that share one activation stage): as few as
// bring the launch down to one workgroup per compute unit or fewer, at most 8 and at most a quarter of the staged
// rows.  Measured, 16 rows: 4096x4096 (256 tiles) 6.3 us at 1 tile against 7.2 at 2; 8192x8192 (512)
// 13.4 at 2 against 17.8 at 4; 11008x4096 (688) 10.1 at 4 against 11.3 at 2 and 14.2 at 8;
// 28672x8192 (1792) 28.3 at 8 against 30.6 at 4 and 32.8 at 2.  8 rows: 4096x4096 5.4 at 1
// against 6.4 at 2; 5120x5120 (320) 7.7 at 2 against 9.3 at 1; 10240x8192 (640) 14.7 at 4
// against 15.5 at 2; 11008x4096 9.0 at 4 against 9.7 at 2; 28672x8192 27.6 at 4 against 29.5 at 2.
// Still more workgroups than compute units: a count just above a multiple of 256 leaves most
// of the last round idle, and halving the tiles per workgroup evens that out (18944x3584,
// 8 rows: 296 workgroups of 4 tiles 12.8 us, 592 of 2 tiles 11.8; 22016x4096: 14.4 / 13.3):
// the largest count whose last round is at least three quarters full.
inline int lds_staged_tiles_per_wg(int tiles, int staged_rows, int cus) {
  int tw = 1;
  while (ceil_div(tiles, tw) > cus && tw * 2 <= 8 && tw * 4 <= staged_rows) tw *= 2;
  if (ceil_div(tiles, tw) > cus) {
    for (int t = tw; t >= 1; t /= 2) {
      const int wgs = ceil_div(tiles, t);
      if (wgs * 4 >= ceil_div(wgs, cus) * cus * 3) return t;
    }
  }
  return tw;
}

// Two fp16 rows, int8, more than 8 tiles per compute unit and 5-14 k steps: up to eight waves of one or two units instead of
// whole-k waves or walks (us of the rules / here: 57592x1728 g96 scale only 21.0 / 18.7, 131144x1792 g64 42.3 / 39.1, 75760x1280
// 19.5 / 18.3; 0.74-1.06 of the time on 540 launches, mean 0.93).  Fewer tiles and longer reductions gain and lose.
inline int two_int8_rows_split(int tiles, int ksteps, int cus) {
  return tiles > 8 * cus && ksteps >= 5 && ksteps <= 14 ? (ksteps < 8 ? ksteps : 8) : 0;
}

// Two and more rows, int4, in the same manner: launches that belong to another kernel, or to the same one in more workgroups,
// than the rules have it.  Times are us, the rules' / here, or here as a part of theirs.
//   fp16, 9-16 rows, a group size that divides the k step: the k-stationary kernel, since its rows 8-15 are requested with the
//     first eight --
//       at most one tile per compute unit, 64 tiles and more, 5-14 k steps (15 up to 14 rows): 0.73-1.06 on 2370 launches, mean
//         0.89 (1776x3456 g64 at 13 rows 6.16 / 5.04, 2760x6400 at 14 8.97 / 7.72); 15 k steps 0.96 on 117, at 16 rows 1.01-1.06;
//         16 k steps 0.87-1.05, mean 0.98, left with the rules;
//       two tiles per compute unit at 13-16 rows (from 1.25, which the LDS-staged kernel's pairs of tiles fill as well), 5-16
//         k steps: 0.80-1.03 on 451, mean 0.91 (5224x3072 at 13 rows 7.15 / 5.90, 6536x3968 per column 7.42 / 6.51, 8192x8192 g64 with a
//         bias at 16 13.1 / 12.5).  12 k steps (0.88-1.05, mean 0.97) and 8 on 512 tiles (0.84-0.93, mean 0.90) keep the rules' plan
//         because a launch test holds one shape of each to it.
//   bf16, 2 rows:
//     3 k steps, walks of 20 and more: k-stationary, four workgroups per compute unit (93308x1408 scale only 23.7 / 17.6; the VALU
//       kernel before; 0.85 on 23), and 4 k steps, walks of 12 and more: two (84860x1792 g64 35.3 / 25.7, 104424x2048 per column 29.6 /
//       23.9; 0.84, 0.65-1.07, on 80); shorter walks gain and lose;
//     5-16 k steps, walks of 7 and more: the LDS-staged kernel with workgroups of 4 tiles where the busiest SIMD would
//       have 1.15 times as many units on the k-stationary one (as in use_k_stationary_bf16): 58536x2560 g64 32.9 / 24.5, 29560x4608
//       24.8 / 21.8; 0.64-1.02 on 420 launches, mean 0.84.  A lookup per block moves that line, since the LDS-staged kernel does
//       more of them: 1.25 on walks of 7 and 8, 1.16 on longer ones (1.15 on all of them took 24992x3072 g96 scale only from 13.6 to 14.8,
//       25152x4608 18.4 / 19.6, 57600x6624 47.2 / 52.3; the launches between the lines took 1.05 times as long);
//   bf16, 8 k steps, walks of 31 to 40 (two rows: 27 to 48): the k-stationary kernel in two, three or four workgroups per compute unit
//     at 2 / 3 / 4 rows, which share the LDS that the partial sums of one long walk would take whole.  With 2 and 3 rows it is the rules'
//     kernel too, in one workgroup; with 4 the rules take the LDS-staged one, since 33 KB of rows and 31 or more tiles' sums, reckoned
//     in blocks of 17 entries, are over 160 KB.  (Blocks of the 9 entries that 8 waves write would fit; the rule does not know.)  0.94-0.99 /
//     0.95-1.014 / 0.96-1.004 of the time on 11, 9 and 8 launches, 0.86-1.02 on 90 more (128256x4096 64.5 / 61.6, 65.0 / 61.5, 64.4 / 62.7);
//     shorter walks gain and lose 3 %.
void set_multi_row_ranges(PlanKnobs& kn, int m_batch, int tiles, int ksteps, int cus, bool bf16, bool generic_groups) {
  const int walk = ceil_div(tiles, cus);
  auto choose = [&](int variant, int workgroups) {
    kn.matrix_core_min_batch = 1;
    kn.matrix_core_variant = variant;
    kn.workgroups = workgroups;
  };
  if (!bf16) {
    if (m_batch < 9 || generic_groups || ksteps < 5) return;
    const bool one_tile = walk == 1 && tiles * 4 >= cus && (ksteps <= 14 || (ksteps == 15 && m_batch <= 14));
    const bool two_tiles = walk == 2 && m_batch >= 13 && tiles * 4 > cus * 5 && ksteps <= 16 && ksteps != 12 &&
                           !(ksteps == 8 && tiles == 2 * cus);
    if (one_tile || two_tiles) choose(MGEMV_MATRIX_CORE_K_STATIONARY, 0);
    return;
  }
  if (ksteps == 8 && m_batch <= 4 && (m_batch == 2 ? walk >= 27 && walk <= 48 : walk >= 31 && walk <= 40)) {
    choose(MGEMV_MATRIX_CORE_K_STATIONARY, m_batch * cus);
  } else if (m_batch == 2 && ksteps <= 4) {
    if (ksteps == 3 && walk >= 20) choose(MGEMV_MATRIX_CORE_K_STATIONARY, 4 * cus);
    if (ksteps == 4 && walk >= 12) choose(MGEMV_MATRIX_CORE_K_STATIONARY, 2 * cus);
  } else if (m_batch == 2 && ksteps <= 16 && walk >= 7) {
    const int tw = lds_staged_tiles_per_wg(tiles, 8, cus);
    const long long here = 4ll * walk * ceil_div(ksteps, 4), there = (long long)ceil_div(ceil_div(tiles, tw), cus) * tw * ksteps;
    const int ahead_from = !generic_groups ? 115 : walk <= 8 ? 125 : 116;
    if (tw == 4 && here * 100 >= there * ahead_from) choose(MGEMV_MATRIX_CORE_LDS_STAGED, 0);
  }
}

// Two and more rows: workgroups per tile on the part-tile matrix-core kernel (launch_mfma_parts.hip); 0: not on that kernel.
// Part of the built-in measured plans, as the ranges above.  Over 2500 launches of random shapes whose plan it changes
// (2 tiles and more, up to 32768 k) 0.76 of the time of what was there (0.32-1.035, 3 of them above 1.02).  Geometric means:
//   at most a quarter as many tiles as compute units, 2-4 rows: four parts -- fp16 0.73 at 2 rows, 0.68 at 3 and 4, bf16 0.61 and
//     0.59, int8 0.75-0.84 and 0.64-0.75 (964x12416 3 rows 8.7 us / 5.7; 616x13368 per column bf16 2 rows 12.3 / 5.2);
//   at most half as many: two parts -- 2-4 rows fp16 0.84 and 0.74, bf16 0.75 and 0.66, 5-8 rows 0.82 and 0.76, int8 0.75-0.86
//     (2048x11008 4 rows 8.4 / 6.1; 1924x28288 bf16 8 rows 20.9 / 15.1); four parts there, two workgroups per compute unit, 1.0-1.2;
//   at most as many: one part, four waves with a stage of their own, where the reduction is long, or as rows and bits say: 0.91-0.96
//     from 17 k steps (4096x14336 bf16 8 rows 12.8 / 11.9), 9-16 rows on few tiles 0.80-0.90, int8 0.83-0.91.  Two parts 1.1-1.5;
//   more, int4 from 17 k steps: bf16 at 2-4 rows up to 1.5 tiles per compute unit two parts 0.85, one part where the LDS-staged kernel's
//     pairs of tiles fill the machine badly, 2 to 3 tiles per compute unit 0.87 (bf16 4 to 5 as well, 0.92).  Elsewhere 0.95-1.4.
// Fewer than 5 k steps gain less, and launch tests hold such shapes to their older plans, as they hold: 3 and 4 rows of int8 on more than
// a quarter as many tiles up to 17 k steps (0.85-0.91 here), bf16 on exactly half as many up to 8 (0.80-0.88) and two bf16 rows on
// 112-127 (16 k steps) and 128 tiles.  (Several problems: plan_of_batch_rows.)  9-16 fp16 rows of up to 8 k steps on few tiles (0.94) keep the rules' plan for the same reason.
inline int part_tiles(int m_batch, int tiles, int ksteps, int bits, bool bf16, int cus) {
  if (m_batch < 2 || tiles < 2 || ksteps < (m_batch == 2 && bits == 8 ? 8 : 5)) return 0;
  if (tiles * 4 <= cus && m_batch <= 4) return 4;
  if (tiles * 2 <= cus && m_batch <= 8) {
    if (bits == 8 && m_batch <= 4 && ksteps <= 17) return 0;
    if (bf16 && m_batch == 2 && tiles * (ksteps > 16 ? 2 : 16) >= cus * (ksteps > 16 ? 1 : 7)) return 0;
    if (bf16 && tiles * 2 == cus && ksteps <= 8) return 0;
    return 2;
  }
  if (tiles <= cus) {
    if (m_batch == 2 || (bits == 8 && m_batch <= 4)) return 0;
    if (ksteps > 16) return 1;
    if (bits == 8) return !bf16 || tiles * 2 < cus ? 1 : 0;
    return m_batch >= 9 && (bf16 ? tiles * 2 < cus : tiles * 4 < cus && ksteps > 8) ? 1 : 0;
  }
  if (bits == 8 || ksteps <= 16) return 0;
  if (bf16 && m_batch <= 4 && tiles * 2 <= 3 * cus) return 2;
  if (m_batch >= 3 && m_batch <= (bf16 ? 8 : 4) && tiles > 2 * cus && tiles <= 3 * cus) return 1;
  return bf16 && m_batch >= 3 && m_batch <= 8 && tiles > 4 * cus && tiles <= 5 * cus ? 1 : 0;
}

// Process-wide overrides win over the tables (they are what a tuner sweeps); then the caller's
// entry for exactly this group size, then its entry for any group size, then the built-in table and
// the measured ranges, then the built-in rules.  whole_tiles: nothing in parts (the measurement builds, which have none).
PlanKnobs knobs_for(int n_out, int k, int bits, int group_size, int m_batch, int act, int num_cus, bool whole_tiles) {
  PlanKnobs kn;
  kn.split_k = g_override_split_k.load();
  kn.tiles_per_wg = g_override_tiles_per_wg.load();
  kn.tiles_per_wave = g_override_tiles_per_wave.load();
  kn.workgroups = g_override_workgroups.load();
  kn.matrix_core_min_batch = g_matrix_core_min_batch.load();
  kn.matrix_core_variant = g_matrix_core_variant.load();
  kn.stages = g_override_stages.load();
  const bool overridden = kn.split_k || kn.tiles_per_wg || kn.tiles_per_wave || kn.workgroups || kn.stages ||
                          kn.matrix_core_min_batch || kn.matrix_core_variant != MGEMV_MATRIX_CORE_AUTO;
  if (overridden) return kn;
  const int element = act == kActBf16 ? MGEMV_ELEMENT_BF16 : MGEMV_ELEMENT_F16;
  if (g_tuned_count.load() != 0) {
    std::lock_guard<std::mutex> lock(g_tuned_mutex);
    auto it = g_tuned_plans.find(PlanKey{n_out, k, bits, group_size, m_batch, element});
    if (it == g_tuned_plans.end() && group_size != 0) it = g_tuned_plans.find(PlanKey{n_out, k, bits, 0, m_batch, element});
    if (it != g_tuned_plans.end()) return it->second;
  }
  if (num_cus == kDefaultPlanCus && g_default_plans_enabled.load() != 0) {
    for (const mgemv_tuned_plan* p = kDefaultPlans; p->n_out != 0; ++p)
      if (p->n_out == n_out && p->k == k && p->weight_bits == bits && p->m_batch == m_batch && p->element == element &&
          (p->group_size == group_size || p->group_size == 0))
        return knobs_of_plan(*p);
    const int tiles = num_tiles(n_out), ksteps = num_ksteps(k, bits);
    const bool bf16 = act == kActBf16;
    const int lookups = lookups_per_run(k, group_size, bits);
    kn.split_left_over = !whole_tiles;
    if (m_batch == 1 || (m_batch == 2 && bits == 8 && !bf16)) {
      const int split = m_batch == 1 ? single_row_split(tiles, ksteps, bits, num_cus, bf16, lookups)
                                     : two_int8_rows_split(tiles, ksteps, num_cus);
      if (split != 0) {
        kn.split_k = split;
        kn.tiles_per_wg = 1;
      }
    }
    const bool in_parts = !whole_tiles && kn.split_k == 0;
    if (in_parts && m_batch == 1) kn.parts = single_row_parts(tiles, ksteps, bits, bf16, num_cus);
    if (const int parts = in_parts ? part_tiles(m_batch, tiles, ksteps, bits, bf16, num_cus) : 0) {
      kn.matrix_core_min_batch = 1;
      kn.matrix_core_variant = MGEMV_MATRIX_CORE_LDS_STAGED;
      kn.parts = parts;
    } else if (m_batch > 1 && bits == 4) {
      set_multi_row_ranges(kn, m_batch, tiles, ksteps, num_cus, bf16, lookups == 4);
    }
  }
  return kn;
}

// Which row counts go to the matrix cores.  From 5 rows the VALU kernel would need a second pass
// over the weights (4096x4096: 8.8 us against 5.5).  The VALU kernel pays per row, the matrix-core kernels
// (almost) not, but the VALU kernel is at its best with at most one workgroup per compute unit:
// measured over 21 shapes, 3 and 4 rows are faster on the matrix cores whenever there are more
// than 256 tiles (5120x4096, 3 rows: 6.45 us against 6.74; 14336x4096, 4 rows: 9.2 against 11.4;
// the one exception found, 11008x4096 at 3 rows, loses 5 %) and on the VALU kernel below that
// (4096x14336, 4 rows: 10.6 against 11.3); 2 rows only from about 1536 tiles (32000x4096: 15.1
// against 16.4; 28672x8192: 25.9 against 27.3; 10240x8192: 14.2 against 12.7 the other way), and
// with fewer than 8 k steps only when one-unit VALU waves would not fit the machine (50304x2048,
// 12576 units: 15.2 against 12.8 the other way; 151936x2048, 37984 units: 33.1 against 35.1).
// cus: compute units of the device; the tile and unit counts the rules were measured at (on 256
// compute units) scale with it.
inline bool use_matrix_cores(int m_batch, int tiles, int ksteps, int forced, bool bf16, int bits, int cus) {
  if (forced > 0) return m_batch >= forced;
  // int8 weights: twice the bytes per VALU instruction, so the VALU kernel holds out longer --
  // ahead at 2-4 rows on every shape measured (8192x8192, 3 rows: 13.0 us against 14.8; 4096x11008,
  // 4 rows: 10.4 against 11.5) except the largest (28672x8192, 3 rows: 41.4 against 39.7).
  if (bits == 8) return m_batch >= 5 || (m_batch >= 3 && tiles >= 6 * cus);
  const long long units = (long long)tiles * ksteps;
  // 4 rows on up to 256 tiles: the barrier-free one-tile matrix-core launch is ahead from 16 k steps
  // (4096x8192: 6.9 us against 7.4; 4096x14336: 9.7 against 10.7; 3584x18944: 12.3 against 13.8)
  // and level below (4096x4096: 5.07 against 5.00); 2 and 3 rows stay on the VALU kernel there.
  return m_batch >= 5 || (m_batch >= 3 && tiles > cus && units >= 8ll * cus) ||
         (m_batch >= 4 && tiles >= 2 && ksteps >= 16) ||  // also on few tiles: 1536x8960 7.4 / 8.2; 1024x14336 9.0 / 10.2; 512x16384 9.9 / 10.9
         (m_batch >= 2 && !bf16 && tiles >= 6 * cus && (ksteps >= 8 || units > 64ll * cus));  // bf16, 28672x8192, 2 rows: 40.6 us against 37.8
}


// Where the k-stationary matrix-core kernel (one wave per k step, one workgroup per compute unit walking
// ceil(tiles / cus) tiles) is ahead of the others; fp16, 4 to 16 k steps, 2 to 16 rows (int4 unless noted).  Its waves hold
// their activation operand in registers, so its loop has neither barriers nor LDS reads and costs the same at 1 to
// 8 rows; what it pays is a fixed start (operand through LDS, 0.8-1.6 us) and end (one barrier, one combine), and a
// tail: when the weight stream ends, every wave of a SIMD still has a unit to compute.  Measured against the
// built-in choice otherwise (us, k-stationary first):
//   up to 8 k steps (at most 2 waves per SIMD), 3-8 rows, more tiles than compute units (4-5 k steps: 1.5 times
//     as many; 2 rows: 8 k steps and 2.5 times as many): 4608x4096 4 rows 5.60 / 6.41; 5120x3072 5.52 / 6.82; 8192x4096 6.06 / 6.88;
//     10240x4096 7.25 / 8.77, 8 rows 7.66 / 8.89; 11008x4096 3 rows 7.29 / 8.80; 22016x4096 2 rows 11.43 / 12.77;
//     28672x4096 8 rows 13.92 / 15.50; 8192x2048 7 rows 4.75 / 5.17; 50304x2048 4 rows 13.98 / 15.61; 128256x4096
//     4 rows 46.3 / 50.2; but 4608x2048 4 rows 4.58 / 4.49, and with 1-2 k steps there are 1-2 waves per compute
//     unit (32768x1024 10.4 / 7.2);
//   9-16 k steps: wherever its one-workgroup-per-compute-unit walks fill the machine better than the LDS-staged
//     kernel's workgroups of 1-4 tiles do -- 9216x8192 4 rows 12.48 / 14.18; 10240x8192 12.65 / 14.14, 8 rows 13.37
//     / 14.49; 12288x8192 3 rows 12.94 / 14.42; 18432x8192 17.73 / 22.40; 20480x8192 18.23 / 22.61; 28672x8192 2 /
//     4 / 8 rows 22.3 / 22.5 / 23.4 against 24.7 / 24.9 / 26.2 -- and, where the two fill it alike: at 3-4 rows with
//     walks of up to 3 tiles or tiles that divide evenly (5120x5120 6.82 / 7.62; 8192x7168 8.79 / 10.03; 8192x8192
//     10.34 / 10.37; 16384x8192 14.79 / 15.36; but 13312x8192 14.99 / 14.63, 13824x5120 10.97 / 10.60), at 5-8 rows
//     only up to 12 k steps with walks of 2 (8192x6144 7.80 / 8.64; but 8192x8192 11.01 / 10.50, 16384x8192 16.42 /
//     15.95, 14336x8192 16.0 / 15.3), at 2 rows from walks of 3 (12288x8192 12.74 / 13.28; 8192x8192 9.93 / 9.05);
//   1 row: never by this rule -- the single-row path is the VALU kernel by design.  Forced (threshold 1, this
//     variant) it is ahead only with 9-16 k steps and even walks of 7 tiles or more: 28672x8192 22.2 / 22.5 (three
//     leases: 1.9, 1.8, 0.5 % ahead), 32768x8192 25.5 / 26.9, 57344x8192 40.0 / 43.9; below that the VALU kernel's
//     finer pipeline wins (16384x8192 14.9 / 13.1; 128256x4096, 8 waves, 47.8 / 45.7);
//   int8 weights (a k step is 256 long, the operand 32 registers): ahead on every shape tried at 3-8 rows, 16 waves
//     and walks of 2 included -- 8192x4096 3 / 8 rows 7.68 / 8.12, 8.18 / 9.02; 11008x4096 8 rows 10.02 / 11.76;
//     14336x2048 4 rows 7.49 / 8.58; 16384x4096 6 rows 12.87 / 14.34; 28672x4096 8 rows 20.69 / 21.57 -- so the
//     rule of up to 8 k steps serves 8-16 there (78 launches on 19 further shapes: median +7.9 %; with 4-6 k steps
//     it is 5-7 % behind);
//   9-16 rows: the operand takes two rounds through LDS and twice the registers' worth of L2 traffic per wave, and
//     the LDS-staged kernel shares a stage between up to 8 tiles there.  Ahead where that kernel's workgroups fill
//     the machine worse by a tenth or more -- 11008x4096 16 rows 8.99 / 9.92; 10240x4096 8.68 / 9.87; 17408x4096
//     12.59 / 14.40; 12288x8192 12 rows 15.04 / 16.31; 18432x8192 16 rows 20.56 / 25.39; 20480x8192 20.99 / 25.48;
//     28672x8192 12 / 16 rows 25.75 / 27.08, 26.32 / 27.73 -- except on long walks of 8-wave workgroups (28672x4096
//     12 rows 15.34 / 14.87; 22016x4096, walks of 6, 13.68 / 13.98 still ahead); level or behind where the two fill
//     it alike (8192x6144 16 rows 10.44 / 9.90; 14336x8192 18.1 / 17.0; 14336x4096 12 rows 10.18 / 10.16) or where
//     the partial sums of a walk do not fit the LDS and the workgroups double (32768x8192 35.1 / 30.0).
//   * group sizes that do not divide the k step (one scale / zero lookup per block: PlanKnobs::generic_groups) stay
//     with the other kernels, the caller sees to that: 11008x3072 g96 at 4 rows 10.98 / 9.61; 14336x4608 g96 16.0 /
//     13.95; 28672x8064 g96 36.45 / 33.08; 8192x6144 g192 12.34 / 10.83; 20480x5120 g160 19.9 / 19.9.
// (The LDS-staged figures here are from before its loop took whole pairs of steps, which brought it 0-20 %, most with one tile per
// workgroup.  Of 1033 fp16 launches of random shapes that these rules give to this kernel the LDS-staged one is now more than
// 3 % ahead on 49, of 677 bf16 ones on 8.)
inline bool use_k_stationary(int m_batch, int tiles, int ksteps, int bits, int cus) {
  if (m_batch == 1 || ksteps < 4) return false;  // a single row stays on the VALU kernel, whatever was measured (above)
  const int walk = ceil_div(tiles, cus);
  const long long slots = (long long)walk * cus;  // tiles the launch has room for
  if (m_batch > 8) {
    // 9-16 rows: only where it fills the machine better than the LDS-staged kernel's workgroups of up to 8 tiles,
    // the partial sums of a whole walk fit the LDS, and -- with up to 8 k steps, 2 waves per SIMD -- walks stay short
    const int tw16 = lds_staged_tiles_per_wg(tiles, 16, cus);
    const long long lds_slots16 = (long long)ceil_div(ceil_div(tiles, tw16), cus) * cus * tw16;
    const long long park = (long long)walk * kKSlices * m_batch * kKStationaryParkSlots * 16;
    // int8 weights: the operand is half as many registers and the stage half as long, and the kernel is ahead by
    // 4-37 % on all 52 launches tried at 10-16 rows with 4-16 k steps and more tiles than compute units, as long as
    // the partial sums of a walk fit the LDS (11008x4096 at 16 rows 10.74 us / 12.94; 18944x3584 14.80 / 19.09;
    // 9216x3072 at 12 rows 7.80 / 10.67; 22016x2048 10.98 / 12.17; 11008x1024 5.78 / 6.14; where the workgroups double
    // for the LDS it loses: 32000x4096 at 16 rows 25.66 / 24.19, 50304x2048 22.62 / 21.19)
    if (bits == 8) return tiles > cus && park <= kMaxKStationaryLds;
    // a tile count that leaves the LDS-staged kernel only pairs of tiles on a large matrix: ahead even where the partial
    // sums of a walk need twice the workgroups (36400x5376 at 12 / 16 rows 23.1 / 29.3 us against 33.5 / 35.0)
    if (tw16 <= 2 && tiles > 4 * cus) return true;
    // up to 12 rows on walks of 2: 5120x5120 7.86 / 8.89; 7792x6016 8.98 / 9.83; 6144x4096 6.95 / 7.32; 8192x8192 level
    if (m_batch <= 12 && walk == 2 && park <= kMaxKStationaryLds) return true;
    return lds_slots16 * 10 >= slots * 11 && park <= kMaxKStationaryLds && (ksteps > 8 || walk <= 6);
  }
  if (tiles <= cus) {
    // At most one tile per compute unit, so no walk: still ahead of the VALU kernel's chunks of rows and of the
    // LDS-staged kernel at 3-7 rows with 9-14 k steps (4096x4608 4 rows 5.38 / 6.53; 2048x5120 5.10 / 6.44; 3072x6144
    // 5.43 / 6.29; 4096x6656 6.39 / 7.19; 3584x7168 6.31 / 7.14; 6 rows 4-7 % -- but 4096x7680, 15 k steps, 6 rows 7.72 /
    // 6.92 and 4096x8192, 16 waves, 3 / 4 / 8 rows 7.44 / 6.70, 7.70 / 6.98, 8.38 / 7.21) and at 4-7 rows with 5-8
    // (2560x2560 4 rows 4.35 / 4.74; 4096x3072 4.70 / 4.94; 4096x4096 6 rows 4.85 / 5.13; 3 rows lose 4-7 %; 8 rows
    // level).  Measured from 128 tiles up, int4.
    if (bits == 8 || tiles * 2 < cus || m_batch > 7) return false;
    if (ksteps <= 8) return ksteps >= 5 && m_batch >= 4;
    return m_batch >= 3 && (ksteps <= 14 || (ksteps == 15 && m_batch <= 4));
  }
  // tile counts that leave the LDS-staged kernel without a tidy grouping (it falls back to a workgroup per tile, no
  // stage shared): 16880x5376 at 3 / 5 / 8 rows 12.6 / 12.9 / 14.0 us against 17.4 / 17.7 / 17.8; 17408x8192 17.2 / 17.6 /
  // 18.4 against 24.1 / 24.1 / 24.3; int8 17728x1792 at 6 rows 7.9 / 10.2
  const int tw = lds_staged_tiles_per_wg(tiles, 8, cus);
  if (tw == 1 && tiles > 2 * cus && m_batch >= 3) return true;
  if (bits == 8 && ksteps < 7) return false;  // 8192x1024 int8, 3 rows: 4.9 us against 4.6; 32768x1536: 10.9 / 10.3 (but 11264x1792, 7 k steps, 4 rows: 5.9 / 7.0)
  if (ksteps <= 8 || bits == 8) {
    // the VALU kernel's two rows are cheap (8192x4096 5.90 / 5.95; 6144x3072 5.46 / 5.19; 12288x2560, 5 k steps, 6.71 /
    // 5.57): from 6 k steps and 2.5 tiles per compute unit (10240x3584 7.01 / 7.27; 12288x3072 6.84 / 7.30; 18944x3584
    // 9.88 / 10.47; 22016x3072 10.17 / 11.44; 37888x3584 15.89 / 17.87; 50304x3072 18.79 / 20.75)
    if (m_batch == 2) return (bits == 8 ? ksteps == 8 : ksteps >= 6) && tiles * 2 >= cus * 5;
    // five waves on four SIMDs: one SIMD carries two of them through every tile, and on longer walks the LDS-staged
    // kernel is ahead (26208x2176 at 3 rows 10.1 us / 11.3; 30112x2176 10.3 / 12.1; 14240x2560 at 8 rows 7.3 / 7.8)
    if (ksteps == 5 && walk >= 4) return false;
    return ksteps <= 5 ? tiles * 2 >= cus * 3 : tiles > cus;
  }
  const long long lds_slots = (long long)ceil_div(ceil_div(tiles, tw), cus) * cus * tw;
  if (lds_slots * 10 >= slots * 11) return m_batch >= 3 || walk >= 3;  // fills the machine better by a tenth or more
  // two rows: from walks of 3 tiles, evenly filled or not (21024x7808, walks of 6 at 85 %, 19.1 us / 21.8; 22016x8192 20.1 /
  // 22.2; 30064x6144 19.2 / 20.5; 14336x8192 and 16336x5632 level; 13824x5120, whose whole-k VALU waves fit well, 10.9 / 10.55)
  if (m_batch == 2) return walk >= 3;
  // walks of 4 up to 5 rows and 15 k steps: 13584x5632 11.1-11.2 / 12.0; 15360x6144 11.6-11.7 / 12.4-12.5; 12480x7424
  // 13.6-14.1 / 14.7; 16384x6144 at 5 rows 12.0 / 12.8 (13824x5120 10.9 / 10.7; with 16 k steps 13312x8192 15.1 / 14.7)
  if (m_batch <= 5 && walk == 4 && ksteps <= 15) return true;
  // ... and up to 8 rows with 9-11 k steps (12480x5632 at 6 rows 10.8 / 11.9; 13584x5632 at 8 rows 11.4 / 12.2; with 12-16
  // k steps 6-8 rows lose 3-5 %: 15360x6144, 14336x8192)
  if (walk == 4 && ksteps <= 11) return true;
  if (m_batch <= 4) return walk == 2 || walk == 3 || walk >= 5 || slots == tiles;  // (walks of 5 and more: 22944x7680 at 4 rows 19.7 / 22.4)
  // 5-8 rows: walks of 2 up to 12 k steps, and walks of 5 or more (22144x7936 at 6 rows 20.9 us / 23.8; 20672x8064 at 8
  // rows 20.3 / 23.1; 23104x7680 at 5 rows 20.8 / 23.1; 29024x5760 19.3 / 21.2); walks of 4 lose 3-5 % at 6-8 rows
  return (walk == 2 && ksteps <= 12) || walk >= 5;
}

// The bf16 build of the k-stationary kernel (its activation rows stay in LDS), measured against the built-in choice
// otherwise on 7900 launches of random shapes and 5-16 k steps, 120 tiles to walks of 14, geometric means (worst):
//   3-8 rows, walks of 1 / 2 / 3 tiles 0.83 / 0.85 / 0.80 of the time (0.96): 4096x4096 at 8 rows 5.61 us / 6.48;
//     8192x8192 g64 at 3 rows 12.1 / 13.6; 5004x5280 g96 at 3 rows 8.24 / 9.84; int8 11008x4096 at 4 rows 10.0 / 11.9;
//     fewer k steps leave SIMDs without a wave: 4 0.95 (1.1), 2 1.06 (1.4);
//   walks of 5 0.79 (0.99): the LDS-staged kernel's workgroups of 4 tiles need a second round there; other longer
//     walks by the units of the busiest SIMD, here against there (a workgroup of n k steps puts ceil(n/4) waves on a
//     SIMD): walks of 4 and 6 up to 1.15 times as many 0.90 (1.06), then 1.02 (1.13); walks from 7 up to 1.05 times
//     0.92 (1.07), then 1.03 (1.3).  28672x8192 at 4 rows 31.3 / 35.1, 28672x4096 17.9 / 20.1; 13824x5120 level;
//   2 rows, against the VALU kernel's waves: 5-8 k steps 0.85 (1.1), 28672x4096 17.7 / 18.9; 9-16 k steps, 3500 launches,
//     0.87 (1.07), 28672x8192 31.3 / 34.2 -- but 1.0 (1.13) on walks of 4 with 9, 10 or 13 k steps, where the waves of a
//     workgroup leave a SIMD or two idle a sixth of the time and more, and four groups per lane run do not make up for it
//     (15312x4608 13.5 / 12.0).  int8 at 2 rows: one scale lookup per lane run level, four 0.90 from 9 k steps;
//   9-16 rows, where they fit: walks of 1-3 tiles 0.84 (0.96), longer ones up to 2.0;
//   one row: 0.97 with a spread of 0.8-1.3, so it stays on the VALU kernel.
inline bool use_k_stationary_bf16(int m_batch, int tiles, int ksteps, int bits, int cus, bool generic_groups) {
  if (m_batch < 2 || ksteps < 5 || tiles * 2 < cus) return false;
  const int walk = ceil_div(tiles, cus);
  if (m_batch == 2) {
    if (bits == 8) return generic_groups && ksteps >= 9;
    return ksteps <= 8 || walk != 4 || generic_groups || 4 * ceil_div(ksteps, 4) * 6 < ksteps * 7;
  }
  if (walk <= 3) return true;
  if (m_batch > 8) return false;
  if (walk == 5) return true;
  const int tw = lds_staged_tiles_per_wg(tiles, 8, cus);
  const long long here = 4ll * walk * ceil_div(ksteps, 4), there = (long long)ceil_div(ceil_div(tiles, tw), cus) * tw * ksteps;
  return here * 100 <= there * (walk <= 6 ? 115 : 105);
}

// LDS stages of the k-stationary kernel's waves: 8 rows each to turn the operand round in (fp16), or the rows that stay (bf16).
// (With left-over tiles in parts the rows stay in fp16 as well.)
inline size_t kstat_stage_bytes(int waves, int bits, int m_batch, bool bf16, int parts = 0) {
  return (size_t)waves * (bf16 || parts != 0 ? m_batch : 8) * (step_k(bits) * 2 + 16);
}

// Workgroups per left-over tile of a k-stationary launch; 0: walks of whole tiles, some one longer than the others.  313 tiles
// on 256 compute units are walks of two for 57 of them, and the launch takes as long as two tiles everywhere; with four parts to
// a left-over tile each compute unit has a quarter more than its first.  What a launch has to gain is units of its busiest SIMD (a
// wave per k step, dealt out to four SIMDs in turn); what it pays is one barrier at its start and a unit in code nobody has
// fetched yet, 0.4-0.5 us, so one unit saved is not enough but with 8 bf16 k steps, and fp16, whose units are shorter, pays less
// often.  Part of the built-in measured plans.  Of the time of whole tiles, same kernel, 1300 launches of random shapes:
//   bf16 walks of 1 / 2 / 3: four parts 0.93 / 0.92 / 0.95 (9 k steps 0.87; 5004x5280 g96 at 3 rows 9.7 us / 8.8, 9104x5632 at 3 rows
//     12.5 / 11.5), two parts 0.97 / 0.93 / 0.96 (14-16 k steps on other walks than 2: 0.99-1.01, left out);
//   fp16, from 9 k steps: four parts 0.90-0.99 (4608x8192 at 4 rows 9.4 / 8.6; 11-14 k steps 0.98-1.02, left out), two parts on walks
//     of 2 and 3 0.94-0.97 / 0.97-0.99 (9104x8192 at 4 rows 13.1 / 11.2), on walks of 1 1.0.  5 and 6 k steps take 1.03-1.07 on 180
//     launches (9700x2440 at 7 rows 5.7 / 6.0): a part's unit in code nobody has fetched yet is longer than the two short ones saved.
// Longer walks and one unit saved: 0.98-1.1.  int8, whose rows are half as long, 1.03-1.15; four lookups per run in fp16 have
// no registers for it.
inline int left_over_parts(int m_batch, int tiles, int ksteps, int bits, int cus, bool bf16, bool generic_groups) {
  const int walk = tiles / cus, left_over = tiles % cus;
  if (bits != 4 || walk < 1 || walk > 3 || left_over == 0 || ksteps < 5 || (!bf16 && generic_groups)) return 0;
  const int parts = m_batch <= 4 && left_over * 4 <= cus ? 4 : m_batch <= 8 && left_over * 2 <= cus ? 2 : 0;
  if (parts == 0) return 0;
  // units of the busiest SIMD: now, and with a part's units dealt out as kstat_tail_unit has it
  int most = 0;
  for (int simd = 0; simd < 4; ++simd) {
    int units = 0;
    for (int kw = simd; kw < ksteps; kw += 4) units += walk + (kstat_tail_unit(kw, ksteps) * parts < ksteps ? 1 : 0);
    most = units > most ? units : most;
  }
  const int saved = (walk + 1) * ceil_div(ksteps, 4) - most;
  if (bf16) {
    if (ksteps == 8) return parts;
    return saved >= 2 && (walk < 3 || ksteps != 12) && (parts == 4 || ksteps <= 13 || walk == 2) ? parts : 0;
  }
  if (saved < 2 || ksteps < 9) return 0;
  return parts == 4 ? (ksteps <= 10 || ksteps >= 15 ? parts : 0) : walk >= 2 ? parts : 0;
}

// Several problems: the next one's workgroups fill the place of the shorter walks, so parts pay only where they are a quarter of the
// compute units or more: 0.96 of the time of whole tiles (0.82-1.06, 157 launches of two to eight problems).  Fewer took 1.03-1.09,
// up to 1.18 (eight problems of 4232x4608 at 8 rows in bf16 39.0 us / 46.2).  Nor do they with 5 and 8 k steps, where the busiest SIMD
// saves a unit or none: 1.0 (0.92-1.19).
inline bool left_over_parts_of_batch(int m_batch, int tiles, int ksteps, int cus) {
  if (ksteps < 6 || ksteps == 8) return false;
  const int left_over = tiles % cus, parts = m_batch <= 4 && left_over * 4 <= cus ? 4 : 2;
  return left_over * parts * 4 >= cus;
}

LaunchPlan plan_launch(int n_out, int k, int bits, int m_batch, const PlanKnobs& knobs) {
  const int tiles = num_tiles(n_out), ksteps = num_ksteps(k, bits);
  const int cus = knobs.num_cus > 0 ? knobs.num_cus : kNumCus;  // the thresholds below were measured on 256 and scale with it
  const int ov_sk = knobs.split_k, ov_tw = knobs.tiles_per_wg;
  const int ov_t = knobs.tiles_per_wave;
  const bool mc = use_matrix_cores(m_batch, tiles, ksteps, knobs.matrix_core_min_batch, knobs.wide_waves, bits, cus);
  // K-stationary kernel: one wave per k step (so at most 16 k steps), one workgroup per compute unit
  // or fewer, each walking a contiguous run of tiles; more workgroups only where a walk's partial
  // sums would not fit the LDS or its weights not a 32-bit offset.
  // bf16 (the operand stays in LDS, beside the partial sums): where the two fit.
  const long long park_bytes = (long long)kKSlices * m_batch * kKStationaryParkSlots * 16;  // partial sums per tile of a walk
  const long long stage_bytes = knobs.wide_waves ? (long long)kstat_stage_bytes(ksteps, bits, m_batch, true) : 0;  // bf16: the rows stay
  const long long most_lds = knobs.wide_waves ? kMaxKStationaryBf16Lds : kMaxKStationaryLds;
  const bool kstat_exists = ksteps <= kMaxWavesPerWorkgroup && stage_bytes + park_bytes <= most_lds;
  const bool kstat_asked = mc && knobs.matrix_core_variant == MGEMV_MATRIX_CORE_K_STATIONARY;
  const bool kstat_by_rule = knobs.matrix_core_variant == MGEMV_MATRIX_CORE_AUTO && knobs.matrix_core_min_batch == 0 &&
                             ov_sk == 0 && ov_tw == 0 && ov_t == 0 &&
                             (knobs.wide_waves ? stage_bytes + ceil_div(tiles, cus) * park_bytes <= most_lds &&
                                                     use_k_stationary_bf16(m_batch, tiles, ksteps, bits, cus, knobs.generic_groups)
                                               : !knobs.generic_groups && use_k_stationary(m_batch, tiles, ksteps, bits, cus));
  if (kstat_exists && (kstat_asked || kstat_by_rule)) {
    LaunchPlan lp{};
    lp.matrix_core = true;
    lp.k_stationary = true;
    lp.split_k = ksteps;
    lp.steps_per_wave = 1;
    lp.tiles_per_wg = 1;
    lp.tiles_per_wave = 1;
    lp.stages = 2;
    lp.workgroups = knobs.workgroups > 0 ? knobs.workgroups : cus;
    if (lp.workgroups > tiles) lp.workgroups = tiles;
    auto walk = [&]() { return ceil_div(tiles, lp.workgroups); };
    while (lp.workgroups < tiles &&
           ((long long)(walk() + 2) * ksteps * kUnitBytes >= (1ll << 31) ||  // (the loop requests up to two tiles past the walk)
            stage_bytes + walk() * park_bytes > most_lds))
      lp.workgroups = lp.workgroups * 2 < tiles ? lp.workgroups * 2 : tiles;
    lp.tiles_in_sequence = walk();
    lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
    lp.threads = kWave * lp.split_k;
    if (knobs.split_left_over && lp.workgroups == cus) {
      const int parts = left_over_parts(m_batch, tiles, ksteps, bits, cus, knobs.wide_waves, knobs.generic_groups);
      if (parts != 0 && (long long)kstat_stage_bytes(ksteps, bits, m_batch, true, parts) + walk() * park_bytes <=
                            kMaxKStationaryBf16Lds - kKStationaryStagedBytes)
        lp.parts = parts;
    }
    return lp;
  }
  // The LDS-staged kernel serves every matrix-core launch of two or more tiles.  (While its loop
  // still had a workgroup barrier per k step, the register-operand kernel was ahead on problems of
  // up to 256 tiles with up to 5 rows or up to 4 k steps; without the barrier the LDS-staged kernel
  // with one tile per workgroup wins there too -- 4096x4096, 5 rows: 4.98 us against 5.34;
  // 2048x8192, 5 rows: 6.5 against 7.5; 2048x2048, 8 rows: 3.68 against 3.91 -- or is level,
  // 2048x2048, 5 rows: 3.62 against 3.57.)
  if (mc && knobs.matrix_core_variant != MGEMV_MATRIX_CORE_REGISTER_OPERAND && tiles >= 2) {
    // LDS-staged kernel: the tiles of a workgroup share the activation stage; k split as long as
    // the launch stays within 2048 waves (measured: 8192x8192 best at 4 k-split waves, 11008x4096
    // at 2, 28672x8192 at 1).
    LaunchPlan lp{};
    lp.matrix_core = true;
    lp.staged_rows = m_batch <= 8 ? 8 : 16;
    lp.tiles_per_wg = lds_staged_tiles_per_wg(tiles, lp.staged_rows, cus);
    // Long reductions on many tiles (more than 16 k steps, more than 4 tiles per compute unit; the k-stationary kernel
    // does not reach these) want about two workgroups per compute unit, of few waves that walk the whole reduction:
    // 2 tiles per workgroup, or 4 where that still leaves more than 2.75 workgroups per compute unit; up to 8 rows,
    // workgroups of 2 tiles split k in two.  Against what the rules above give (us): 34576x8576 at 12 rows 40.9 / 47.7;
    // 33664x8832 at 16 rows 43.8 / 52.0; 19056x10112 at 3 / 12 rows 24.7 / 27.8, 32.8 / 38.1; 16400x9216 at 16 rows
    // 29.4 / 35.0; 28672x8704 at 5 / 16 rows 29.0 / 32.2, 33.0 / 36.2; 22016x11008 at 8 rows 30.4 / 33.6.
    const bool long_reduction = ksteps > 16 && tiles > 4 * cus;
    // (Up to 8 rows, 4 tiles only where their workgroups fill the last round to three quarters -- 28672x8704 and int8
    // 27216x4224 do, 23648x11392 and int8 33616x4352 do not: 4-12 % either way.)
    if (long_reduction) {
      const int wgs4 = ceil_div(tiles, 4);
      const bool four = lp.staged_rows == 16 ? ceil_div(tiles, 2) * 4 > cus * 11 : wgs4 * 4 >= ceil_div(wgs4, cus) * cus * 3;
      lp.tiles_per_wg = four ? 4 : 2;
    }
    // Parts of tiles (measured ranges only): the waves of a workgroup share the units of `parts` k steps.
    if (knobs.parts > 0 && knobs.parts * m_batch <= kTileRows) {
      lp.tiles_per_wg = lp.tiles_per_wave = lp.tiles_in_sequence = 1;
      lp.parts = knobs.parts;
      lp.staged_rows = lp.parts < 4 && lp.parts * m_batch <= 8 ? 8 : 16;
      lp.workgroups = tiles * lp.parts;
      // Up to 8 units a wave each (0.90-0.96 of the time of half as many waves of two); more of them four waves, one per SIMD:
      // what such a launch waits for is a compute unit's path to memory, not latency, and 8 take 1.0-1.08 times as long
      // (bf16 on up to 64 tiles 0.97-1.0).
      const int units = ceil_div(ksteps, lp.parts);
      const int units_per_wave = ceil_div(units, units <= kMaxWavesPerMfmaWorkgroup ? units : 4);
      lp.steps_per_wave = units_per_wave * lp.parts;
      lp.split_k = ceil_div(units, units_per_wave);
      lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
      lp.threads = kWave * lp.split_k;
      lp.stages = 2;
      return lp;
    }
    // the kernel exists for 2, 4, 8 or 16 staged rows per wave of a k range
    if (ov_tw > 0 && ov_tw <= 8 && lp.staged_rows % ov_tw == 0 && lp.staged_rows / ov_tw >= 2) lp.tiles_per_wg = ov_tw;
    lp.workgroups = ceil_div(tiles, lp.tiles_per_wg);
    const int max_split = kMaxWavesPerMfmaWorkgroup / lp.tiles_per_wg < 4 ? kMaxWavesPerMfmaWorkgroup / lp.tiles_per_wg : 4;
    int split = 1;
    // (a tile count that left every tile a workgroup of its own, on a large matrix: single-wave workgroups are the worst
    // of all -- 16880x5376 bf16 at 5 rows 28.7 us against 22.6 with four k-split waves -- so those may use twice the waves)
    const int lds_wave_budget = (lp.tiles_per_wg == 1 && tiles > 2 * cus ? 20 : 8) * cus;
    while (split < max_split && split * 2 <= ksteps && (long long)lp.workgroups * lp.tiles_per_wg * split * 2 <= lds_wave_budget) split *= 2;
    if (long_reduction) split = lp.staged_rows == 8 && lp.tiles_per_wg == 2 ? 2 : 1;
    // three k steps: a wave each instead of 2 + 1 (2048x1408, 8 / 16 rows: 3.52 / 3.96 us against 4.11 / 4.69)
    if (ksteps == 3 && split == 2 && max_split >= 3 && (long long)lp.workgroups * lp.tiles_per_wg * 3 <= 8 * cus) split = 3;
    // A split that leaves the last wave nearly idle (10 k steps over 4 waves: 3, 3, 3, 1) loses
    // to half as many evenly loaded waves, as long as the workgroup keeps four (5120x5120, 8 rows,
    // 2 tiles: 7.6 us at 2 waves per tile against 8.1 at 4; 6912x5120, 16 rows: 9.0 against 9.6;
    // but 4096x6656, 8 rows, 1 tile: 9.1 at 2 against 7.8 at 4).
    auto padded_steps = [&](int s) { const int st = ceil_div(ksteps, s); return st * ceil_div(ksteps, st); };
    if (lp.tiles_per_wg * split >= 8 && padded_steps(split) * 100 > ksteps * 115 &&
        padded_steps(split / 2) < padded_steps(split))
      split /= 2;
    if (ov_sk > 0) split = ov_sk > max_split ? max_split : ov_sk;
    if (split > ksteps) split = ksteps;
    lp.steps_per_wave = ceil_div(ksteps, split);
    lp.split_k = ceil_div(ksteps, lp.steps_per_wave);
    lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
    lp.threads = kWave * lp.split_k * lp.tiles_per_wg;
    lp.tiles_per_wave = 1;
    lp.tiles_in_sequence = 1;
    lp.stages = 2;
    return lp;
  }
  // Matrix-core path: a wave that works on T tiles fetches the activation operands of a k step
  // once for all of them.  Measured on 8192 x 8192 (512 tiles): T = 2 is 1.5-1.8x faster than
  // T = 1 at 8-16 activation rows; T = 4 leaves too few waves to cover the load latency.
  int tiles_per_wave = 1;
  if (mc) {
    tiles_per_wave = tiles >= cus ? 2 : 1;
    if (ov_t == 1 || ov_t == 2 || ov_t == 4) tiles_per_wave = ov_t;
  }
  // One row, parts of tiles (measured ranges only).
  if (!mc && m_batch == 1 && knobs.parts > 0) {
    LaunchPlan lp{};
    lp.tiles_per_wg = lp.tiles_per_wave = lp.tiles_in_sequence = 1;
    lp.parts = knobs.parts;
    lp.workgroups = tiles * lp.parts;
    const int units = ceil_div(ksteps, lp.parts);
    const int units_per_wave = ceil_div(units, units <= kMaxWavesPerWideWorkgroup ? units : units <= kMaxWavesPerWorkgroup && lp.parts == 1 ? kMaxWavesPerWideWorkgroup : 4);
    lp.steps_per_wave = units_per_wave * lp.parts;
    lp.split_k = ceil_div(units, units_per_wave);
    lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
    lp.threads = kWave * lp.split_k;
    lp.stages = 2;
    return lp;
  }
  const int groups = ceil_div(tiles, tiles_per_wave);
  // (The VALU figures from here on are from before its builds by length.  On a device of 256 compute units single_row_split is asked
  // first for a single row on more tiles than that.)
  // Shapes that the exact-fit rule below does not take (measured on MI355X; one tile group per
  // workgroup is best throughout):
  //  * about one workgroup per compute unit or fewer (<= 384 tile groups): few, longer waves --
  //    4 k-split waves, each pipelining two or more units -- beat more, shorter ones
  //    (4096x4096: 4.08 us at 4 waves against 4.33 us at 8);
  //  * more tile groups than that: split as far as the units allow while the launch stays under
  //    ~8k waves, and fall back to two units per wave when that still leaves >= 4096 waves.
  const int max_waves = mc ? kMaxWavesPerMfmaWorkgroup
                        : m_batch >= 3 || knobs.wide_waves ? kMaxWavesPerWideWorkgroup
                                                  : kMaxWavesPerWorkgroup;
  int split_k;
  // 288-512 tiles and a longer reduction: two tiles per workgroup, two k-split waves each (four
  // up to 384 tiles from 20 k steps) -- at most one workgroup per compute unit and one wave per
  // SIMD, the exact fit below without its divisibility -- beat one tile per workgroup with four
  // waves (5120x5120: 5.8 us against 6.2; 6144x8192: 7.7 against 8.3; 5120x14336: 11.0 against
  // 11.5) and one-unit or two-unit waves (7168x8192: 7.8 against 8.7; 6656x11008: 9.9 against
  // 11.3; 7168x14336: 11.8 against 15.3); at 260 tiles they are 1-3 % behind (4160x8192).
  const bool pair_tiles = !mc && tiles * 8 >= cus * 9 && tiles <= 2 * cus && ksteps >= 9;
  if (pair_tiles) {
    split_k = tiles <= cus * 3 / 2 && ksteps >= 20 ? 4 : 2;
  } else if (groups <= cus * 3 / 2) {
    split_k = ksteps < 4 ? ksteps : 4;
    // With workgroups for at most half the compute units, one unit per wave is 4-5 % ahead up to
    // 16 k steps (1024x4096: 3.38 us against 3.54; 1024x8192: 4.54 against 4.77); with a longer
    // reduction it is not (2048x11008: 6.35 at 8 waves against 6.12).
    if (!mc && tiles <= cus / 2 && ksteps <= 16) split_k = ksteps;
    // More than one workgroup per compute unit and 5-8 k steps, one or two rows: four waves would take
    // two units each, the one length at which the two-deep pipeline overlaps nothing; one unit
    // per wave is 6-7 % ahead (4608x4096: 4.81 us against 5.13; 6144x4096: 4.98 against 5.29),
    // while at 256 tiles four waves win (4096x4096: 4.08 against 4.33).
    if (!mc && m_batch <= 2 && tiles > cus && ceil_div(ksteps, 4) == 2) split_k = ksteps;
    if (mc) split_k = ksteps < max_waves ? ksteps : max_waves;  // not pipelined: wants waves
  } else {
    // One or two rows and up to 8 k steps: workgroups of up to 8 one-unit waves stay ahead of two-unit
    // waves well past 8192 waves (22016x4096, 11008 waves: 10.9 us against 11.8; 27200x4096,
    // 13600 waves: 12.6 against 13.0; 36864x2560: 11.8 against 12.3).
    // (int8 weights: the same reductions are twice as many k steps, and with half the arithmetic per byte more,
    // shorter waves stay ahead there as well -- 22016x4096 at 1 / 2 rows 15.6 / 15.5 us with 8 waves per tile against
    // 16.6 / 17.1 with 4; 11008x4096 at 2 rows 8.93 / 9.61; 12288x4096 9.55 / 10.19; 28672x4096 19.1 / 20.2.)
    const bool short_single_row = !mc && m_batch <= 2 && ksteps <= (bits == 8 ? 16 : 8);
    const int kWaveBudget = (short_single_row ? 64 : 32) * cus;
    const int kSimds = cus * 4;
    split_k = ksteps < max_waves ? ksteps : max_waves;
    if (short_single_row && bits == 8 && split_k > 8) split_k = 8;  // 16 one-unit waves lose: 11008x4096, 2 rows, 11.0 us / 8.9
    // One wave per unit does not fit the machine at once, and one wave per tile fills at least
    // 75 % of the SIMDs of its last round: the whole-k waves win (13824x5120: 9.1 us against
    // 10.3 at 5 waves per tile; 27648x5120: 15.6 against 17.5 at 3; 14848x6144: 10.6 against 12.1
    // at 6; 13824x8192: 12.6 against 13.7 at 8).  With a worse fit they lose (17408x5120, 1088
    // tiles: 13.8 against 12.4), and the halving below stands.
    const bool whole_k_waves = !mc && !knobs.wide_waves && m_batch <= 2 && (long long)groups * split_k > kWaveBudget &&
                               (long long)tiles * 100 >= (long long)ceil_div(tiles, kSimds) * kSimds * 75;  // (12432x6144, 76 %: 10.2 us / 11.5)
    if (whole_k_waves) split_k = 1;
    while (split_k > 1 && (long long)groups * split_k > kWaveBudget) split_k = (split_k + 1) / 2;
    if (!mc && !short_single_row && split_k > 1 && ceil_div(ksteps, split_k) < 2 &&
        (long long)groups * ((split_k + 1) / 2) >= 16 * cus)
      split_k = (split_k + 1) / 2;
    // From 16 k steps four waves with longer pipelines are level with or ahead of more, shorter
    // ones (9216x14336: 16.9 us against 18.1 at 7 waves; 10240x11008: 14.8 against 15.3 at 11;
    // 10240x8192 and 11008x8192: level).
    if (!mc && !short_single_row && ksteps >= 16 && split_k > 4) split_k = 4;
    // The bfloat16 kernels are bound by their arithmetic, and two-unit waves are their worst
    // length by far (13824x5120: 18.9 us at 5 waves of 2 units against 14.0 at 2 waves of 5).
    if (knobs.wide_waves && !mc && split_k > 1 && ceil_div(ksteps, split_k) == 2) split_k = (split_k + 1) / 2;
    // A single bf16 row on 700 and more tiles, up to 16 k steps.  A wave per k step leaves the SIMDs with unequal numbers
    // of them and turns workgroups over for one unit each: int4, 3 or 4 waves instead take, geometric means (worst), with 5
    // k steps 0.80 of the time (1.04), 6 0.87 (1.0), 7 0.91-0.95 (1.05), 8 level (but with four groups per
    // lane run 0.85); int8 is level.  So is one wave with 4 k steps (0.92, int8 0.85).
    if (knobs.wide_waves && !mc && m_batch == 1 && tiles * 8 >= cus * 22 && ksteps <= 16) {
      if (bits == 4 && ksteps >= 5 && split_k == ksteps) {
        if (ksteps < 8 || knobs.generic_groups) split_k = ksteps <= 6 ? 3 : 4;
      } else if (!knobs.generic_groups && split_k == 1 && ksteps == 4) {
        split_k = 4;
      }
    }
    // Where the wave budget stops at two bf16 waves per tile, four (three with 5 and 6 k steps).  Two do not give a SIMD enough to
    // choose from, and 2300-2560 tiles of them are on the machine all at once with nothing left to even out its end:
    // two / four waves 37976x4352 int8 34.3 us / 30.9, 38400x5376 g96 37.4 / 32.7, 38232x8576 g64 at two rows 58.7 / 51.1; over 3300
    // launches of 1300-8000 tiles 0.80-1.04, mean 0.936.  int8 with
    // 9 and 10 k steps is level (0.99-1.02) and keeps two, but for single rows with one or two groups per run, which take 0.99.
    const bool level = bits == 8 && (ksteps == 9 || ksteps == 10) && (m_batch > 1 || knobs.generic_groups);
    if (knobs.wide_waves && !mc && split_k == 2 && ksteps >= 5 && !level) split_k = 4;
  }
  int tiles_per_wg = pair_tiles ? 2 : 1;
  int workgroup_cap = 0;
  if (!mc && tiles >= cus && ksteps >= 5) {
    // "Exact fit": when the tiles divide (nearly) evenly over the compute units, one workgroup
    // of four waves per compute unit -- one wave per SIMD, all with the same amount of work --
    // beats any over-subscribed launch (8192x8192: 8.7 us against 10.2 us; 28672x8192: 2 %).
    // The four waves are tw tile sequences x 4/tw k-split waves, tw as large as still fits evenly.
    // Walks of more than 7 tiles lose to one tile per workgroup (128256x4096, 8 tiles per wave:
    // 51.5 us against 47.3; 151936x2048, 19 tiles: 31.9 against 29.8), so those are left out.
    // (The bfloat16 kernels want every SIMD busy more than they want equal walks: 28672x8192 takes
    // 35.5 us with one tile and four waves per workgroup against 38.4 with walks of 7 tiles.)
    const int tw = even_fit(tiles, ksteps, knobs.wide_waves ? 1 : 7, cus);
    if (tw != 0) {
      tiles_per_wg = tw;
      split_k = 4 / tw;
      workgroup_cap = cus;
    }
  }
  if (ov_sk > 0) split_k = ov_sk;
  if (ov_tw > 0) tiles_per_wg = ov_tw;
  split_k = split_k > max_waves ? max_waves : split_k;
  split_k = split_k > ksteps ? ksteps : split_k;
  const int steps = ceil_div(ksteps, split_k);
  split_k = ceil_div(ksteps, steps);
  if (tiles_per_wg * split_k > max_waves) tiles_per_wg = max_waves / split_k;
  LaunchPlan lp{};
  lp.split_k = split_k;
  lp.tiles_per_wg = tiles_per_wg;
  lp.steps_per_wave = steps;
  lp.workgroups = ceil_div(groups, tiles_per_wg);
  lp.tiles_in_sequence = 1;
  lp.staged_rows = 0;
  lp.matrix_core = mc;
  lp.stages = !mc && knobs.stages == 1 ? 1 : 2;
  if (!mc) {
    // VALU path: fewer workgroups than tile groups means every wave walks several tiles.
    const int ov_wg = knobs.workgroups;
    int cap = ov_wg > 0 ? ov_wg : (workgroup_cap > 0 && ov_sk == 0 && ov_tw == 0) ? workgroup_cap : lp.workgroups;
    if (cap < lp.workgroups) lp.workgroups = cap;
    const int rows = m_batch < kMaxValuBatch ? m_batch : kMaxValuBatch;
    auto seq_tiles = [&]() { return ceil_div(tiles, lp.workgroups * tiles_per_wg); };
    // limits: a wave's weight range is addressed with 32-bit offsets; the combine parks
    // tiles x waves x rows x 64 floats in LDS
    while (lp.workgroups < ceil_div(groups, tiles_per_wg) &&
           ((long long)seq_tiles() * ksteps * kUnitBytes >= (1ll << 31) ||
            (long long)seq_tiles() * tiles_per_wg * split_k * rows * kWave * 4 > 64 * 1024))
      lp.workgroups = lp.workgroups * 2 < ceil_div(groups, tiles_per_wg) ? lp.workgroups * 2 : ceil_div(groups, tiles_per_wg);
    lp.tiles_in_sequence = seq_tiles();
  }
  lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
  lp.threads = kWave * split_k * tiles_per_wg;
  lp.tiles_per_wave = tiles_per_wave;
  return lp;
}

int check_problem(const void* weights, const void* scale, const void* zero_add, int n_out, int k, int& group_size,
                  int quant_op, int weight_bits) {
  if (quant_op != MGEMV_PER_COLUMN_SCALE_ONLY && quant_op != MGEMV_FINEGRAINED_SCALE_ONLY &&
      quant_op != MGEMV_FINEGRAINED_SCALE_AND_ZEROS)
    return MGEMV_ERR_QUANT_OP;
  if (weight_bits != 4 && weight_bits != 8) return MGEMV_ERR_QUANT_TYPE;
  if (n_out <= 0 || k <= 0) return MGEMV_ERR_SIZE;
  if (n_out % 4) return MGEMV_ERR_ROWS;
  if (k % 8) return MGEMV_ERR_COLS;  // utils/preprocess.h:324-327
  if (quant_op == MGEMV_PER_COLUMN_SCALE_ONLY) {
    group_size = k;  // mixed_gemv_test.cu:142-143
  } else {
    if (group_size < 64) return MGEMV_ERR_GROUP_SIZE;  // gemv/device/gemv_adaptor.h:199-203
    if (group_size % 32 || k % group_size) return MGEMV_ERR_GROUP_SIZE;
  }
  if (weights == nullptr || scale == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (quant_op == MGEMV_FINEGRAINED_SCALE_AND_ZEROS && zero_add == nullptr) return MGEMV_ERR_NULL_POINTER;
  // 32-bit index arithmetic inside the kernels
  const long long groups = k / group_size;
  if (groups * (long long)n_out >= (1ll << 30)) return MGEMV_ERR_SIZE;
  if (num_ksteps(k, weight_bits) > 0xffff || group_size >= (1 << 24)) return MGEMV_ERR_SIZE;
  if ((long long)k * 2 * MGEMV_MAX_M_BATCH >= (1ll << 31)) return MGEMV_ERR_SIZE;
  if (reinterpret_cast<uintptr_t>(weights) % 16) return MGEMV_ERR_ALIGNMENT;
  if (reinterpret_cast<uintptr_t>(scale) % 2 || reinterpret_cast<uintptr_t>(zero_add) % 2) return MGEMV_ERR_ALIGNMENT;
  return MGEMV_OK;
}

// What a plan asks of the hardware: dynamic LDS of its (largest) launch, the workgroup size limit the
// kernel it picks was compiled for, and how many launches serve all activation rows.
struct LaunchResources {
  size_t lds_bytes;
  int max_threads;
  int launches;
};
LaunchResources launch_resources(const LaunchPlan& lp, int bits, int m_batch, int act) {
  LaunchResources r{};
  r.launches = 1;
  if (lp.matrix_core && lp.k_stationary) {
    r.max_threads = kWave * kMaxWavesPerWorkgroup;
    const size_t stage = kstat_stage_bytes(lp.split_k, bits, m_batch, act == kActBf16, lp.parts), park = (size_t)lp.tiles_in_sequence * kKSlices * m_batch * kKStationaryParkSlots * 16;
    // both when they fit (then no barrier stands between a wave's operand and its walk), else the larger of the two
    r.lds_bytes = act == kActBf16 || lp.parts != 0 || stage + park <= (size_t)kMaxKStationaryLds ? stage + park : stage > park ? stage : park;
    return r;
  }
  if (lp.matrix_core) {
    r.max_threads = kWave * kMaxWavesPerMfmaWorkgroup;
    if (lp.staged_rows != 0) {
      const int row_stride = step_k(bits) * 2 + 16;
      // (a wave of the part-tile kernel has one stage, its own)
      r.lds_bytes = (size_t)lp.split_k * (lp.parts != 0 ? 1 : 2) * lp.staged_rows * row_stride +
                    (lp.split_k > 1 || lp.parts > 1 || lp.chains != 0
                         ? (size_t)lp.tiles_per_wg * lp.split_k * (lp.chains != 0 ? lp.chains_per_wave : 1) * kWave * 4 * sizeof(float) : 0);
    } else {
      r.lds_bytes = lp.split_k == 1 ? 0 : (size_t)lp.tiles_per_wg * lp.split_k * lp.tiles_per_wave * kWave * 4 * sizeof(float);
    }
    return r;
  }
  const int rows = m_batch < kMaxValuBatch ? m_batch : kMaxValuBatch;
  r.launches = (m_batch + kMaxValuBatch - 1) / kMaxValuBatch;
  r.max_threads = kWave * (rows >= 3 || act == kActBf16 || lp.parts != 0 ? kMaxWavesPerWideWorkgroup : kMaxWavesPerWorkgroup);
  r.lds_bytes = (size_t)lp.tiles_in_sequence * lp.tiles_per_wg * lp.split_k * rows * kWave * sizeof(float);
  if (lp.parts != 0) {  // every unit's sums
    int units = lp.split_k * lp.steps_per_wave / lp.parts;
    if (lp.parts == 1 && units > kValuPartsSumsAtOnce) units = lp.split_k;  // every wave adds up its own
    r.lds_bytes = (size_t)ceil_div(units, kValuPartsSumsAtOnce) * kValuPartsSumsAtOnce * kWave * sizeof(float);
  }
  return r;
}

hipError_t launch_gemv(const GemvLaunch& g, int bits, int qop, int mb, int gpr, int act) {
  return act == kActBf16 ? launch_gemv_bf16(g, bits, qop, mb, gpr) : launch_gemv_f16(g, bits, qop, mb, gpr);
}

template <int BITS, int ACT>
hipError_t launch_dequant(const DequantParams& p, int qop, half_t* out, hipStream_t stream) {
  const long long units = (long long)p.tiles * p.ksteps;
  const dim3 block(kWave * kDequantWaves), grid((unsigned)((units + kDequantWaves - 1) / kDequantWaves));
  switch (qop) {
    case 1: return launch(dequantize_kernel<BITS, 1, ACT>, grid, block, 0, stream, p, out);
    case 2: return launch(dequantize_kernel<BITS, 2, ACT>, grid, block, 0, stream, p, out);
    default: return launch(dequantize_kernel<BITS, 3, ACT>, grid, block, 0, stream, p, out);
  }
}

// What the launch path needs to know about a device, looked up once per device and process
// (the first launch on a device pays for one hipGetDeviceProperties call).
struct DeviceInfo {
  bool usable;   // a gfx950 device
  int num_cus;
};
constexpr int kMaxDevices = 64;
std::atomic<int> g_device_state[kMaxDevices];  // 0 unknown, else 1 + (usable ? num_cus : 0)

// The device a stream belongs to (the null stream: the calling thread's current device).
int device_of_stream(hipStream_t stream, int& device) {
  if (stream != nullptr && hipStreamGetDevice(stream, &device) == hipSuccess) return MGEMV_OK;
  return hipGetDevice(&device) == hipSuccess ? MGEMV_OK : MGEMV_ERR_NO_DEVICE;
}

int device_info(int device, DeviceInfo& info) {
  const bool tracked = device >= 0 && device < kMaxDevices;
  int state = tracked ? g_device_state[device].load(std::memory_order_relaxed) : 0;
  if (state == 0) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return MGEMV_ERR_NO_DEVICE;
    const bool usable = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0;
    state = 1 + (usable ? prop.multiProcessorCount : 0);
    if (tracked) g_device_state[device].store(state, std::memory_order_relaxed);
  }
  info.usable = state > 1;
  info.num_cus = state - 1;
  return info.usable ? MGEMV_OK : MGEMV_ERR_NO_DEVICE;
}

// The knobs of a problem with the element type taken into account.
PlanKnobs knobs_for_element(int n_out, int k, int bits, int group_size, int m_batch, int act, int num_cus = kNumCus, bool whole_tiles = false) {
  PlanKnobs knobs = knobs_for(n_out, k, bits, group_size, m_batch, act, num_cus, whole_tiles);
  knobs.num_cus = num_cus;
  // (a group as long as k is the per-column mode, whose kernels look one scale up per row)
  knobs.generic_groups = lookups_per_run(k, group_size, bits) == 4;
  if (act == kActBf16) {
    // bf16: of the matrix-core kernels the LDS-staged and the k-stationary one (both need two tiles here); the VALU
    // kernel's dequantiser wants the registers of 8-wave workgroups
    if (num_tiles(n_out) < 2) knobs.matrix_core_min_batch = MGEMV_MAX_M_BATCH + 1;
    if (knobs.matrix_core_variant == MGEMV_MATRIX_CORE_REGISTER_OPERAND) knobs.matrix_core_variant = MGEMV_MATRIX_CORE_LDS_STAGED;
    knobs.wide_waves = true;
  }
  return knobs;
}

// As many parts, at most the single launch's, as leave a workgroup per compute unit when all problems are taken together.  A problem's
// workgroups are dealt out to the XCDs in equal numbers (the last XCD gets what is left), so each XCD is looked at: six problems of
// 42 workgroups are 36 for the 32 compute units of seven XCDs, and none for the eighth (328x7168 at 8 rows 8.0 us; 21 each 6.0).
int parts_of_batch(int parts, int tiles, int cus, int batch_count) {
  while (parts > 1 && (long long)ceil_div(tiles * parts, kNumXcd) * kNumXcd * batch_count > cus) parts /= 2;
  return parts;
}

// The plan of a batched or routed launch whose problems would each be split into parts.  Every number of parts gives the same bits, and
// up to 16 k steps (8 in bf16) so does the kernel for whole tiles, a wave per k step, so the number of problems may count: as
// many parts as leave a workgroup per compute unit, and where that is not all of them whole tiles, if their kernel gives the bits.
// Of the time of whole tiles, 1770 launches of two to eight problems: four parts 0.69, two 0.78, one 0.97 (1.13 at worst, 5
// launches above 1.05, all with four lookups per run).  With two workgroups per compute unit 1.1-1.5.  fp16 in fewer parts up to 16 k
// steps: 1.0-1.14.
LaunchPlan plan_of_batch(const LaunchPlan& single, int n_out, int k, int bits, PlanKnobs knobs, int batch_count) {
  knobs.parts = parts_of_batch(knobs.parts, num_tiles(n_out), knobs.num_cus, batch_count);
  if (knobs.parts == single.parts) return single;
  if (knobs.parts == 1 || !knobs.wide_waves) {
    PlanKnobs whole = knobs;
    whole.parts = 0;
    const LaunchPlan lp = plan_launch(n_out, k, bits, 1, whole);
    if (lp.steps_per_wave == 1 && lp.split_k > 1) return lp;
  }
  return plan_launch(n_out, k, bits, 1, knobs);
}

// The same for two and more rows on the part-tile matrix-core kernel, in the order of the single launch's sums (CHAINS).  Whole
// chains to up to eight waves where all problems leave a compute unit to each workgroup, else to four: eight there 1.0-1.2 of
// the time, two 1.1-1.5 (and level from 2 workgroups per compute unit on).  As many of them as leave the busiest SIMD the fewest
// chains: twelve on six waves are four, on four waves three (five problems of 800x5456 at 5 rows 8.6 us / 7.2).
// Two to eight problems of at most half as many tiles as compute units, 1445 launches of random shapes, of the time of the
// kernels that were there before parts: 0.89 (41 of them above 1.1, worst 1.26; 2 rows 0.93, 3 and 4 0.84, 5-8 0.93), where the
// single launch's parts took up to 2.2 (eight problems of 1024x9344 at 3 rows in bf16 14.1 us before, 30.8 in four parts each, 12.3
// here; of 2048x4352 at 8 rows 11.8, 24.5, 12.0).  Two rows of short reductions gain least: the VALU kernel had them.
LaunchPlan plan_of_batch_rows(const LaunchPlan& single, int m_batch, int tiles, int cus, int batch_count) {
  LaunchPlan lp = single;
  lp.parts = parts_of_batch(single.parts, tiles, cus, batch_count);
  if (lp.parts == single.parts) return single;
  lp.chains = single.parts / lp.parts;
  lp.workgroups = tiles * lp.parts;
  const int chains = single.split_k * lp.chains, most_waves = (long long)lp.workgroups * batch_count <= cus ? kMaxWavesPerMfmaWorkgroup : 4;
  int least = chains;  // of the busiest SIMD
  for (int waves = most_waves; waves >= 4; --waves) {
    const int per_wave = ceil_div(chains, waves), simd = ceil_div(ceil_div(chains, per_wave), 4) * per_wave;
    if (simd < least || waves == most_waves) {
      least = simd;
      lp.chains_per_wave = per_wave;
    }
  }
  lp.split_k = ceil_div(chains, lp.chains_per_wave);
  lp.staged_rows = lp.parts * m_batch <= 4 && lp.parts == 1 ? 4 : 8;
  lp.wgs_per_xcd = ceil_div(lp.workgroups, kNumXcd);
  lp.threads = kWave * lp.split_k;
  return lp;
}

// act: kActF16 or kActBf16, the type behind every 16-bit operand.
int gemv_any(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
             const uint16_t* bias, uint16_t* y, int batch_count, int n_out, int m_batch, int k, int group_size,
             int quant_op, int weight_bits, int64_t stride_weights, int64_t stride_x, int64_t stride_scale,
             int64_t stride_bias, int64_t stride_y, void* stream, int act, float alpha = 1.0f, float beta = 1.0f,
             int probe = kProbeNone, unsigned long long* trace = nullptr, size_t trace_capacity_waves = 0,
             bool timed_waits = false, const int32_t* route = nullptr, int route_extent = 0) {
  if (batch_count < 1 || batch_count > 65535) return MGEMV_ERR_BATCH;
  if (route != nullptr && route_extent < 1) return MGEMV_ERR_BATCH;
  if (reinterpret_cast<uintptr_t>(route) % 4) return MGEMV_ERR_ALIGNMENT;
  if (m_batch < 1 || m_batch > MGEMV_MAX_M_BATCH) return MGEMV_ERR_BATCH;
  if (const int st = check_problem(weights, scale, zero_add, n_out, k, group_size, quant_op, weight_bits)) return st;
  if (x == nullptr || y == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(y) % 2 ||
      reinterpret_cast<uintptr_t>(bias) % 2)
    return MGEMV_ERR_ALIGNMENT;
  if (stride_weights % 16 || stride_x % 8) return MGEMV_ERR_ALIGNMENT;
  int device = 0;
  if (const int st = device_of_stream(static_cast<hipStream_t>(stream), device)) return st;
  DeviceInfo info{};
  if (const int st = device_info(device, info)) return st;

  GemvLaunch g{};
  g.device = device;
  g.weights = static_cast<const uint8_t*>(weights);
  g.scale = reinterpret_cast<const half_t*>(scale);
  g.zero_add = quant_op == MGEMV_FINEGRAINED_SCALE_AND_ZEROS ? reinterpret_cast<const half_t*>(zero_add) : nullptr;
  g.n_out = n_out;
  g.k = k;
  g.group_size = group_size;
  PlanKnobs knobs = knobs_for_element(n_out, k, weight_bits, group_size, m_batch, act, info.num_cus, probe != kProbeNone);
  const int gpr = groups_per_run(group_size, weight_bits);
  // The plan takes a group as long as k for the per-column mode; with scales or zeros by group such a launch may look up four.
  if (!kstat_has_left_over_parts(weight_bits, quant_op == MGEMV_PER_COLUMN_SCALE_ONLY ? 1 : gpr, act)) knobs.split_left_over = false;
  if (batch_count > 1 && !left_over_parts_of_batch(m_batch, num_tiles(n_out), num_ksteps(k, weight_bits), info.num_cus)) knobs.split_left_over = false;  // the bits are the same
  g.plan = plan_launch(n_out, k, weight_bits, m_batch, knobs);
  const bool in_parts = g.plan.parts != 0 && !g.plan.k_stationary;  // a single problem
  if (batch_count > 1 && in_parts)
    g.plan = m_batch == 1 ? plan_of_batch(g.plan, n_out, k, weight_bits, knobs, batch_count)
                          : plan_of_batch_rows(g.plan, m_batch, num_tiles(n_out), info.num_cus, batch_count);
  g.form = unit_form(g.plan, batch_count, info.num_cus);
  if (in_parts && g.plan.parts == 0 && g.form == kOneUnit) g.form = kOneUnitFinitePast;
  g.tail.bias = reinterpret_cast<const half_t*>(bias);
  g.tail.split_k = g.plan.split_k;
  g.tail.num_groups = k / group_size;
  g.tail.flags = g_dequant_flags.load() | (g.plan.stages == 1 ? kSingleStage : 0) | (timed_waits ? kTimelineWaits : 0);
  g.tail.alpha = alpha;
  g.tail.beta = beta;
  g.tail.trace = trace;
  {
    const int sequences = g.plan.workgroups * g.plan.tiles_per_wg;
    g.tail.seq_base = num_tiles(n_out) / sequences;
    g.tail.seq_rem = g.plan.k_stationary && g.plan.parts != 0 ? 0 : num_tiles(n_out) % sequences;  // the rest in parts
  }
  g.tail.stride_weights = stride_weights;
  g.tail.stride_x = stride_x;
  g.tail.stride_scale = stride_scale;
  g.tail.stride_bias = stride_bias;
  g.tail.stride_y = stride_y;
  if (route != nullptr) {  // the two change places (place_problem)
    g.tail.stack = g.weights;
    g.weights = reinterpret_cast<const uint8_t*>(route);
    g.tail.route_extent = route_extent;
  }
  g.grid = dim3((unsigned)(g.plan.wgs_per_xcd * kNumXcd), 1, (unsigned)batch_count);
  g.block = dim3((unsigned)(kWave * g.plan.split_k), (unsigned)g.plan.tiles_per_wg, 1);
  g.stream = static_cast<hipStream_t>(stream);

  if (g.plan.matrix_core) {
    g.x = reinterpret_cast<const half_t*>(x);
    g.tail.y = reinterpret_cast<half_t*>(y);
    g.tail.m_batch = m_batch;
    g.lds = launch_resources(g.plan, weight_bits, m_batch, act).lds_bytes;
    if (g.plan.k_stationary) {
      const size_t stage = kstat_stage_bytes(g.plan.split_k, weight_bits, m_batch, act == kActBf16, g.plan.parts);
      if (g.lds > stage && g.lds - stage >= (size_t)g.plan.tiles_in_sequence * kKSlices * m_batch * kKStationaryParkSlots * 16)
        g.tail.flags |= kParkBehindStage;
      if (probe != kProbeNone) {
        if (probe == kProbeTimeline || !mfma_kstat_probe_exists(weight_bits, quant_op, gpr, act)) return MGEMV_ERR_QUANT_OP;
        return launch_mfma_kstat_probe(g, gpr, probe) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
      }
      return launch_mfma_kstat(g, weight_bits, quant_op, gpr, act) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
    }
    if (probe != kProbeNone) {
      const int rounds = g.plan.staged_rows != 0 ? g.plan.staged_rows / g.plan.tiles_per_wg : 0;
      if (probe == kProbeTimeline || rounds == 0 ||
          !mfma_lds_probe_exists(weight_bits, quant_op, gpr, rounds, act, g.plan.tiles_per_wg))
        return MGEMV_ERR_QUANT_OP;
      return launch_mfma_lds_probe(g, gpr, rounds, probe) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
    }
    if (g.plan.parts != 0) return launch_mfma_parts(g, weight_bits, quant_op, gpr, act) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
    if (g.plan.staged_rows != 0) {
      return launch_mfma_lds(g, weight_bits, quant_op, gpr, g.plan.staged_rows / g.plan.tiles_per_wg, act) == hipSuccess
                 ? MGEMV_OK
                 : MGEMV_ERR_LAUNCH;
    }
    return launch_mfma(g, weight_bits, quant_op, gpr) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
  }
  if (probe != kProbeNone) {
    // measurement builds exist for the headline kernel only: int4, scale and zero, one group per run, one row, fp16
    if (weight_bits != 4 || quant_op != MGEMV_FINEGRAINED_SCALE_AND_ZEROS || gpr != 1 || m_batch != 1 || act != kActF16)
      return MGEMV_ERR_QUANT_OP;
    g.x = reinterpret_cast<const half_t*>(x);
    g.tail.y = reinterpret_cast<half_t*>(y);
    g.lds = (size_t)g.plan.tiles_in_sequence * g.plan.tiles_per_wg * g.plan.split_k * kWave * sizeof(float);
    // every launched wave writes its own row of the trace: the caller's buffer must hold them all
    if (probe == kProbeTimeline &&
        (size_t)g.grid.x * (size_t)(g.plan.split_k * g.plan.tiles_per_wg) > trace_capacity_waves)
      return MGEMV_ERR_SIZE;
    return launch_gemv_probe(g, probe) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
  }
  if (g.plan.parts != 0) {
    g.x = reinterpret_cast<const half_t*>(x);
    g.tail.y = reinterpret_cast<half_t*>(y);
    g.lds = launch_resources(g.plan, weight_bits, m_batch, act).lds_bytes;
    return launch_valu_parts(g, weight_bits, quant_op, gpr, act) == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
  }
  // VALU path: activation rows are processed kMaxValuBatch at a time.
  for (int m0 = 0; m0 < m_batch; m0 += kMaxValuBatch) {
    const int mb = m_batch - m0 < kMaxValuBatch ? m_batch - m0 : kMaxValuBatch;
    g.x = reinterpret_cast<const half_t*>(x) + (size_t)m0 * (size_t)k;
    g.tail.y = reinterpret_cast<half_t*>(y) + (size_t)m0 * (size_t)n_out;
    g.lds = (size_t)g.plan.tiles_in_sequence * g.plan.tiles_per_wg * g.plan.split_k * mb * kWave * sizeof(float);
    if (launch_gemv(g, weight_bits, quant_op, mb, gpr, act) != hipSuccess) return MGEMV_ERR_LAUNCH;
  }
  return MGEMV_OK;
}

int dequantize_any(const void* weights, const uint16_t* scale, const uint16_t* zero_add, uint16_t* out, int n_out,
                   int k, int group_size, int quant_op, int weight_bits, void* stream, int act) {
  if (const int st = check_problem(weights, scale, zero_add, n_out, k, group_size, quant_op, weight_bits)) return st;
  if (out == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(out) % 4) return MGEMV_ERR_ALIGNMENT;
  int device = 0;
  if (const int st = device_of_stream(static_cast<hipStream_t>(stream), device)) return st;
  DeviceInfo info{};
  if (const int st = device_info(device, info)) return st;
  DequantParams p{};
  p.weights = static_cast<const uint8_t*>(weights);
  p.scale = reinterpret_cast<const half_t*>(scale);
  p.zero_add = quant_op == MGEMV_FINEGRAINED_SCALE_AND_ZEROS ? reinterpret_cast<const half_t*>(zero_add) : nullptr;
  p.n_out = n_out;
  p.k = k;
  p.group_size = group_size;
  p.num_groups = k / group_size;
  p.tiles = num_tiles(n_out);
  p.ksteps = num_ksteps(k, weight_bits);
  p.flags = g_dequant_flags.load();
  half_t* const o = reinterpret_cast<half_t*>(out);
  hipStream_t const st = static_cast<hipStream_t>(stream);
  hipError_t e;
  if (act == kActBf16)
    e = weight_bits == 4 ? launch_dequant<4, kActBf16>(p, quant_op, o, st) : launch_dequant<8, kActBf16>(p, quant_op, o, st);
  else
    e = weight_bits == 4 ? launch_dequant<4, kActF16>(p, quant_op, o, st) : launch_dequant<8, kActF16>(p, quant_op, o, st);
  return e == hipSuccess ? MGEMV_OK : MGEMV_ERR_LAUNCH;
}

}  // namespace mgemv

extern "C" {

int mgemv_gemv_batched(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
                       const uint16_t* bias, uint16_t* y, int batch_count, int n_out, int m_batch, int k,
                       int group_size, int quant_op, int weight_bits, int64_t stride_weights, int64_t stride_x,
                       int64_t stride_scale, int64_t stride_bias, int64_t stride_y, void* stream) {
  return mgemv::gemv_any(weights, x, scale, zero_add, bias, y, batch_count, n_out, m_batch, k, group_size, quant_op,
                         weight_bits, stride_weights, stride_x, stride_scale, stride_bias, stride_y, stream,
                         mgemv::kActF16);
}

int mgemv_gemv_batched_bf16(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
                            const uint16_t* bias, uint16_t* y, int batch_count, int n_out, int m_batch, int k,
                            int group_size, int quant_op, int weight_bits, int64_t stride_weights, int64_t stride_x,
                            int64_t stride_scale, int64_t stride_bias, int64_t stride_y, void* stream) {
  return mgemv::gemv_any(weights, x, scale, zero_add, bias, y, batch_count, n_out, m_batch, k, group_size, quant_op,
                         weight_bits, stride_weights, stride_x, stride_scale, stride_bias, stride_y, stream,
                         mgemv::kActBf16);
}

int mgemv_gemv_routed(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
                      const uint16_t* bias, uint16_t* y, const int32_t* route, int route_extent, int batch_count,
                      int n_out, int m_batch, int k, int group_size, int quant_op, int weight_bits,
                      int64_t stride_weights, int64_t stride_x, int64_t stride_scale, int64_t stride_bias,
                      int64_t stride_y, void* stream) {
  if (route == nullptr) return MGEMV_ERR_NULL_POINTER;
  return mgemv::gemv_any(weights, x, scale, zero_add, bias, y, batch_count, n_out, m_batch, k, group_size, quant_op,
                         weight_bits, stride_weights, stride_x, stride_scale, stride_bias, stride_y, stream,
                         mgemv::kActF16, 1.0f, 1.0f, mgemv::kProbeNone, nullptr, 0, false, route, route_extent);
}

int mgemv_gemv_routed_bf16(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
                           const uint16_t* bias, uint16_t* y, const int32_t* route, int route_extent, int batch_count,
                           int n_out, int m_batch, int k, int group_size, int quant_op, int weight_bits,
                           int64_t stride_weights, int64_t stride_x, int64_t stride_scale, int64_t stride_bias,
                           int64_t stride_y, void* stream) {
  if (route == nullptr) return MGEMV_ERR_NULL_POINTER;
  return mgemv::gemv_any(weights, x, scale, zero_add, bias, y, batch_count, n_out, m_batch, k, group_size, quant_op,
                         weight_bits, stride_weights, stride_x, stride_scale, stride_bias, stride_y, stream,
                         mgemv::kActBf16, 1.0f, 1.0f, mgemv::kProbeNone, nullptr, 0, false, route, route_extent);
}

int mgemv_gemv_bf16(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
                    const uint16_t* bias, uint16_t* y, int n_out, int m_batch, int k, int group_size, int quant_op,
                    int weight_bits, void* stream) {
  return mgemv_gemv_batched_bf16(weights, x, scale, zero_add, bias, y, 1, n_out, m_batch, k, group_size, quant_op,
                                 weight_bits, 0, 0, 0, 0, 0, stream);
}

int mgemv_dequantize_bf16(const void* weights, const uint16_t* scale, const uint16_t* zero_add, uint16_t* out, int n_out,
                          int k, int group_size, int quant_op, int weight_bits, void* stream) {
  return mgemv::dequantize_any(weights, scale, zero_add, out, n_out, k, group_size, quant_op, weight_bits, stream,
                               mgemv::kActBf16);
}

int mgemv_gemv(const void* weights, const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add,
               const uint16_t* bias, uint16_t* y, int n_out, int m_batch, int k, int group_size, int quant_op,
               int weight_bits, void* stream) {
  return mgemv_gemv_batched(weights, x, scale, zero_add, bias, y, 1, n_out, m_batch, k, group_size, quant_op,
                            weight_bits, 0, 0, 0, 0, 0, stream);
}

int mgemv_dequantize(const void* weights, const uint16_t* scale, const uint16_t* zero_add, uint16_t* out, int n_out,
                     int k, int group_size, int quant_op, int weight_bits, void* stream) {
  return mgemv::dequantize_any(weights, scale, zero_add, out, n_out, k, group_size, quant_op, weight_bits, stream,
                               mgemv::kActF16);
}

namespace {
int probe_kind(int kind) {
  return kind == MGEMV_PROBE_LOADS_ONLY     ? mgemv::kProbeLoadsOnly
         : kind == MGEMV_PROBE_COMPUTE_ONLY ? mgemv::kProbeComputeOnly
                                            : mgemv::kProbeTimeline;   // with or without the per-unit waits
}
}  // namespace

int mgemv_probe_gemv_rows(int kind, int m_batch, const void* weights, const uint16_t* x, const uint16_t* scale,
                          const uint16_t* zero_add, uint16_t* y, int n_out, int k, int group_size, void* stream) {
  if (kind != MGEMV_PROBE_LOADS_ONLY && kind != MGEMV_PROBE_COMPUTE_ONLY) return MGEMV_ERR_SIZE;
  return mgemv::gemv_any(weights, x, scale, zero_add, nullptr, y, 1, n_out, m_batch, k, group_size,
                         MGEMV_FINEGRAINED_SCALE_AND_ZEROS, 4, 0, 0, 0, 0, 0, stream, mgemv::kActF16, 1.0f, 1.0f,
                         probe_kind(kind), nullptr);
}

int mgemv_probe_gemv(int kind, unsigned long long* trace, size_t trace_capacity_waves, const void* weights,
                     const uint16_t* x, const uint16_t* scale, const uint16_t* zero_add, uint16_t* y, int n_out, int k,
                     int group_size, void* stream) {
  if (kind != MGEMV_PROBE_LOADS_ONLY && kind != MGEMV_PROBE_TIMELINE && kind != MGEMV_PROBE_COMPUTE_ONLY &&
      kind != MGEMV_PROBE_TIMELINE_WAITS)
    return MGEMV_ERR_SIZE;
  if ((kind == MGEMV_PROBE_TIMELINE || kind == MGEMV_PROBE_TIMELINE_WAITS) && (trace == nullptr || reinterpret_cast<uintptr_t>(trace) % 8)) return MGEMV_ERR_NULL_POINTER;
  return mgemv::gemv_any(weights, x, scale, zero_add, nullptr, y, 1, n_out, 1, k, group_size,
                         MGEMV_FINEGRAINED_SCALE_AND_ZEROS, 4, 0, 0, 0, 0, 0, stream, mgemv::kActF16, 1.0f, 1.0f,
                         probe_kind(kind), trace, trace_capacity_waves, kind == MGEMV_PROBE_TIMELINE_WAITS);
}

// gemv/device/gemv_adaptor.h:114-178 as one plain struct.
int mgemv_gemv_arguments(const mgemv_arguments* a, void* stream) {
  if (a == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (a->element != MGEMV_ELEMENT_F16 && a->element != MGEMV_ELEMENT_BF16) return MGEMV_ERR_QUANT_TYPE;
  // The operands are the reference's dense ones; a leading dimension may repeat what the reference
  // passes (mixed_gemv_test.cu:136-140, 153-154) or be 0 = "dense", nothing else.
  const int64_t n = a->n_out, k = a->k;
  if (a->lda != 0 && a->lda != 4 * k && a->lda != k) return MGEMV_ERR_LEADING_DIMENSION;
  if (a->ldb != k && !(a->ldb == 0 && a->m_batch == 1)) return MGEMV_ERR_LEADING_DIMENSION;
  if (a->ld_scale != 0 && a->ld_scale != n) return MGEMV_ERR_LEADING_DIMENSION;
  if (a->ld_zero != 0 && a->ld_zero != n) return MGEMV_ERR_LEADING_DIMENSION;
  if (a->ldc != 0 && a->ldc != n) return MGEMV_ERR_LEADING_DIMENSION;
  if (a->ldd != 0 && a->ldd != n) return MGEMV_ERR_LEADING_DIMENSION;
  return mgemv::gemv_any(a->weights, a->x, a->scale, a->zero_add, a->bias, a->y, a->batch_count, a->n_out,
                         a->m_batch, a->k, a->group_size, a->quant_op, a->weight_bits, a->batch_stride_weights,
                         a->batch_stride_x, a->batch_stride_scale, a->batch_stride_bias, a->batch_stride_y, stream,
                         a->element == MGEMV_ELEMENT_BF16 ? mgemv::kActBf16 : mgemv::kActF16, a->alpha, a->beta);
}

// host/mixed_gemv.h:60-70 on the GPU: un-preprocessed weights and int8 zero points in host
// memory in, result in host memory out.  Both entry points below share everything but where their
// staging memory comes from.
namespace {

struct HostGemvLayout {
  size_t tiled_bytes, table, off_w, off_x, off_s, off_z, off_b, off_y, total;
  bool has_zero;
};

int host_gemv_layout(int batch, int n_out, int m_batch, int k, int& group_size, const void* weights, const void* x,
                     const void* scale, const void* zero_point, const void* y, bool has_bias, int quant_op, int weight_bits,
                     HostGemvLayout& l) {
  if (batch != 1) return MGEMV_ERR_BATCH;  // host/mixed_gemv.h:77-80
  if (m_batch < 1 || m_batch > MGEMV_MAX_M_BATCH) return MGEMV_ERR_BATCH;
  if (weights == nullptr || x == nullptr || scale == nullptr || y == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (quant_op != MGEMV_PER_COLUMN_SCALE_ONLY && quant_op != MGEMV_FINEGRAINED_SCALE_ONLY &&
      quant_op != MGEMV_FINEGRAINED_SCALE_AND_ZEROS)
    return MGEMV_ERR_QUANT_OP;
  if (weight_bits != 4 && weight_bits != 8) return MGEMV_ERR_QUANT_TYPE;
  l.has_zero = quant_op == MGEMV_FINEGRAINED_SCALE_AND_ZEROS;
  if (l.has_zero && zero_point == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (n_out <= 0 || k <= 0) return MGEMV_ERR_SIZE;
  if (quant_op == MGEMV_PER_COLUMN_SCALE_ONLY) group_size = k;
  if (group_size <= 0 || k % group_size) return MGEMV_ERR_GROUP_SIZE;
  if (n_out % 4) return MGEMV_ERR_ROWS;  // what the preprocessor would refuse (utils/preprocess.h:319-327),
  if (k % 8) return MGEMV_ERR_COLS;      // before any memory is touched
  l.table = (size_t)(k / group_size) * (size_t)n_out;
  const size_t shape[2] = {(size_t)k, (size_t)n_out};
  l.tiled_bytes = mgemv_preprocessed_size(shape, 2, weight_bits == 4 ? MGEMV_W4_A16 : MGEMV_W8_A16);
  // one piece of memory, 256-byte aligned parts
  auto align = [](size_t v) { return (v + 255) / 256 * 256; };
  l.off_w = 0;
  l.off_x = l.off_w + align(l.tiled_bytes);
  l.off_s = l.off_x + align((size_t)m_batch * k * 2);
  l.off_z = l.off_s + align(l.table * 2);
  l.off_b = l.off_z + align(l.has_zero ? l.table * 2 : 0);
  l.off_y = l.off_b + align(has_bias ? (size_t)n_out * 2 : 0);
  l.total = l.off_y + align((size_t)m_batch * n_out * 2);
  return MGEMV_OK;
}

// dev: device staging of l.total bytes; host_stage: host memory laid out the same way, of which the
// weight and zero parts are used.
int host_gemv_staged(const HostGemvLayout& l, uint8_t* dev, uint8_t* host_stage, int n_out, int m_batch, int k,
                     int group_size, const uint8_t* weights, const uint16_t* x, const uint16_t* scale,
                     const int8_t* zero_point, const uint16_t* bias, uint16_t* y, int quant_op, int weight_bits) {
  const size_t shape[2] = {(size_t)k, (size_t)n_out};
  const int quant_type = weight_bits == 4 ? MGEMV_W4_A16 : MGEMV_W8_A16;
  uint8_t* const tiled = host_stage + l.off_w;
  if (const int st = mgemv_preprocess_weights(tiled, weights, shape, 2, MGEMV_COLUMN_MAJOR, quant_type)) return st;
  uint16_t* const zero_add = reinterpret_cast<uint16_t*>(host_stage + l.off_z);
  if (l.has_zero) {
    if (const int st = mgemv_fold_zero_points(zero_add, scale, zero_point, l.table)) return st;  // utils/preprocess.h:94-101
  }
  int st = MGEMV_OK;
  auto up = [&](size_t off, const void* src, size_t bytes) {
    if (st == MGEMV_OK && bytes && hipMemcpy(dev + off, src, bytes, hipMemcpyHostToDevice) != hipSuccess) st = MGEMV_ERR_LAUNCH;
  };
  up(l.off_w, tiled, l.tiled_bytes);
  up(l.off_x, x, (size_t)m_batch * k * 2);
  up(l.off_s, scale, l.table * 2);
  if (l.has_zero) up(l.off_z, zero_add, l.table * 2);
  if (bias) up(l.off_b, bias, (size_t)n_out * 2);
  if (st == MGEMV_OK)
    st = mgemv_gemv(dev + l.off_w, reinterpret_cast<const uint16_t*>(dev + l.off_x),
                    reinterpret_cast<const uint16_t*>(dev + l.off_s),
                    l.has_zero ? reinterpret_cast<const uint16_t*>(dev + l.off_z) : nullptr,
                    bias ? reinterpret_cast<const uint16_t*>(dev + l.off_b) : nullptr,
                    reinterpret_cast<uint16_t*>(dev + l.off_y), n_out, m_batch, k, group_size, quant_op, weight_bits, nullptr);
  // the blocking copy on the null stream is ordered behind the kernel
  if (st == MGEMV_OK && hipMemcpy(y, dev + l.off_y, (size_t)m_batch * n_out * 2, hipMemcpyDeviceToHost) != hipSuccess)
    st = MGEMV_ERR_LAUNCH;
  return st;
}

}  // namespace

int mgemv_host_gemv(int batch, int n_out, int m_batch, int k, int group_size, const uint8_t* weights,
                    const uint16_t* x, const uint16_t* scale, const int8_t* zero_point, const uint16_t* bias,
                    uint16_t* y, int quant_op, int weight_bits) {
  HostGemvLayout l{};
  if (const int st = host_gemv_layout(batch, n_out, m_batch, k, group_size, weights, x, scale, zero_point, y,
                                      bias != nullptr, quant_op, weight_bits, l))
    return st;
  std::vector<uint8_t> host_stage(l.off_b);  // the weight and zero parts are what the host side fills
  uint8_t* dev = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&dev), l.total) != hipSuccess) return MGEMV_ERR_ALLOCATION;
  const int st = host_gemv_staged(l, dev, host_stage.data(), n_out, m_batch, k, group_size, weights, x, scale, zero_point,
                                  bias, y, quant_op, weight_bits);
  (void)hipFree(dev);
  return st;
}

// The allocation-free variant: the same staging in a static device array (one copy per GPU, at
// its own address there) and a static host array.  The array's name is a host-side handle, not a
// device address: host code only ever uses the pointer hipGetSymbolAddress returned for the
// device at hand.
static __device__ __align__(256) unsigned char scratch[MGEMV_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxScratchDevices = 64;
alignas(256) unsigned char g_static_host_stage[MGEMV_STATIC_SCRATCH_BYTES];
unsigned char* g_scratch_of_device[kMaxScratchDevices];  // what hipGetSymbolAddress gave, per device
std::mutex g_static_mutex;                               // one call at a time: the arrays are shared

// The address of `scratch` on the current device (looked up once per device, with it current).
int static_scratch_of_current_device(unsigned char*& ptr) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return MGEMV_ERR_NO_DEVICE;
  if (device < 0 || device >= kMaxScratchDevices) return MGEMV_ERR_NO_DEVICE;
  if (g_scratch_of_device[device] == nullptr) {
    mgemv::DeviceInfo info{};
    if (const int st = mgemv::device_info(device, info)) return st;  // gfx950 only: other devices hold no copy of the array
    unsigned char* p = nullptr;
    if (hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr)
      return MGEMV_ERR_NO_DEVICE;
    g_scratch_of_device[device] = p;
  }
  ptr = g_scratch_of_device[device];
  return MGEMV_OK;
}
}  // namespace

size_t mgemv_static_scratch_bytes_needed(int n_out, int m_batch, int k, int group_size, int quant_op, int weight_bits,
                                         int has_bias) {
  HostGemvLayout l{};
  static const int dummy = 0;  // the layout only asks whether the pointers are there
  if (host_gemv_layout(1, n_out, m_batch, k, group_size, &dummy, &dummy, &dummy, &dummy, &dummy, has_bias != 0, quant_op,
                       weight_bits, l))
    return 0;
  return l.total;
}

int mgemv_host_gemv_static(int batch, int n_out, int m_batch, int k, int group_size, const uint8_t* weights,
                           const uint16_t* x, const uint16_t* scale, const int8_t* zero_point, const uint16_t* bias,
                           uint16_t* y, int quant_op, int weight_bits) {
  HostGemvLayout l{};
  if (const int st = host_gemv_layout(batch, n_out, m_batch, k, group_size, weights, x, scale, zero_point, y,
                                      bias != nullptr, quant_op, weight_bits, l))
    return st;
  if (l.total > MGEMV_STATIC_SCRATCH_BYTES) return MGEMV_ERR_SCRATCH_SIZE;
  std::lock_guard<std::mutex> lock(g_static_mutex);
  unsigned char* dev = nullptr;
  if (const int st = static_scratch_of_current_device(dev)) return st;
  return host_gemv_staged(l, dev, g_static_host_stage, n_out, m_batch, k, group_size, weights, x, scale, zero_point, bias, y,
                          quant_op, weight_bits);
}

int mgemv_set_launch_override(int split_k_waves, int tiles_per_workgroup, int tiles_per_wave, int max_workgroups) {
  if (split_k_waves < 0 || tiles_per_workgroup < 0 || tiles_per_wave < 0 || max_workgroups < 0) return MGEMV_ERR_SIZE;
  if (tiles_per_wave != 0 && tiles_per_wave != 1 && tiles_per_wave != 2 && tiles_per_wave != 4) return MGEMV_ERR_SIZE;
  mgemv::g_override_split_k.store(split_k_waves);
  mgemv::g_override_tiles_per_wg.store(tiles_per_workgroup);
  mgemv::g_override_tiles_per_wave.store(tiles_per_wave);
  mgemv::g_override_workgroups.store(max_workgroups);
  return MGEMV_OK;
}

int mgemv_set_matrix_core_threshold(int min_m_batch) {
  if (min_m_batch < 0 || min_m_batch > MGEMV_MAX_M_BATCH + 1) return MGEMV_ERR_BATCH;
  mgemv::g_matrix_core_min_batch.store(min_m_batch);
  return MGEMV_OK;
}

int mgemv_set_matrix_core_variant(int variant) {
  if (variant != MGEMV_MATRIX_CORE_AUTO && variant != MGEMV_MATRIX_CORE_REGISTER_OPERAND &&
      variant != MGEMV_MATRIX_CORE_LDS_STAGED && variant != MGEMV_MATRIX_CORE_K_STATIONARY)
    return MGEMV_ERR_SIZE;
  mgemv::g_matrix_core_variant.store(variant);
  return MGEMV_OK;
}

int mgemv_set_prefetch_stages(int stages) {
  if (stages < 0 || stages > 2) return MGEMV_ERR_SIZE;
  mgemv::g_override_stages.store(stages);
  return MGEMV_OK;
}

int mgemv_set_dequant_form(int form) {
  if (form != MGEMV_DEQUANT_AUTO && form != MGEMV_DEQUANT_EXACT_INTEGER) return MGEMV_ERR_SIZE;
  mgemv::g_dequant_flags.store(form == MGEMV_DEQUANT_EXACT_INTEGER ? mgemv::kExactIntegerFormOnly : 0);
  return MGEMV_OK;
}

namespace {
int check_tuned_key(int n_out, int k, int weight_bits, int group_size, int m_batch) {
  if (weight_bits != 4 && weight_bits != 8) return MGEMV_ERR_QUANT_TYPE;
  if (n_out <= 0 || k <= 0) return MGEMV_ERR_SIZE;
  if (group_size < 0) return MGEMV_ERR_GROUP_SIZE;
  if (m_batch < 1 || m_batch > MGEMV_MAX_M_BATCH) return MGEMV_ERR_BATCH;
  return MGEMV_OK;
}
}  // namespace

int mgemv_tuned_plan_set(const mgemv_tuned_plan* plan) {
  if (plan == nullptr) return MGEMV_ERR_NULL_POINTER;
  const int st = check_tuned_key(plan->n_out, plan->k, plan->weight_bits, plan->group_size, plan->m_batch);
  if (st != MGEMV_OK) return st;
  if (plan->split_k_waves < 0 || plan->tiles_per_workgroup < 0 || plan->max_workgroups < 0) return MGEMV_ERR_SIZE;
  if (plan->stages < 0 || plan->stages > 2) return MGEMV_ERR_SIZE;
  if (plan->element != MGEMV_ELEMENT_F16 && plan->element != MGEMV_ELEMENT_BF16) return MGEMV_ERR_QUANT_TYPE;
  const int t = plan->tiles_per_wave;
  if (t != 0 && t != 1 && t != 2 && t != 4) return MGEMV_ERR_SIZE;
  if (plan->kernel < MGEMV_KERNEL_AUTO || plan->kernel > MGEMV_KERNEL_MATRIX_CORE_K_STATIONARY) return MGEMV_ERR_SIZE;
  const mgemv::PlanKnobs kn = mgemv::knobs_of_plan(*plan);
  std::lock_guard<std::mutex> lock(mgemv::g_tuned_mutex);
  mgemv::g_tuned_plans[mgemv::PlanKey{plan->n_out, plan->k, plan->weight_bits, plan->group_size, plan->m_batch,
                                      plan->element}] = kn;
  mgemv::g_tuned_count.store((int)mgemv::g_tuned_plans.size());
  return MGEMV_OK;
}

int mgemv_tuned_plan_erase(const mgemv_tuned_plan* plan) {
  if (plan == nullptr) return MGEMV_ERR_NULL_POINTER;
  std::lock_guard<std::mutex> lock(mgemv::g_tuned_mutex);
  mgemv::g_tuned_plans.erase(
      mgemv::PlanKey{plan->n_out, plan->k, plan->weight_bits, plan->group_size, plan->m_batch, plan->element});
  mgemv::g_tuned_count.store((int)mgemv::g_tuned_plans.size());
  return MGEMV_OK;
}

int mgemv_set_default_plans(int enable) {
  mgemv::g_default_plans_enabled.store(enable != 0 ? 1 : 0);
  return MGEMV_OK;
}

int mgemv_default_plan_count(void) { return mgemv::default_plan_count(); }

int mgemv_tuned_plan_clear(void) {
  std::lock_guard<std::mutex> lock(mgemv::g_tuned_mutex);
  mgemv::g_tuned_plans.clear();
  mgemv::g_tuned_count.store(0);
  return MGEMV_OK;
}

int mgemv_tuned_plan_count(void) { return mgemv::g_tuned_count.load(); }

namespace {
int query_launch_any(int n_out, int m_batch, int k, int weight_bits, int group_size, int act, int out[8],
                     int num_cus = mgemv::kNumCus);
}

int mgemv_query_launch_for(int n_out, int m_batch, int k, int weight_bits, int group_size, int element,
                           int num_compute_units, int out[12]) {
  if (element != MGEMV_ELEMENT_F16 && element != MGEMV_ELEMENT_BF16) return MGEMV_ERR_QUANT_TYPE;
  if (num_compute_units < 1 || num_compute_units > 4096) return MGEMV_ERR_SIZE;
  const int act = element == MGEMV_ELEMENT_BF16 ? mgemv::kActBf16 : mgemv::kActF16;
  if (const int st = query_launch_any(n_out, m_batch, k, weight_bits, group_size, act, out, num_compute_units)) return st;
  const mgemv::LaunchPlan lp = mgemv::plan_launch(
      n_out, k, weight_bits, m_batch, mgemv::knobs_for_element(n_out, k, weight_bits, group_size, m_batch, act, num_compute_units));
  const mgemv::LaunchResources r = mgemv::launch_resources(lp, weight_bits, m_batch, act);
  out[8] = (int)r.lds_bytes;
  out[9] = r.max_threads;
  out[10] = lp.stages;
  out[11] = r.launches;
  return MGEMV_OK;
}

int mgemv_plan_coverage(int n_out, int m_batch, int k, int weight_bits, int group_size, int element,
                        int num_compute_units, int64_t out[8]) {
  using namespace mgemv;
  if (out == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (element != MGEMV_ELEMENT_F16 && element != MGEMV_ELEMENT_BF16) return MGEMV_ERR_QUANT_TYPE;
  if (num_compute_units < 1 || num_compute_units > 4096) return MGEMV_ERR_SIZE;
  if (const int st = check_tuned_key(n_out, k, weight_bits, group_size, m_batch)) return st;
  const int act = element == MGEMV_ELEMENT_BF16 ? kActBf16 : kActF16;
  const LaunchPlan lp = plan_launch(n_out, k, weight_bits, m_batch,
                                    knobs_for_element(n_out, k, weight_bits, group_size, m_batch, act, num_compute_units));
  const LaunchResources res = launch_resources(lp, weight_bits, m_batch, act);
  const int tiles = num_tiles(n_out), ksteps = num_ksteps(k, weight_bits);
  const int grid = lp.wgs_per_xcd * kNumXcd;
  const int sequences = lp.workgroups * lp.tiles_per_wg;
  const bool left_over_parts = lp.k_stationary && lp.parts != 0;
  const int seq_base = tiles / sequences, seq_rem = left_over_parts ? 0 : tiles % sequences;  // as gemv_any passes them
  const bool multi = (!lp.matrix_core || lp.k_stationary) && lp.tiles_in_sequence > 1;
  const int rows = m_batch < kMaxValuBatch ? m_batch : kMaxValuBatch;
  const int parts = lp.parts > 0 ? lp.parts : 1;
  std::vector<int> covered((size_t)tiles * parts, 0);  // k steps of each tile, or part of one
  std::vector<char> block_seen((size_t)lp.workgroups, 0);
  int64_t idle_waves = 0, busy_waves = 0, max_span = 0, max_lds = 0, bad_ranges = 0, max_units = 0;
  for (int block = 0; block < grid; ++block) {
    const int wg = logical_workgroup_of(block, lp.wgs_per_xcd);
    if (wg >= lp.workgroups) continue;  // the kernels leave at this test
    if (block_seen[(size_t)wg]++) ++bad_ranges;   // two blocks with one logical id
    for (int ty = 0; ty < lp.tiles_per_wg; ++ty) {
      for (int kw = 0; kw < lp.split_k; ++kw) {
        const PartWork part = part_wave_work(parts, wg, kw, lp.steps_per_wave, ksteps);
        const WaveWork w = lp.parts != 0 && !lp.k_stationary ? WaveWork{part.tile, part.tile < tiles ? 1 : 0, part.ks_begin, part.units}
                           : lp.matrix_core && !lp.k_stationary
                               ? (lp.staged_rows != 0
                                      ? staged_wave_work(wg, ty, kw, lp.tiles_per_wg, tiles, lp.steps_per_wave, ksteps)
                                      : mfma_wave_work(lp.tiles_per_wave, wg, ty, kw, lp.tiles_per_wg, tiles,
                                                       lp.steps_per_wave, ksteps))
                               : valu_wave_work(multi, wg, ty, kw, lp.tiles_per_wg, seq_base, seq_rem, tiles,
                                                lp.steps_per_wave, ksteps);
        if (w.units <= 0) ++bad_ranges;  // every kernel relies on each wave along k having units
        // whole units, a column for every row and k step
        if (parts * m_batch > kTileRows || (!lp.k_stationary && lp.steps_per_wave % parts != 0)) ++bad_ranges;
        if (left_over_parts) {  // the wave's unit of its workgroup's part of a left-over tile
          const int tile = seq_base * lp.workgroups + wg / parts, unit = kstat_tail_unit(kw, lp.split_k);
          if (tile < tiles && unit * parts < ksteps)
            covered[(size_t)tile * parts + wg % parts] += ksteps - unit * parts < parts ? ksteps - unit * parts : parts;
        }
        if (w.tiles <= 0 || w.units <= 0) {
          ++idle_waves;
          continue;
        }
        ++busy_waves;
        if (w.tile_begin < 0 || w.tile_begin + w.tiles > tiles || w.ks_begin < 0 || w.ks_begin + w.units > ksteps) {
          ++bad_ranges;
          continue;
        }
        for (int t = 0; t < w.tiles; ++t)
          for (int q = 0; q < parts; ++q)
            if (lp.k_stationary || q == part.part || lp.parts == 0) covered[(size_t)(w.tile_begin + t) * parts + q] += w.units;
        // the bytes one weight descriptor spans: tiles are ksteps units apart
        const int64_t span = (int64_t)(w.tiles - 1) * ksteps * kUnitBytes + (int64_t)w.units * kUnitBytes;
        max_span = span > max_span ? span : max_span;
        const int64_t walk_units = (int64_t)w.tiles * w.units;
        max_units = walk_units > max_units ? walk_units : max_units;
        if (!lp.matrix_core) {
          // last float this wave parks for the combine (tile t of its walk at t * park_stride)
          const int64_t park_stride = (int64_t)lp.tiles_per_wg * lp.split_k * rows * kWave;
          const int64_t last = (int64_t)(multi ? w.tiles - 1 : 0) * park_stride +
                               ((int64_t)(ty * lp.split_k + kw) * rows + (rows - 1)) * kWave + (kWave - 1);
          max_lds = (last + 1) * 4 > max_lds ? (last + 1) * 4 : max_lds;
        }
      }
    }
  }
  int64_t wrong = 0;
  for (const int steps : covered) wrong += steps != ksteps;
  out[0] = wrong;                 // tiles whose k steps are not covered exactly once
  out[1] = bad_ranges;            // waves with a range outside the problem or without units, duplicate workgroup ids
  out[2] = max_span;              // most bytes behind one weight descriptor
  out[3] = max_lds;               // VALU kernel: bytes of LDS up to the last parked partial sum
  out[4] = (int64_t)res.lds_bytes;
  out[5] = busy_waves;
  out[6] = idle_waves;
  out[7] = max_units;             // most units any wave computes
  return MGEMV_OK;
}

int mgemv_probe_unit_form(int n_out, int m_batch, int k, int weight_bits, int group_size, int element, int batch_count,
                          int num_compute_units, int* form) {
  using namespace mgemv;
  if (form == nullptr) return MGEMV_ERR_NULL_POINTER;
  if (element != MGEMV_ELEMENT_F16 && element != MGEMV_ELEMENT_BF16) return MGEMV_ERR_QUANT_TYPE;
  if (num_compute_units < 1 || num_compute_units > 4096) return MGEMV_ERR_SIZE;
  if (batch_count < 1 || batch_count > 65535) return MGEMV_ERR_BATCH;
  if (const int st = check_tuned_key(n_out, k, weight_bits, group_size, m_batch)) return st;
  const int act = element == MGEMV_ELEMENT_BF16 ? kActBf16 : kActF16;
  // a single row on whole tiles, as the measurement builds have it
  const LaunchPlan lp = plan_launch(n_out, k, weight_bits, m_batch,
                                    knobs_for_element(n_out, k, weight_bits, group_size, m_batch, act, num_compute_units, m_batch == 1));
  *form = unit_form(lp, batch_count, num_compute_units);
  return MGEMV_OK;
}

int mgemv_query_launch(int n_out, int m_batch, int k, int weight_bits, int group_size, int out[8]) {
  return query_launch_any(n_out, m_batch, k, weight_bits, group_size, mgemv::kActF16, out);
}

int mgemv_query_launch_bf16(int n_out, int m_batch, int k, int weight_bits, int group_size, int out[8]) {
  return query_launch_any(n_out, m_batch, k, weight_bits, group_size, mgemv::kActBf16, out);
}

namespace {
int query_launch_any(int n_out, int m_batch, int k, int weight_bits, int group_size, int act, int out[8], int num_cus) {
  if (out == nullptr) return MGEMV_ERR_NULL_POINTER;
  const int st = check_tuned_key(n_out, k, weight_bits, group_size, m_batch);
  if (st != MGEMV_OK) return st;
  const mgemv::LaunchPlan lp = mgemv::plan_launch(
      n_out, k, weight_bits, m_batch, mgemv::knobs_for_element(n_out, k, weight_bits, group_size, m_batch, act, num_cus));
  out[0] = lp.wgs_per_xcd * mgemv::kNumXcd;
  out[1] = lp.threads;
  out[2] = lp.split_k;
  out[3] = lp.tiles_per_wg;
  out[4] = lp.steps_per_wave;
  out[5] = !lp.matrix_core ? 0 : lp.k_stationary ? 3 : lp.staged_rows != 0 ? 2 : 1;
  out[6] = lp.tiles_per_wave;
  out[7] = lp.tiles_in_sequence;
  return MGEMV_OK;
}
}  // namespace

}  // extern "C"
