// Shared by the kernels of this library and their launchers: launch constants, the kernel
// argument block, small device helpers, and the host-side description of a launch.
#ifndef MIXED_GEMV_AMD_KERNEL_COMMON_H_
#define MIXED_GEMV_AMD_KERNEL_COMMON_H_

#include <hip/hip_runtime.h>

#include "device_math.h"
#include "mixed_gemv.h"
#include "mixed_gemv_probes.h"
#include "tile_layout.h"

namespace mgemv {

constexpr int kWave = 64;
constexpr int kMaxWavesPerWorkgroup = 16;
constexpr int kMaxWavesPerWideWorkgroup = 8;  // VALU kernel with 3-4 activation rows: 256 VGPRs per wave
constexpr int kMaxWavesPerMfmaWorkgroup = 8;  // leaves each wave of the matrix-core kernel 256 VGPRs
constexpr int kNumXcd = 8;
constexpr int kNumCus = 256;
constexpr int kKStationaryParkSlots = kMaxWavesPerWorkgroup + 1;  // k-stationary matrix-core kernel: entries of 16 bytes per block of partial sums
constexpr int kMaxKStationaryLds = 128 * 1024;  // most LDS the k-stationary matrix-core kernel parks partial sums in
constexpr int kKStationaryZeroBytes = 256;  // ... with bf16 operands: zeros, a k run of the operand of a batch row that does not exist
constexpr int kMaxKStationaryBf16Lds = 160 * 1024 - kKStationaryZeroBytes;  // ... most LDS its activation rows and partial sums take together
constexpr int kKStationaryStagedBytes = kMaxWavesPerWorkgroup * 4;  // ... with left-over tiles in parts: a word for each wave
constexpr int kValuPartsSumsAtOnce = 16;  // VALU kernel for parts of tiles: units whose sums are added up at a time
constexpr int kMaxValuBatch = 4;  // activation rows handled per launch by the VALU kernel
constexpr int kExactIntegerFormOnly = 1;  // GemvTail::flags: never take the short int4 dequantiser
constexpr int kSingleStage = 2;           // GemvTail::flags: no load in flight while a unit is computed (VALU kernel)
constexpr int kParkBehindStage = 16;      // GemvTail::flags, k-stationary matrix-core kernel: the partial sums have LDS of their own behind the activation stages
constexpr int kTimelineWaits = 8;         // GemvTail::flags, timeline probe: time the wait in front of every unit as well
constexpr int kTimelineWordsPerWave = MGEMV_PROBE_TIMELINE_WORDS;  // 64-bit words the timeline probe writes per wave
constexpr int kProbeNone = 0, kProbeLoadsOnly = 1, kProbeTimeline = 2, kProbeComputeOnly = 3;  // measurement builds of the VALU kernel

// Kernel arguments.  The first ten (four pointers and six 32-bit words, 14 dwords) are what a
// wave needs to address its first loads, and they are preloaded into SGPRs (build flag
// -amdgpu-kernarg-preload-count=14); everything else sits in GemvTail.
struct GemvTail {
  const half_t* bias;
  half_t* y;
  int split_k;         // waves of a workgroup that share one tile (blockDim.x / 64)
  int m_batch;         // activation rows (matrix-core kernel)
  int num_groups;      // k / group_size (1 in per-column mode): extent of the scale / zero tables
  int flags;           // kExactIntegerFormOnly | kSingleStage
  // Routed launch: problem b takes weights, scales, zeros and bias of entry route[b] of the stack; route itself is the launch's
  // `weights` argument (place_problem).  From here to stride_scale: one 64-byte line of the arguments.
  const uint8_t* stack;  // the weights of entry 0; null: not routed
  int route_extent;    // entries in the stack: a problem routed outside [0, route_extent) is left alone
  int seq_base;        // VALU kernel: tiles / sequences ...
  long long stride_weights, stride_x, stride_scale, stride_bias, stride_y;  // per batch problem
  float alpha, beta;   // epilogue: y = alpha * acc + beta * bias (gemv/device/gemv_adaptor.h:123, epilogue{alpha, beta})
  int seq_rem;         // ... and tiles % sequences (the first seq_rem sequences get one tile more)
  unsigned long long* trace;  // timeline probe: kTimelineWordsPerWave words per wave, else unused
};

// Scalar view of one problem inside a kernel.
struct Problem {
  const uint8_t* weights;
  const half_t* x;
  const half_t* scale;
  const half_t* zero_add;
  int n_out;
  int k;
  int ksteps;          // ceil(k / kStepK)
  int steps_per_wave;  // units per wave
  int workgroups;      // logical workgroups = ceil(tiles / tiles_per_wg)
  int wgs_per_xcd;     // ceil(workgroups / 8); gridDim.x = 8 * wgs_per_xcd
  int group_size;
  int tiles_per_wg;    // blockDim.y
};

constexpr uint32_t pack_steps(int ksteps, int steps_per_wave) { return (uint32_t)ksteps | ((uint32_t)steps_per_wave << 16); }
// group size in bits 0-23, tiles per workgroup in bits 24-30, bit 31: the launch is routed (GemvTail::stack)
constexpr uint32_t kRoutedLaunch = 0x80000000u;
constexpr uint32_t pack_group(int group_size, int tiles_per_wg, bool routed) {
  return (uint32_t)group_size | ((uint32_t)tiles_per_wg << 24) | (routed ? kRoutedLaunch : 0u);
}
constexpr int tiles_per_wg_of(uint32_t packed_group) { return (int)((packed_group >> 24) & 0x7fu); }

// ---------------------------------------------------------------------------------------------
// Which part of the problem a wave works on.  Plain integer functions, compiled for the device
// (the kernels call them) and for the host (which replays them over a whole grid to check that a
// launch plan covers every tile and k step exactly once).
// ---------------------------------------------------------------------------------------------

// Workgroups are handed to the 8 XCDs round-robin by linear id.  Neighbouring tiles read
// neighbouring 32-byte pieces of the same scale/zero cache lines, so give each XCD (and its
// private L2) a contiguous range of tiles instead of every eighth one.
__host__ __device__ __forceinline__ int logical_workgroup_of(int block, int wgs_per_xcd) {
  const int xcd = block % kNumXcd;
  const int slot = block / kNumXcd;
  return xcd * wgs_per_xcd + slot;
}

struct WaveWork {
  int tile_begin, tiles;  // tiles tile_begin .. tile_begin + tiles - 1 (tiles may be 0)
  int ks_begin, units;    // k steps ks_begin .. ks_begin + units - 1 of each of them (units may be <= 0)
};

// k range of the kw-th wave along k.
__host__ __device__ __forceinline__ void wave_k_range(WaveWork& w, int kw, int steps_per_wave, int ksteps) {
  w.ks_begin = kw * steps_per_wave;
  const int end = w.ks_begin + steps_per_wave < ksteps ? w.ks_begin + steps_per_wave : ksteps;
  w.units = end - w.ks_begin;
}

// VALU kernel.  The tiles are dealt out evenly, in contiguous runs, to the (workgroups x
// tiles_per_wg) tile sequences of the launch (multi: sequence s takes seq_base tiles, the first
// seq_rem sequences one more); the split_k waves of a sequence walk its tiles together, each on
// its own part of k.  Without walks (multi false) sequence s is tile s.
__host__ __device__ __forceinline__ WaveWork valu_wave_work(bool multi, int wg, int ty, int kw, int tiles_per_wg,
                                                            int seq_base, int seq_rem, int tiles, int steps_per_wave,
                                                            int ksteps) {
  WaveWork w;
  const int seq = wg * tiles_per_wg + ty;
  w.tile_begin = multi ? seq * seq_base + (seq < seq_rem ? seq : seq_rem) : seq;
  w.tiles = multi ? seq_base + (seq < seq_rem ? 1 : 0) : (seq < tiles ? 1 : 0);
  wave_k_range(w, kw, steps_per_wave, ksteps);
  return w;
}

// Register-operand matrix-core kernel: a wave takes tiles_per_wave consecutive tiles.
__host__ __device__ __forceinline__ WaveWork mfma_wave_work(int tiles_per_wave, int wg, int ty, int kw, int tiles_per_wg,
                                                            int tiles, int steps_per_wave, int ksteps) {
  WaveWork w;
  w.tile_begin = (wg * tiles_per_wg + ty) * tiles_per_wave;
  const int left = tiles - w.tile_begin;
  w.tiles = left <= 0 ? 0 : left < tiles_per_wave ? left : tiles_per_wave;
  wave_k_range(w, kw, steps_per_wave, ksteps);
  return w;
}

// LDS-staged matrix-core kernel: one tile per wave; a wave past the last tile has no tile of
// its own (it still stages activation rows and meets the barriers).
__host__ __device__ __forceinline__ WaveWork staged_wave_work(int wg, int ty, int kw, int tiles_per_wg, int tiles,
                                                              int steps_per_wave, int ksteps) {
  WaveWork w;
  w.tile_begin = wg * tiles_per_wg + ty;
  w.tiles = w.tile_begin < tiles ? 1 : 0;
  wave_k_range(w, kw, steps_per_wave, ksteps);
  return w;
}

// Part-tile kernels: a workgroup takes 16 / parts rows of one tile, a wave a range of whole units of `parts` k steps.
struct PartWork {
  int tile, part, ks_begin, units;  // units: k steps, the last unit of the reduction may be short
};
__host__ __device__ __forceinline__ PartWork part_wave_work(int parts, int wg, int kw, int steps_per_wave, int ksteps) {
  WaveWork w;
  wave_k_range(w, kw, steps_per_wave, ksteps);
  return PartWork{wg / parts, wg % parts, w.ks_begin, w.units};
}

// K-stationary kernel with left-over tiles split into parts: which unit of `parts` k steps of its workgroup's part a wave takes (one
// past the last: none).  The waves are dealt out to the four SIMDs in turn; the first units go to those that have a wave less.
__host__ __device__ __forceinline__ int kstat_tail_unit(int kw, int waves) {
  const int unit = kw - waves % 4;
  return unit < 0 ? unit + waves : unit;
}

__device__ __forceinline__ int logical_workgroup(const Problem& p) {
  return logical_workgroup_of((int)blockIdx.x, p.wgs_per_xcd);
}

// Where the operands of problem blockIdx.z begin (gemv/kernel/mixed_gemv.h:140-149, 222-223): moves the pointers of p, gives the
// entry whose weights, scales, zeros and bias it takes (x and y stay with the problem), or false: routed outside the stack.
// The way to the first weight of a routed launch was three scalar loads one behind the other, each a miss of the cold cache: the
// route's address, the entry, the strides.  The route's address is a preloaded argument now (the weights' is not, which needs
// the entry first), and the rest is requested with the entry.  8 of 64 matrices of 1408x2048 4.63 us / 4.34; 0.93-0.99 of the time on 40
// routed launches of random shapes.
__device__ __forceinline__ bool place_problem(Problem& p, const GemvTail& tail, uint32_t packed_group, long long& owner) {
  const long long batch = blockIdx.z;
  owner = batch;
  if ((blockIdx.z | (packed_group & kRoutedLaunch)) == 0) return true;  // one test on the way of an unbatched launch
  long long stride_weights = tail.stride_weights, stride_x = tail.stride_x, stride_scale = tail.stride_scale;
  bool there = true;
  if ((packed_group & kRoutedLaunch) != 0) {
    typedef const __attribute__((address_space(4))) int* Route;
    int entry = ((Route)p.weights)[batch], extent = tail.route_extent;
    const uint8_t* stack = tail.stack;
    // (in front of the first use of any of them, or the compiler requests the strides behind the test of the entry)
    asm volatile("" : "+s"(entry), "+s"(extent), "+s"(stack), "+s"(stride_weights), "+s"(stride_x), "+s"(stride_scale));
    there = (unsigned)entry < (unsigned)extent;
    owner = entry;
    p.weights = stack;
  }
  p.weights += owner * stride_weights;
  p.x += batch * stride_x;
  p.scale += owner * stride_scale;
  p.zero_add += owner * stride_scale;  // only dereferenced in scale+zero mode
  return there;
}

// Group index of reduction position k_index (host/mixed_gemv.h:88), clamped to the last
// group for the padded positions past k.
// GROUPS_PER_RUN 1 or 2: the group size divides the k step, so it is a power of two.  4: any size; launches of that kind look
// four groups up per unit.  Group sizes are multiples of 32, so the quotient is that of whole 32s, at most 2^21: in fp32,
// (q + 1/2) / d lies at least 1/(2 d) from the next integer, and its error is at most 3/8 of 1/d.  Five instructions where an
// integer division takes 25 (groups of 96: 28672x8064 at 1 / 4 rows 31.5 / 31.6 us, was 34.6 / 34.2; 4096x4128, one row, 6.0 / 6.6).
template <int GROUPS_PER_RUN>
__device__ __forceinline__ int group_of(const Problem& p, int k_index) {
  k_index = k_index < p.k ? k_index : p.k - 1;
  const bool pow2 = (p.group_size & (p.group_size - 1)) == 0;
  if (GROUPS_PER_RUN != 4 || pow2) return k_index >> __builtin_ctz((unsigned)p.group_size);
  return (int)(((float)(k_index >> 5) + 0.5f) * __builtin_amdgcn_rcpf((float)(p.group_size >> 5)));
}

// 16-bit buffer load into the low half of a 32-bit register.  The upper half is left
// unspecified on purpose: zero-extending it would be a VALU instruction on the loaded value,
// and the compiler places that instruction -- and the wait for the data -- next to the load,
// in front of the loads that should be issued behind it.
__device__ __forceinline__ uint32_t load_b16_low(__amdgpu_buffer_rsrc_t rsrc, int voffset) {
  const uint16_t bits = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, voffset, 0, kCacheDefault);
  half2_t v;  // element 1 deliberately not set
  v[0] = __builtin_bit_cast(half_t, bits);
  return as_u32(v);
}
__device__ __forceinline__ uint32_t load_half_bits(const half_t* p) {
  return (uint32_t)*reinterpret_cast<const uint16_t*>(p);
}
__device__ __forceinline__ half2_t splat_low(uint32_t bits) {
  const half_t h = __builtin_bit_cast(half_t, (uint16_t)bits);
  return half2_t{h, h};
}

// The last k step of a reduction may be short.  Activations past it are zero, but an infinite scale (there the last group's, or the
// row's) or zero point times zero is not: groups of a lane's run that lie past it take finite ones, of the short form's range.  k_run:
// first reduction index of the run; group_k: from a group to the next.
template <int ACT>
constexpr uint32_t kAnyScale = ACT == kActBf16 ? 0x3c00u : 0x2000u;  // 2^-7
template <int ACT, int GROUPS>
__device__ __forceinline__ void finite_past_reduction(uint32_t (&s)[GROUPS], uint32_t (&z)[GROUPS], int k_run, int group_k, int k) {
#pragma unroll
  for (int gi = 0; gi < GROUPS; ++gi) {
    const bool past = k_run + gi * group_k >= k;
    s[gi] = past ? kAnyScale<ACT> : s[gi];
    z[gi] = past ? 0u : z[gi];
  }
}

struct ScaleTables {
  __amdgpu_buffer_rsrc_t scale, zero;
};

// True when the scales of all lanes and groups of the unit permit the short form; wave-uniform, so that the choice costs
// one scalar branch per unit.  int4 weights with bf16 scales: short4 is what the short form takes, prepared here, so that
// the units behind the branch are the same code for both kinds of range.  28672x8192, groups of 128 with zeros, at 1 / 4 rows:
// scales of the unmoved range 29.1 / 30.3 us, of any other 12 binades 30.0 / 31.0 (with one range per wave, set around its
// first lane's scale, that lane decided, and most such waves took the general form: 50.4 / 49.4); general form 53.0 / 52.0.
// (A third form for all positive scales -- the products in fp32, fused, 35.7 / 35.9 -- costs the others 0.7 %, up to 2.7 %
// with 16 rows, in registers.)
template <int BITS, int ACT, int GROUPS>
__device__ __forceinline__ bool wave_takes_short_form(const uint32_t (&scale_bits)[GROUPS], Int4ScaleBf16 (&short4)[GROUPS]) {
  auto all_within = [&](uint32_t first, uint32_t past) {
    bool ok = true;
#pragma unroll
    for (int gi = 0; gi < GROUPS; ++gi) ok = ok && (scale_bits[gi] & 0xffffu) - first < past - first;
    return __builtin_amdgcn_ballot_w64(!ok) == 0;
  };
  if constexpr (ACT != kActBf16) return all_within(kShortF16First, kShortF16Past);
  if constexpr (BITS == 8) return all_within(kShortBf16Int8First, kShortBf16Int8Past);
#pragma unroll
  for (int gi = 0; gi < GROUPS; ++gi) short4[gi] = Int4ScaleBf16{bf16_low_to_f32(scale_bits[gi]), kNoShift};
  if (all_within(kShortBf16Int4First, kShortBf16Int4Past)) return true;
  // other magnitudes: for every four rows and group the 12 binades from their smallest scale on
  bool ok = true;
#pragma unroll
  for (int gi = 0; gi < GROUPS; ++gi) {
    const uint32_t exponent = (scale_bits[gi] & 0xffffu) >> 7;  // (with the sign: negative scales are beyond the largest)
    uint32_t first = exponent;
    first = min(first, (uint32_t)__builtin_amdgcn_mov_dpp((int)first, 0xb1, 0xf, 0xf, true));  // quad_perm 1 0 3 2
    first = min(first, (uint32_t)__builtin_amdgcn_mov_dpp((int)first, 0x4e, 0xf, 0xf, true));  // quad_perm 2 3 0 1
    first = min(first, kShortBf16Int4FirstExponent + kShortBf16MaxShift);
    ok = ok && first >= kShortBf16Int4FirstExponent + kShortBf16MinShift && exponent - first < kShortBf16Int4Binades;
    const int shift = (int)(first - kShortBf16Int4FirstExponent);
    short4[gi].s = __builtin_bit_cast(float, (scale_bits[gi] << 16) - ((uint32_t)shift << 23));
    const uint32_t power = (uint32_t)(15 + shift) << 10;
    short4[gi].power = power | power << 16;
  }
  return __builtin_amdgcn_ballot_w64(!ok) == 0;
}

// Epilogue value before the final rounding: alpha * acc + beta * bias in fp32, the outer
// multiply-add fused -- what the reference's LinearCombination computes (alpha * accumulator +
// source, epilogue/threadblock/epilogue.h:64, 93; one `a * b + c` per element, which nvcc
// contracts).  With alpha = beta = 1 this is the single rounded fp32 add of
// host/mixed_gemv.h:102-103, bit for bit, and without a bias it adds +0 as the reference does.
__device__ __forceinline__ float epilogue_value(const GemvTail& tail, float acc, bool has_bias, float bias) {
  return __builtin_fmaf(tail.alpha, acc, has_bias ? tail.beta * bias : 0.0f);
}

// Sum over the four k slices of a wave: lanes l, l+16, l+32, l+48 hold the same row.
// The result is valid in lanes 0..15.
__device__ __forceinline__ float reduce_k_slices(float v) {
  v += __shfl_down(v, 32);
  v += __shfl_down(v, 16);
  return v;
}

// The kernel arguments behind the preloaded ones, read where the caller stands instead of at the
// kernel's entry.  A by-value kernel argument is fetched by scalar loads that the compiler puts
// in front of everything else, and as soon as one of the registers they target is needed for
// something else the wave waits for them -- a miss of the (just invalidated) scalar cache on the way
// to the first weight loads.  Reading the words through the kernarg segment pointer behind a
// statement the compiler cannot look through keeps those loads where they are written.
// The ten arguments in front of the tail occupy 56 bytes in every kernel of this library.
constexpr int kTailKernargOffset = 56;
static_assert(alignof(GemvTail) == 8 && kTailKernargOffset % alignof(GemvTail) == 0 && sizeof(GemvTail) % 4 == 0,
              "GemvTail follows four pointers and six 32-bit words without padding");
__device__ __forceinline__ GemvTail read_tail_here() {
  typedef const __attribute__((address_space(4))) uint32_t* KernargWords;
  KernargWords words = (KernargWords)__builtin_amdgcn_kernarg_segment_ptr() + kTailKernargOffset / 4;
  asm volatile("" : "+s"(words) : : "memory");
  uint32_t raw[sizeof(GemvTail) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(GemvTail) / 4); ++i) raw[i] = words[i];
  GemvTail t;
  __builtin_memcpy(&t, raw, sizeof(GemvTail));
  return t;
}

// The lane number, recomputed.  Used behind the unit loop so that the value computed in front
// of it need not stay in a register (or be spilled) across the loop.
__device__ __forceinline__ int lane_after_loop() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// ---------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------

struct LaunchPlan {
  int split_k, tiles_per_wg, steps_per_wave, workgroups, wgs_per_xcd, threads;
  int tiles_per_wave;  // 1 on the VALU path; 1, 2 or 4 on the matrix-core path
  int tiles_in_sequence;  // VALU path: most tiles any wave walks one after the other
  int staged_rows;        // LDS-staged and part-tile matrix-core kernels: 8 or 16 activation rows per stage; 0 = other kernels
  int parts;              // part-tile kernels: workgroups per tile (1, 2 or 4; VALU: 1 in batched launches only); 0 = other kernels
                          // k-stationary kernel: workgroups per tile left over (2 or 4); 0 = walks of whole tiles
  int chains, chains_per_wave;  // part-tile matrix-core kernel, batched launches in fewer parts than a single one (else 0): the single
                          // launch's parts are parts * chains, split_k waves take chains_per_wave chains of units each
  int stages;             // VALU path: 2 = the next unit is in flight while one is computed, 1 = it is not
  bool matrix_core;       // one of the matrix-core kernels (else the VALU kernel)
  bool k_stationary;      // the matrix-core kernel whose waves keep one k step each while the workgroup walks tiles_in_sequence tiles
};

// How a wave of the VALU kernel goes through its units (one build of the kernel each).
constexpr int kUnitLoop = 0;  // any number of them
constexpr int kTwoUnits = 1;  // one or two, on one tile
constexpr int kTwoAhead = 2;  // any number, on one tile; the first two are requested together
constexpr int kOneUnit = 3;   // one, on one tile
// The same for batched launches whose problems take parts of tiles by themselves: with finite scales past the reduction, as the kernel
// for parts has them (finite_past_reduction).  A build of its own: kOneUnit with it takes 1.01 of the time of short launches.
constexpr int kOneUnitFinitePast = 4;

// The build a launch takes.  All four compute the same bits, so the number of problems in a batched or routed launch may
// count here, which it does not in the plan.  kTwoAhead is for launches of at most one wave per SIMD, all problems taken
// together: nine problems of 4516x2112 int8 g96 18.7 us / 17.7 in the loop, ten of 3504x5568 g96 25.0 / 24.2, eleven of
// 1740x5120 int8 17.4 / 16.8; 0.946-1.026 of the time on 109 launches of random shapes, mean 0.99.  The figures of single problems
// stand at the kernel's builds.
inline int unit_form(const LaunchPlan& plan, int batch_count, int cus) {
  if (plan.matrix_core || plan.tiles_in_sequence != 1 || plan.stages != 2 || plan.parts != 0) return kUnitLoop;
  if (plan.steps_per_wave <= 2) return plan.steps_per_wave == 1 ? kOneUnit : kTwoUnits;
  return (long long)plan.workgroups * plan.split_k * plan.tiles_per_wg * batch_count <= 4ll * cus ? kTwoAhead : kUnitLoop;
}

// Launches through hipLaunchKernel so that the status returned is this launch's own, not a
// stale sticky error left behind by some other runtime call of the process.
template <typename Kernel, typename... Args>
hipError_t launch(Kernel kernel, dim3 grid, dim3 block, size_t lds, hipStream_t stream, Args... args) {
  void* argv[] = {static_cast<void*>(&args)...};
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, argv, lds, stream);
}

// Host-side description of one GEMV launch.
struct GemvLaunch {
  const uint8_t* weights;
  const half_t* x;
  const half_t* scale;
  const half_t* zero_add;
  int n_out, k, group_size;
  LaunchPlan plan;
  int form;  // VALU kernel: unit_form
  GemvTail tail;
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
  int device;  // the device `stream` belongs to
};

// Dispatchers, one translation unit each (the kernels are templates on weight width, quant mode,
// activation rows, groups per run, ...; the run-time values pick the instantiation).
hipError_t launch_gemv_f16(const GemvLaunch& g, int bits, int qop, int mb, int gpr);
hipError_t launch_gemv_bf16(const GemvLaunch& g, int bits, int qop, int mb, int gpr);
hipError_t launch_valu_parts(const GemvLaunch& g, int bits, int qop, int gpr, int act);
hipError_t launch_mfma(const GemvLaunch& g, int bits, int qop, int gpr);
hipError_t launch_mfma_lds(const GemvLaunch& g, int bits, int qop, int gpr, int rounds, int act);
hipError_t launch_mfma_parts(const GemvLaunch& g, int bits, int qop, int gpr, int act);
hipError_t launch_mfma_kstat(const GemvLaunch& g, int bits, int qop, int gpr, int act);
// Which launches of the k-stationary kernel have a build for left-over tiles in parts; lookups: of scales per lane run, as launched.
// (int8 gains nothing by it, and four lookups per run in fp16 have no registers for it.)
constexpr bool kstat_has_left_over_parts(int bits, int lookups, int act) { return bits == 4 && (act == kActBf16 || lookups != 4); }
// ... and of the k-stationary matrix-core kernel (kProbeLoadsOnly / kProbeComputeOnly), where they exist.
bool mfma_kstat_probe_exists(int bits, int qop, int gpr, int act);
hipError_t launch_mfma_kstat_probe(const GemvLaunch& g, int gpr, int probe);
// Measurement builds of the single-row int4 scale-and-zero fp16 VALU kernel (probe: kProbeLoadsOnly / kProbeTimeline / kProbeComputeOnly).
hipError_t launch_gemv_probe(const GemvLaunch& g, int probe);
// ... and of the LDS-staged matrix-core kernel (kProbeLoadsOnly / kProbeComputeOnly), where they exist.
bool mfma_lds_probe_exists(int bits, int qop, int gpr, int rounds, int act, int tiles_per_wg);
hipError_t launch_mfma_lds_probe(const GemvLaunch& g, int gpr, int rounds, int probe);

}  // namespace mgemv

#endif  // MIXED_GEMV_AMD_KERNEL_COMMON_H_
