// The VALU GEMV kernel for parts of tiles, gfx950 (MI355X), wave64, one activation row, and its dispatcher.
#include "gemv_dpp_kernel.h"

namespace mgemv {

// ---------------------------------------------------------------------------------------------
// One activation row, one workgroup per PART of a tile: 16 / PARTS of its rows, and PARTS consecutive k steps at a time.
//
// With one tile per workgroup a matrix of few tiles leaves compute units without work and the others with a long reduction:
// 744x23064 in bf16, 47 workgroups of four waves with twelve units each, took 17.8 us, one unit after the other at the rate
// that a wave alone on its SIMD issues at (its bytes take 1.4).  The 16 lanes of a k slice are 16 rows of one k step there, because
// all of them take their activations from one register of the slice by a row broadcast.  Here a lane is
//
//   lane % 16 = k_part * (16 / PARTS) + row        row of the part, k step s + k_part
//
// and four lanes, which always are rows of one k step, hold the activations of their own slice and k step between them: lane J
// of the four those of word J of each block, sixteen registers (int8: eight) where the row broadcast needs four (two),
// and the dot takes them by a quad broadcast.  The arithmetic of a unit is unchanged; a wave reads 4 KiB of weights per unit as
// before, in pieces of 16 / PARTS neighbouring chunks.  512x5120, one row, groups of 128 with zeros 3.9 us / 3.1, 1024x16384 7.3 / 5.0
// (1.8 TB/s); 900x4608 per column in bf16 5.5 / 3.3.  What bounds it: start and end of a launch, then a compute unit's path to
// memory.
// PARTS 1, by row broadcast, is for batched launches, which have the bits of single ones (plan_of_batch): the sums of every unit
// are added up in an order of their own, parked in the LDS up to 16 k steps, beyond by a wave for every fourth k step (LONG).
// 1224 such launches of two to eight problems take 0.97 of the time of the kernel for whole tiles, 1.0 with four lookups per run (0.57-1.13).
// (Every sum parked and units in one loop: 1.02, with a lookup per block on 9-16 k steps up to 1.35: 2048x4896 g96 in bf16, six
// problems, 9.65 us whole, 13.0 so, 9.7 here.)
// Not taken: eight waves beyond eight units (1.0-1.1 of the time of four); requests behind a wave's last unit (1.05-1.2, half of
// what a wave of two units issues).
// ---------------------------------------------------------------------------------------------

// Everything one lane needs for one unit of a part: PARTS k steps of 16 / PARTS rows.
template <int BITS, int GROUPS_PER_RUN, int PARTS>
struct PartFragment {
  static constexpr int kXPieces = PARTS == 1 ? 1 : kBlocksPerUnit;
  u32x4 w[kBlocksPerUnit];                   // 4 chunks of this lane's row and k step
  uint32_t x[kXPieces][BITS == 4 ? 4 : 2];   // the activations that word lane % 4 of each block pairs with (PARTS 1: word lane % 16 of the unit)
  uint32_t s[GROUPS_PER_RUN], z[GROUPS_PER_RUN];   // low 16 bits; the rest is unspecified
};

// Block I of a unit.  Lane J of a quad holds the activations that word J of the quad's four rows pairs with.
template <int BITS, int QOP, int GROUPS_PER_RUN, int PARTS, bool SHORT, int I, int ACT>
__device__ __forceinline__ void compute_part_block(float& acc, const PartFragment<BITS, GROUPS_PER_RUN, PARTS>& f, const ConvertRegs& c,
                                                   const Int4ScaleBf16 (&short4)[GROUPS_PER_RUN]) {
  constexpr bool kHasZero = QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS;
  constexpr int gi = I * GROUPS_PER_RUN / kBlocksPerUnit;
  constexpr int kPairs = BITS == 4 ? 4 : 2;
  auto dot = [&](auto word, int h, auto d) {
    constexpr int J = decltype(word)::value;
    if constexpr (ACT == kActBf16) {
      if constexpr (PARTS == 1) dot2_row_bcast_bf16<4 * I + J>(acc, f.x[0][h], d);
      else dot2_quad_bcast_bf16<J>(acc, f.x[I][h], d);
    } else {
      if constexpr (PARTS == 1) dot2_row_bcast<4 * I + J>(acc, f.x[0][h], d);
      else dot2_quad_bcast<J>(acc, f.x[I][h], d);
    }
  };
  if constexpr (ACT == kActBf16) {
    const Bf16Scale bs = make_bf16_scale<BITS, SHORT>(f.s[gi], kHasZero ? f.z[gi] : 0u, make_identity4(), short4[gi]);
    auto two_words = [&](auto first) {
      constexpr int J = decltype(first)::value;
      uint32_t d[2 * kPairs];
      if constexpr (BITS == 4) dequant_int4_words_bf16<kHasZero, SHORT, 2>({f.w[I][J], f.w[I][J + 1]}, c, bs, d);
      else dequant_int8_words_bf16<kHasZero, SHORT, 2>({f.w[I][J], f.w[I][J + 1]}, bs, d);
#pragma unroll
      for (int h = 0; h < kPairs; ++h) dot(first, h, d[h]);
#pragma unroll
      for (int h = 0; h < kPairs; ++h) dot(std::integral_constant<int, J + 1>{}, h, d[kPairs + h]);
    };
    two_words(std::integral_constant<int, 0>{});
    two_words(std::integral_constant<int, 2>{});
  } else {
    const half2_t s2 = splat_low(f.s[gi]);
    half2_t z2 = half2_t{};
    if constexpr (kHasZero) z2 = splat_low(f.z[gi]);
    ShortFormScale sf{};
    if constexpr (BITS == 4 && SHORT) sf = make_short_form_scale(s2);
    auto word = [&](auto which) {
      constexpr int J = decltype(which)::value;
      half2_t d[kPairs];
      if constexpr (BITS == 4 && SHORT) {
        dequant_int4_word_short<kHasZero>(f.w[I][J], c, sf, z2, d);
      } else {
        half2_t q[kPairs];
        if constexpr (BITS == 4) convert_int4_word(f.w[I][J], c, q); else convert_int8_word(f.w[I][J], c, q);
#pragma unroll
        for (int h = 0; h < kPairs; ++h) d[h] = dequant_pair<kHasZero>(q[h], s2, z2);
      }
#pragma unroll
      for (int h = 0; h < kPairs; ++h) dot(which, h, d[h]);
    };
    word(std::integral_constant<int, 0>{});
    word(std::integral_constant<int, 1>{});
    word(std::integral_constant<int, 2>{});
    word(std::integral_constant<int, 3>{});
  }
}

// The sums of one unit, added to acc.
template <int BITS, int QOP, int GROUPS_PER_RUN, int PARTS, int ACT>
__device__ __forceinline__ void compute_part_unit(float& acc, const PartFragment<BITS, GROUPS_PER_RUN, PARTS>& f, const ConvertRegs& regs,
                                                  bool short_allowed) {
  Int4ScaleBf16 short4[GROUPS_PER_RUN] = {};
  auto all_blocks = [&](auto form) {
    constexpr bool SHORT = decltype(form)::value;
    const ConvertRegs c = (ACT == kActF16 && BITS == 4 && !SHORT) ? general_form_regs(regs) : regs;
    compute_part_block<BITS, QOP, GROUPS_PER_RUN, PARTS, SHORT, 0, ACT>(acc, f, c, short4);
    compute_part_block<BITS, QOP, GROUPS_PER_RUN, PARTS, SHORT, 1, ACT>(acc, f, c, short4);
    compute_part_block<BITS, QOP, GROUPS_PER_RUN, PARTS, SHORT, 2, ACT>(acc, f, c, short4);
    compute_part_block<BITS, QOP, GROUPS_PER_RUN, PARTS, SHORT, 3, ACT>(acc, f, c, short4);
    settle_dot_chain(acc);  // (the two forms meet again behind this)
  };
  if constexpr (BITS == 4 || ACT == kActBf16) {
    if (short_allowed && wave_takes_short_form<BITS, ACT>(f.s, short4)) {
      all_blocks(std::true_type{});
      return;
    }
  }
  all_blocks(std::false_type{});
}

// blockDim = 64 * split_k.  Dynamic LDS: 64 floats for each unit, units in whole kValuPartsSumsAtOnce.
// LONG: PARTS 1 and more k steps than kValuPartsSumsAtOnce -- four waves, each every fourth k step, which adds up their sums itself.
// (PARTS 1 otherwise: waves of one or two units.)
template <int BITS, int QOP, int GROUPS_PER_RUN, int PARTS, int ACT, bool LONG = false>
__global__ void __launch_bounds__(kWave * kMaxWavesPerWideWorkgroup)
gemv_dpp_parts_kernel(const uint8_t* weights, const half_t* x, const half_t* scale, const half_t* zero_add, int n_out, int k,
                      uint32_t packed_steps, int workgroups, int num_groups, uint32_t packed_group, GemvTail tail) {
  extern __shared__ float partials[];
  using G = Geometry<BITS>;
  constexpr int kPartRows = kTileRows / PARTS;
  Problem p;
  p.weights = weights;
  p.x = x;
  p.scale = scale;
  p.zero_add = zero_add;
  p.n_out = n_out;
  p.k = k;
  p.ksteps = (int)(packed_steps & 0xffffu);
  p.steps_per_wave = (int)(packed_steps >> 16);  // a multiple of PARTS
  p.workgroups = workgroups;
  p.wgs_per_xcd = (workgroups + kNumXcd - 1) / kNumXcd;
  p.group_size = (int)(packed_group & 0xffffffu);
  p.tiles_per_wg = 1;
  const long long batch = blockIdx.z;
  long long owner;
  if (!place_problem(p, tail, packed_group, owner)) return;  // whole workgroup, before any barrier

  const int wg = logical_workgroup(p);
  if (wg >= p.workgroups) return;  // whole workgroup leaves before the barrier

  const int lane = threadIdx.x % kWave;
  const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const PartWork work = part_wave_work(PARTS, wg, kw, p.steps_per_wave, p.ksteps);
  const int slice = lane / kTileRows, k_part = lane % kTileRows / kPartRows, row_in_part = lane % kPartRows;
  const int row0 = work.tile * kTileRows + work.part * kPartRows;
  const int row = row0 + row_in_part < p.n_out ? row0 + row_in_part : p.n_out - 1;  // padding: never stored
  constexpr int kUnitSteps = LONG ? 4 : PARTS;  // k steps from a unit to the next
  const int ks_begin = LONG ? kw : work.ks_begin;
  const int wave_steps = LONG ? p.ksteps - kw : work.units;
  const int units = (wave_steps + kUnitSteps - 1) / kUnitSteps;  // >= 1 by the host's geometry
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(
      p.weights + ((size_t)work.tile * (size_t)p.ksteps + (size_t)ks_begin) * (size_t)kUnitBytes,
      (uint32_t)wave_steps * (uint32_t)kUnitBytes);  // k steps past the reduction read zeros, and so do their activations
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(p.x, (uint32_t)p.k * 2u);
  ScaleTables tables;
  const uint32_t table_bytes = (uint32_t)num_groups * (uint32_t)p.n_out * 2u;
  tables.scale = make_rsrc(p.scale, table_bytes);
  tables.zero = make_rsrc(p.zero_add, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS ? table_bytes : 0u);
  const int w_lane = k_part * kUnitBytes + (slice * kTileRows + work.part * kPartRows + row_in_part) * kChunkBytes;
  const int k_lane = (ks_begin + k_part) * G::kStepK + slice * G::kRunK;  // first reduction index of the lane's run

  // One or two groups per run: the group size divides the k step, and a lane's scales lie a constant step apart.
  int first_offset[GROUPS_PER_RUN], offset_step = 0;
  if constexpr (GROUPS_PER_RUN != 4) {
    const int shift = __builtin_ctz((unsigned)p.group_size);
    const bool per_column = QOP == MGEMV_PER_COLUMN_SCALE_ONLY;
    offset_step = per_column ? 0 : kUnitSteps * (G::kStepK >> shift) * p.n_out * 2;
#pragma unroll
    for (int gi = 0; gi < GROUPS_PER_RUN; ++gi)
      first_offset[gi] = ((per_column ? 0 : (k_lane + gi * (G::kRunK / GROUPS_PER_RUN)) >> shift) * p.n_out + row) * 2;
  }

  PartFragment<BITS, GROUPS_PER_RUN, PARTS> fa, fb;
  // A unit past the wave's is sent past every descriptor: such loads come back at once.
  auto request = [&](PartFragment<BITS, GROUPS_PER_RUN, PARTS>& f, int u) {
    const int away = u < units ? 0 : 0x40000000;
    const int k_run = k_lane + u * (kUnitSteps * G::kStepK);
    const int x_voffset = (k_run + lane % (PARTS == 1 ? 16 : 4) * (G::kChunkK / 4)) * 2 + away;
#pragma unroll
    for (int i = 0; i < f.kXPieces; ++i) {
      if constexpr (BITS == 4) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, x_voffset + i * (G::kChunkK * 2), 0, kCacheDefault);
        f.x[i][0] = v[0]; f.x[i][1] = v[1]; f.x[i][2] = v[2]; f.x[i][3] = v[3];
      } else {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(x_rsrc, x_voffset + i * (G::kChunkK * 2), 0, kCacheDefault);
        f.x[i][0] = v[0]; f.x[i][1] = v[1];
      }
    }
#pragma unroll
    for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) {
      int off;
      if constexpr (GROUPS_PER_RUN == 4) off = (group_of<4>(p, k_run + gi * G::kChunkK) * p.n_out + row) * 2 + away;
      else off = first_offset[gi] + u * offset_step + away;
      f.s[gi] = load_b16_low(tables.scale, off);
      if constexpr (QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS) f.z[gi] = load_b16_low(tables.zero, off);
    }
#pragma unroll
    for (int i = 0; i < kBlocksPerUnit; ++i)
      f.w[i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_lane + u * (kUnitSteps * kUnitBytes) + i * kBlockBytes, 0, kCacheStream);
    __builtin_amdgcn_sched_barrier(0);
  };
  request(fa, 0);
  GemvTail late = read_tail_here();
  const bool has_bias = late.bias != nullptr;
  const __amdgpu_buffer_rsrc_t bias_rsrc = make_rsrc(late.bias + owner * late.stride_bias, has_bias ? (uint32_t)p.n_out * 2u : 0u);
  const uint32_t bias_bits = load_b16_low(bias_rsrc, (row0 + lane) * 2);  // lanes of the part's rows
  __builtin_amdgcn_sched_barrier(0);
  request(fb, 1);
  const bool short_ok = (late.flags & kExactIntegerFormOnly) == 0;
  const ConvertRegs c = make_convert_regs();
  float* const my_sums = partials + ks_begin / PARTS * kWave + lane;
  float so_far = 0.0f;  // LONG
  auto compute = [&](PartFragment<BITS, GROUPS_PER_RUN, PARTS>& f, int u) {
    const int k_unit = (ks_begin + u * kUnitSteps) * G::kStepK;
    if (k_unit + PARTS * G::kStepK > p.k) {
      finite_past_reduction<ACT>(f.s, f.z, k_lane + u * (kUnitSteps * G::kStepK), G::kRunK / GROUPS_PER_RUN, p.k);
    }
    float acc = 0.0f;
    compute_part_unit<BITS, QOP, GROUPS_PER_RUN, PARTS, ACT>(acc, f, c, short_ok);
    if constexpr (LONG) so_far += acc;
    else my_sums[u * kWave] = acc;
    __builtin_amdgcn_sched_barrier(0);
  };
  int u = 0;
  if constexpr (PARTS == 1 && !LONG) {
    compute(fa, 0);
    if (units > 1) compute(fb, 1);
  } else if constexpr (GROUPS_PER_RUN == 4) {
    // (in the form below 149-183 registers of a bf16 build with zeros, and 1.05-1.2 of the time where workgroups share a compute unit)
    do {
      compute(fa, u);
      request(fa, u + 2);
      if (u + 1 < units) compute(fb, u + 1);
      __builtin_amdgcn_sched_barrier(0);
      request(fb, u + 3);
      u += 2;
    } while (u < units);
  } else {
    // nothing is requested behind the last units
    for (; u + 2 < units; u += 2) {
      compute(fa, u);
      request(fa, u + 2);
      compute(fb, u + 1);
      request(fb, u + 3);
    }
    compute(fa, u);
    if (u + 1 < units) compute(fb, u + 1);
  }

  if constexpr (LONG) *my_sums = so_far;
  __syncthreads();
  if (kw != 0) return;
  // The order of the sums depends on the number of k steps alone, neither on PARTS nor on the waves, so that a launch of many
  // problems may take other parts than a single one and give the same bits.
  // (All of what follows is worked out here: in front of the loop it would stand in the way of the first loads.  Sums of units that
  // do not exist are read, there is room for them, and left alone.)
  int ksteps = p.ksteps;
  asm volatile("" : "+s"(ksteps));
  const int l = lane_after_loop();
  constexpr int kAtOnce = kValuPartsSumsAtOnce;
  float sum = 0.0f;
  if (PARTS == 1 ? !LONG : ksteps <= kAtOnce) {
    // as the waves of one k step each of the kernel for whole tiles: k steps ascending, then the slices
    const float* part = partials + l / kTileRows * kTileRows + l % kPartRows;
    float piece[kAtOnce];
#pragma unroll
    for (int s = 0; s < kAtOnce; ++s) piece[s] = part[s / PARTS * kWave + s % PARTS * kPartRows];
#pragma unroll
    for (int s = 0; s < kAtOnce; ++s) sum += s < ksteps ? piece[s] : 0.0f;
    sum = reduce_k_slices(sum);
  } else {
    // every fourth k step ascending, the slices, then (0 + 2) + (1 + 3)
    constexpr int kChains = 4 / PARTS;
    float chain[kChains] = {};
    const int total = LONG ? 4 : (ksteps + PARTS - 1) / PARTS;  // entries
    const float* part = partials + l;
    for (int i = 0; i < total; i += kAtOnce) {
      float piece[kAtOnce];
#pragma unroll
      for (int j = 0; j < kAtOnce; ++j) piece[j] = part[(i + j) * kWave];
#pragma unroll
      for (int j = 0; j < kAtOnce; ++j) chain[j % kChains] += i + j < total ? piece[j] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kChains; ++j) chain[j] = reduce_k_slices(chain[j]);
    if constexpr (PARTS == 1) sum = (chain[0] + chain[2 % kChains]) + (chain[1 % kChains] + chain[3 % kChains]);
    if constexpr (PARTS == 2) { sum = chain[0] + chain[1 % kChains]; sum += __shfl_down(sum, 8); }
    if constexpr (PARTS == 4) { sum = chain[0] + __shfl_down(chain[0], 8); sum += __shfl_down(sum, 4); }
  }
  const int n = row0 + l;
  if (l < kPartRows && n < p.n_out) {
    late.y += batch * late.stride_y;
    if constexpr (ACT == kActBf16)
      reinterpret_cast<uint16_t*>(late.y)[n] = (uint16_t)pack_bf16(epilogue_value(late, sum, has_bias, bf16_low_to_f32(bias_bits)), 0.0f);
    else
      late.y[n] = (half_t)epilogue_value(late, sum, has_bias, (float)splat_low(bias_bits)[0]);
  }
}

template <int BITS, int QOP, int GPR, int ACT>
hipError_t launch_valu_parts_kernel(const GemvLaunch& g) {
  const auto kernel = g.plan.parts == 4   ? gemv_dpp_parts_kernel<BITS, QOP, GPR, 4, ACT>
                      : g.plan.parts == 2 ? gemv_dpp_parts_kernel<BITS, QOP, GPR, 2, ACT>
                      : num_ksteps(g.k, BITS) > kValuPartsSumsAtOnce ? gemv_dpp_parts_kernel<BITS, QOP, GPR, 1, ACT, true>
                                                                     : gemv_dpp_parts_kernel<BITS, QOP, GPR, 1, ACT>;
  return launch(kernel, g.grid, g.block, g.lds, g.stream, g.weights, g.x, g.scale, g.zero_add, g.n_out, g.k,
                pack_steps(num_ksteps(g.k, BITS), g.plan.steps_per_wave), g.plan.workgroups, g.tail.num_groups,
                pack_group(g.group_size, 1, g.tail.stack != nullptr), g.tail);
}

template <int BITS, int QOP, int ACT>
hipError_t launch_valu_parts_gpr(const GemvLaunch& g, int gpr) {
  if constexpr (QOP == MGEMV_PER_COLUMN_SCALE_ONLY) {
    return launch_valu_parts_kernel<BITS, QOP, 1, ACT>(g);
  } else {
    switch (gpr) {
      case 1: return launch_valu_parts_kernel<BITS, QOP, 1, ACT>(g);
      case 2: return launch_valu_parts_kernel<BITS, QOP, 2, ACT>(g);
      default: return launch_valu_parts_kernel<BITS, QOP, 4, ACT>(g);
    }
  }
}

template <int ACT>
hipError_t launch_valu_parts_act(const GemvLaunch& g, int bits, int qop, int gpr) {
  if (bits == 4) {
    switch (qop) {
      case 1: return launch_valu_parts_gpr<4, 1, ACT>(g, gpr);
      case 2: return launch_valu_parts_gpr<4, 2, ACT>(g, gpr);
      default: return launch_valu_parts_gpr<4, 3, ACT>(g, gpr);
    }
  }
  switch (qop) {
    case 1: return launch_valu_parts_gpr<8, 1, ACT>(g, gpr);
    case 2: return launch_valu_parts_gpr<8, 2, ACT>(g, gpr);
    default: return launch_valu_parts_gpr<8, 3, ACT>(g, gpr);
  }
}

hipError_t launch_valu_parts(const GemvLaunch& g, int bits, int qop, int gpr, int act) {
  return act == kActBf16 ? launch_valu_parts_act<kActBf16>(g, bits, qop, gpr) : launch_valu_parts_act<kActF16>(g, bits, qop, gpr);
}

}  // namespace mgemv
