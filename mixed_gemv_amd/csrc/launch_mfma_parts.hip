// The matrix-core GEMV kernel for part tiles, gfx950 (MI355X), wave64, and its dispatcher.
#include <atomic>
#include <mutex>
#include <type_traits>

#include "kernel_common.h"
#include "mfma_units.h"

namespace mgemv {

// ---------------------------------------------------------------------------------------------
// Small batches on the matrix cores, one workgroup per PART of a tile: 16 / PARTS of its rows, and PARTS consecutive k steps
// at a time.
//
// A workgroup is split_k waves (at most 8) that share the k steps of its rows; each wave stages its own activation rows in
// LDS, so nothing ties the waves together before the combine.  With one tile per workgroup a matrix of few tiles leaves
// compute units without work and the others with a long reduction.  Rows cannot be spread over lanes any other way -- the 16
// lanes of a matrix operand are 16 rows -- but they need not be 16 rows at the SAME k:
//
//   weight operand, row p * (16 / PARTS) + r        row r of the part, k step s + p
//   activation operand, column p * (16 / PARTS) + b batch row b,       k step s + p
//
// and of the 16 x 16 product only the PARTS blocks on the diagonal (row and column of the same k step) are what is asked for;
// they are added up with the other waves' partial sums, and the rest is never looked at.  The lanes of a wave read 4 KiB of
// weights per unit as before, in pieces of 16 / PARTS neighbouring chunks (128 bytes with two parts, a cache line).
// PARTS * m_batch <= 16.
// What a unit costs is unchanged (dequantiser, sixteen matrix instructions), so a matrix of few tiles is spread over PARTS
// times as many compute units: 1164x12544 at 3 rows, 73 tiles, 8.9 us on the VALU kernel, 8.4 here with one part, 6.4 with two;
// 908x15616 in bf16 10.6 / 9.7 / 7.5, with four 6.1; 2048x11008 at 4 rows 8.4 / 7.8 / 6.1 (2.1 TB/s).
// What bounds it: a compute unit's own path to memory.  Every workgroup needs all of x, PARTS * m_batch KiB beside 4 KiB of
// weights per unit, which the L2 hands a compute unit at 85 GB/s, behind weights at 40-60: per unit 0.29 us at 16 rows, 0.20 of it x
// (0.10 without x and arithmetic), 0.23 at 4 rows, where the arithmetic (0.2) takes over.  Eight waves are therefore no faster
// than four beyond one unit each, and two parts no faster than one once every compute unit has a workgroup.
// ROWS: activation rows staged per unit and wave, 4 (CHAINS > 1), 8 or 16, at least PARTS * m_batch (row b at k step s + p is number
// b * PARTS + p).
// It replaces nothing in the reference, whose kernel is fixed to one activation row
// (gemv/threadblock/default_mma_core_simt.h:68-70); the dequantiser is the one of every kernel here
// (gemv/warp/warp_dequantizer.h:52-59, 86-92), the epilogue host/mixed_gemv.h:102-103.
// blockDim = 64 * split_k.  Dynamic LDS: split_k stages of ROWS x kRowStride bytes, then split_k * chains_per_wave * 256 floats.
// ---------------------------------------------------------------------------------------------
// Byte offsets of the activation rows, in scalar registers; rows that do not exist lie past the descriptor.
constexpr uint32_t kPastActivations = 0x80000000u;  // m_batch * k * 2 bytes are fewer
template <int BATCH_ROWS>
struct RowOffsets {
  uint32_t v[BATCH_ROWS];
};

template <int BITS, int ROWS, int PARTS>
__device__ __forceinline__ void fetch_part_rows(XRows<BITS, ROWS>& r, const RowOffsets<ROWS / PARTS>& rows, int k, __amdgpu_buffer_rsrc_t x_rsrc,
                                                int kstep, int lane) {
  using G = Geometry<BITS>;
  uint32_t at[PARTS];
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    const int k0 = (kstep + p) * G::kStepK + lane * (XStage<BITS>::kLaneBytes / 2);
    at[p] = k0 < k ? (uint32_t)k0 * 2u : kPastActivations;  // k is a multiple of 8: each piece is wholly inside or outside
  }
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    const int off = (int)(at[j % PARTS] + rows.v[j / PARTS]);  // a missing row past k wraps round to the first one's start: never looked at
    if constexpr (BITS == 4) {
      const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, off, 0, kCacheDefault);
      r.v[j][0] = t[0]; r.v[j][1] = t[1]; r.v[j][2] = t[2]; r.v[j][3] = t[3];
    } else {
      const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(x_rsrc, off, 0, kCacheDefault);
      r.v[j][0] = t[0]; r.v[j][1] = t[1];
    }
  }
}

// CHAINS > 1 (batched and routed launches in fewer parts than a single one: plan_of_batch_rows): the bits of the single launch, whose
// parts are PARTS * CHAINS.  A wave of that one adds its products up along `parts` chains at once, chain c the k steps of its range that are
// c modulo the parts; here a unit holds PARTS of them, CHAINS units come to the same k steps, and a wave takes chains_per_wave
// whole chains of units one after the other, whichever range they are of, and parks each one's sums as the single launch's
// wave does.
template <int BITS, int QOP, int GROUPS_PER_RUN, int ROWS, int PARTS, int ACT, int CHAINS = 1>
__global__ void __launch_bounds__(kWave * kMaxWavesPerMfmaWorkgroup)
gemv_mfma_parts_kernel(const uint8_t* weights, const half_t* x, const half_t* scale, const half_t* zero_add, int n_out,
                       int k, uint32_t packed_steps, int workgroups, int num_groups, uint32_t packed_group, GemvTail tail) {
  extern __shared__ float partials[];
  using G = Geometry<BITS>;
  using XS = XStage<BITS>;
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
  constexpr bool kChained = CHAINS > 1;
  const int chains_per_wave = kChained ? tiles_per_wg_of(packed_group) : 1;  // in the place of the tiles per workgroup, which is one
  const long long batch = blockIdx.z;
  long long owner;
  if (!place_problem(p, tail, packed_group, owner)) return;  // whole workgroup, before any barrier
  const bool has_bias = tail.bias != nullptr;
  if constexpr (!kChained) {
    tail.bias += owner * tail.stride_bias;
    tail.y += batch * tail.stride_y;
  }
  const int m_batch = tail.m_batch;

  const int wg = logical_workgroup(p);
  if (wg >= p.workgroups) return;  // whole workgroup leaves before the barrier

  const int lane = threadIdx.x % kWave;
  const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int split_k = tail.split_k;
  PartWork work = part_wave_work(PARTS, wg, kw, p.steps_per_wave, p.ksteps);
  if constexpr (kChained) {
    work.ks_begin = 0;
    work.units = p.ksteps;
  }
  const int slice = lane / kTileRows, column = lane % kTileRows;
  const int k_part = column / kPartRows, row_in_part = column % kPartRows;  // this lane's k step of the unit and its weight row
  const int row0 = work.tile * kTileRows + work.part * kPartRows;
  const int row_raw = row0 + row_in_part;
  const int row = row_raw < p.n_out ? row_raw : p.n_out - 1;

  uint8_t* const lds = reinterpret_cast<uint8_t*>(partials);
  constexpr int kStageBytes = ROWS * XS::kRowStride;
  uint8_t* const stage = lds + kw * kStageBytes;
  // this lane's operand row; columns of batch rows that are not there read row 0 (never stored)
  const int operand_row = (row_in_part < m_batch ? row_in_part : 0) * PARTS + k_part;
  const LdsActivations<BITS> xa{stage + operand_row * XS::kRowStride + slice * G::kRunK * 2};

  const int units = (work.units + PARTS - 1) / PARTS;  // units of PARTS k steps, >= 1 by the host's geometry
  const int ks_begin = work.ks_begin;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(
      p.weights + ((size_t)work.tile * (size_t)p.ksteps + (size_t)ks_begin) * (size_t)kUnitBytes,
      (uint32_t)work.units * (uint32_t)kUnitBytes);  // k steps past the reduction read zeros, and so do their activations
  const int w_lane = k_part * kUnitBytes + (slice * kTileRows + work.part * kPartRows + row_in_part) * kChunkBytes;
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(p.x, (uint32_t)m_batch * (uint32_t)p.k * 2u);
  ScaleTables tables;
  const uint32_t table_bytes = (uint32_t)num_groups * (uint32_t)p.n_out * 2u;
  tables.scale = make_rsrc(p.scale, table_bytes);
  tables.zero = make_rsrc(p.zero_add, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS ? table_bytes : 0u);

  half2_t col_scale = half2_t{};
  const bool short_ok = (tail.flags & kExactIntegerFormOnly) == 0;
  if constexpr (QOP == MGEMV_PER_COLUMN_SCALE_ONLY) col_scale = splat(p.scale[row]);
  const ConvertRegs c = make_convert_regs();

  f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  XRows<BITS, ROWS> xr;
  MfmaWeights<BITS, GROUPS_PER_RUN> wa, wb;
  RowOffsets<ROWS / PARTS> x_rows;
#pragma unroll
  for (int j = 0; j < ROWS / PARTS; ++j) {
    x_rows.v[j] = j < m_batch ? (uint32_t)(j * p.k) * 2u : kPastActivations;
    asm volatile("" : "+s"(x_rows.v[j]));
  }
  // The unit whose first k step is `kstep` behind the wave's first; past the reduction it reads zeros.
  auto request = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& w, int kstep) {
    fetch_part_rows<BITS, ROWS, PARTS>(xr, x_rows, p.k, x_rsrc, ks_begin + kstep, lane);
    load_weights_at<BITS, QOP, GROUPS_PER_RUN, ACT>(w, p, w_rsrc, tables, kstep * kUnitBytes + w_lane,
                                               (ks_begin + kstep + k_part) * G::kStepK + slice * G::kRunK, row);
  };
  // One unit: the rows on their way go to the stage, the next unit's rows and weights are requested (not behind the last),
  // the unit is computed.  The stage belongs to the wave, and the LDS executes a wave's accesses in order: nothing but the
  // compiler has to be kept from reordering them, and one stage is enough.
  auto step = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& now, MfmaWeights<BITS, GROUPS_PER_RUN>& next, int kstep, int next_kstep, auto last) {
    park_x_rows<BITS, ROWS>(xr, stage, lane, 0, 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (!decltype(last)::value) request(next, next_kstep);
    __builtin_amdgcn_sched_barrier(0);
    half2_t s2 = col_scale;
    const int k_unit = (ks_begin + kstep) * G::kStepK;
    if (k_unit + PARTS * G::kStepK > p.k) {
      const int k_run = k_unit + k_part * G::kStepK + slice * G::kRunK;
      s2 = k_run < p.k ? s2 : as_half2(kAnyScale<ACT> | kAnyScale<ACT> << 16);
      finite_past_reduction<ACT>(now.s, now.z, k_run, G::kRunK / GROUPS_PER_RUN, p.k);
    }
    compute_unit_mfma<BITS, QOP, GROUPS_PER_RUN, ACT>(acc, now, xa, c, s2, short_ok);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4* const combine = reinterpret_cast<f32x4*>(lds + split_k * kStageBytes);
  if constexpr (kChained) {
    // Chain e of the workgroup: k steps from range e / CHAINS on, every CHAINS * PARTS.  Chains without a unit (the end of the
    // reduction) and, in the last wave, of no range park zeros.
    f32x4* park = combine + kw * chains_per_wave * kWave + lane;
    for (int j = 0; j < chains_per_wave; ++j) park[j * kWave] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int kStride = CHAINS * PARTS;
    auto first_of = [&](int chain) { return chain / CHAINS * p.steps_per_wave + chain % CHAINS * PARTS; };
    auto end_of = [&](int chain) {
      const int end = (chain / CHAINS + 1) * p.steps_per_wave;
      return end < p.ksteps ? end : p.ksteps;
    };
    int chain = kw * chains_per_wave, kstep = first_of(chain), end = end_of(chain);
    const int past = chain + chains_per_wave;
    auto find_unit = [&]() {  // from kstep on; past the wave's last: past the reduction
      while (kstep >= end && chain < past) {
        ++chain;
        kstep = chain < past ? first_of(chain) : p.ksteps;
        end = end_of(chain);
      }
    };
    find_unit();
    request(wa, kstep);
    int count = 0;
    for (int c = kw * chains_per_wave; c < past; ++c) {
      const int steps = end_of(c) - first_of(c);
      count += steps > 0 ? (steps + kStride - 1) / kStride : 0;
    }
    auto one = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& now, MfmaWeights<BITS, GROUPS_PER_RUN>& next, auto last) {
      const int here = kstep, chain_here = chain;
      kstep += kStride;
      find_unit();
      step(now, next, here, kstep, last);
      if (chain != chain_here) {
        park[(chain_here - (past - chains_per_wave)) * kWave] = acc;
        acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
    };
    int u = 0;
    for (; u + 1 < count; u += 2) {
      one(wa, wb, std::false_type{});
      one(wb, wa, std::false_type{});
    }
    if (u < count) one(wa, wb, std::true_type{});
  } else {
    // whole pairs of units, and a single one behind them (as in the LDS-staged kernel)
    request(wa, 0);
    int u = 0;
    for (; u + 1 < units; u += 2) {
      step(wa, wb, u * PARTS, (u + 1) * PARTS, std::false_type{});
      step(wb, wa, (u + 1) * PARTS, (u + 2) * PARTS, std::false_type{});
    }
    if (u < units) step(wa, wb, u * PARTS, 0, std::true_type{});
  }

  if constexpr (kChained) {  // (read again: there are no registers for it in the loop)
    tail = read_tail_here();
    tail.bias += owner * tail.stride_bias;
    tail.y += batch * tail.stride_y;
  }
  // Lane l holds rows 4 * (l / 16) .. + 3 of the product in column l % 16.  Lane (quad, b) of wave 0 adds up what belongs to
  // rows 4 * quad .. + 3 of the part and batch row b: one entry of every wave and k step of a unit, ascending.
  constexpr int kQuads = kPartRows / 4;
  const int quad = slice % kQuads, b = column % kPartRows;
  const bool sums = kw == 0 && slice < kQuads && column < kPartRows && b < m_batch;
  const int n0 = row0 + 4 * quad;
  float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (sums && has_bias) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = n0 + v < p.n_out ? n0 + v : p.n_out - 1;
      if constexpr (ACT == kActBf16)
        bias[v] = bf16_low_to_f32(reinterpret_cast<const uint16_t*>(tail.bias)[n]);
      else
        bias[v] = (float)tail.bias[n];
    }
  }
  f32x4 sum = acc;
  if (kChained || PARTS > 1 || split_k > 1) {
    if constexpr (!kChained) combine[kw * kWave + lane] = acc;
    const int entries = split_k * chains_per_wave;
    __syncthreads();
    if (!sums) return;
    // entry of k step pt of wave (or chain) w: column pt * kPartRows + b of quad pt * kQuads + quad
    const f32x4* part = combine + quad * kTileRows + b;
    constexpr int kEntry = kQuads * kTileRows + kPartRows;
    sum = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int w = 0;
    for (; w + 4 <= entries; w += 4) {
      f32x4 piece[4 * PARTS];
#pragma unroll
      for (int i = 0; i < 4 * PARTS; ++i) piece[i] = part[(w + i / PARTS) * kWave + i % PARTS * kEntry];
#pragma unroll
      for (int i = 0; i < 4 * PARTS; ++i) sum += piece[i];
    }
    for (; w < entries; ++w) {
#pragma unroll
      for (int i = 0; i < PARTS; ++i) sum += part[w * kWave + i * kEntry];
    }
  }
  if (!sums) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int n = n0 + v;
    if (n < p.n_out) {
      const float r = epilogue_value(tail, sum[v], has_bias, bias[v]);
      if constexpr (ACT == kActBf16)
        reinterpret_cast<uint16_t*>(tail.y)[(size_t)b * (size_t)p.n_out + n] = (uint16_t)pack_bf16(r, 0.0f);
      else
        tail.y[(size_t)b * (size_t)p.n_out + n] = (half_t)r;
    }
  }
}

template <int BITS, int QOP, int GPR, int ROWS, int PARTS, int ACT, int CHAINS = 1>
hipError_t launch_mfma_parts_kernel(const GemvLaunch& g) {
  const auto kernel = gemv_mfma_parts_kernel<BITS, QOP, GPR, ROWS, PARTS, ACT, CHAINS>;
  if (g.lds > 48 * 1024) {
    // More than 48 KiB of dynamic LDS has to be granted per kernel and device; remember the
    // largest grant so that only the first such launch pays for the call.
    constexpr int kMaxDevices = 64;
    static std::atomic<int> granted[kMaxDevices];
    static std::mutex grant_mutex;
    const int device = g.device;
    const bool tracked = device >= 0 && device < kMaxDevices;
    if (!tracked || granted[device].load() < (int)g.lds) {
      std::lock_guard<std::mutex> lock(grant_mutex);
      if (!tracked || granted[device].load() < (int)g.lds) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)g.lds);
        if (e != hipSuccess) return e;
        if (tracked) granted[device].store((int)g.lds);
      }
    }
  }
  return launch(kernel, g.grid, g.block, g.lds, g.stream, g.weights, g.x, g.scale, g.zero_add, g.n_out, g.k,
                pack_steps(num_ksteps(g.k, BITS), g.plan.steps_per_wave), g.plan.workgroups, g.tail.num_groups,
                pack_group(g.group_size, CHAINS > 1 ? g.plan.chains_per_wave : 1, g.tail.stack != nullptr), g.tail);
}

template <int BITS, int QOP, int GPR, int ACT>
hipError_t launch_mfma_parts_rows(const GemvLaunch& g) {
  if (g.plan.chains != 0) {
    if (g.plan.parts == 2) return launch_mfma_parts_kernel<BITS, QOP, GPR, 8, 2, ACT, 2>(g);
    if (g.plan.staged_rows == 8) return launch_mfma_parts_kernel<BITS, QOP, GPR, 8, 1, ACT, 2>(g);
    return g.plan.chains == 2 ? launch_mfma_parts_kernel<BITS, QOP, GPR, 4, 1, ACT, 2>(g) : launch_mfma_parts_kernel<BITS, QOP, GPR, 4, 1, ACT, 4>(g);
  }
  if (g.plan.staged_rows == 8)
    return g.plan.parts == 1 ? launch_mfma_parts_kernel<BITS, QOP, GPR, 8, 1, ACT>(g) : launch_mfma_parts_kernel<BITS, QOP, GPR, 8, 2, ACT>(g);
  switch (g.plan.parts) {
    case 1: return launch_mfma_parts_kernel<BITS, QOP, GPR, 16, 1, ACT>(g);
    case 2: return launch_mfma_parts_kernel<BITS, QOP, GPR, 16, 2, ACT>(g);
    default: return launch_mfma_parts_kernel<BITS, QOP, GPR, 16, 4, ACT>(g);
  }
}

template <int BITS, int QOP, int ACT>
hipError_t launch_mfma_parts_gpr(const GemvLaunch& g, int gpr) {
  if constexpr (QOP == MGEMV_PER_COLUMN_SCALE_ONLY) {
    return launch_mfma_parts_rows<BITS, QOP, 1, ACT>(g);
  } else {
    switch (gpr) {
      case 1: return launch_mfma_parts_rows<BITS, QOP, 1, ACT>(g);
      case 2: return launch_mfma_parts_rows<BITS, QOP, 2, ACT>(g);
      default: return launch_mfma_parts_rows<BITS, QOP, 4, ACT>(g);
    }
  }
}

template <int ACT>
hipError_t launch_mfma_parts_act(const GemvLaunch& g, int bits, int qop, int gpr) {
  if (bits == 4) {
    switch (qop) {
      case 1: return launch_mfma_parts_gpr<4, 1, ACT>(g, gpr);
      case 2: return launch_mfma_parts_gpr<4, 2, ACT>(g, gpr);
      default: return launch_mfma_parts_gpr<4, 3, ACT>(g, gpr);
    }
  }
  switch (qop) {
    case 1: return launch_mfma_parts_gpr<8, 1, ACT>(g, gpr);
    case 2: return launch_mfma_parts_gpr<8, 2, ACT>(g, gpr);
    default: return launch_mfma_parts_gpr<8, 3, ACT>(g, gpr);
  }
}

hipError_t launch_mfma_parts(const GemvLaunch& g, int bits, int qop, int gpr, int act) {
  return act == kActBf16 ? launch_mfma_parts_act<kActBf16>(g, bits, qop, gpr) : launch_mfma_parts_act<kActF16>(g, bits, qop, gpr);
}

}  // namespace mgemv
