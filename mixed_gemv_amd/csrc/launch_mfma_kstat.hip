// The k-stationary matrix-core GEMV kernel for gfx950 (MI355X), wave64, and its dispatcher.
#include <atomic>
#include <mutex>
#include <type_traits>

#include "kernel_common.h"
#include "mfma_units.h"

namespace mgemv {

// ---------------------------------------------------------------------------------------------
// Matrix-core kernel whose waves stay on one k step.
//
// blockDim = 64 * ksteps (at most 16 waves): wave kw of a workgroup owns k step kw of EVERY tile
// the workgroup walks.  The activation operand of a k step -- x[batch row lane % 16][the lane's 8 k
// of each of the 16 matrix instructions], 64 registers for int4 -- therefore never changes: it is
// loaded once, in front of the walk, and the loop over the tiles holds nothing but the weight
// stream (one unit of 4 KiB per wave and tile, the next tile's unit in flight while one is
// computed), the dequantiser and sixteen matrix instructions.  No LDS stage, no barrier and no
// activation traffic inside the loop; a wave's partial products of a tile (a 16 x 16 fp32 block, of
// which m_batch columns matter) are parked in LDS, and after the walk one barrier separates the
// walks from the combine: wave r sums the ksteps partial blocks of tiles r, r + waves, ... and
// stores them.  Per eight int4 weights a lane issues 13 VALU instructions and one matrix
// instruction, against 17 VALU instructions of the DPP-dot kernel, whatever the number of rows.
// bf16: the dequantiser needs the registers, so the operand stays in the wave's stage instead and is read from LDS, two
// matrix instructions ahead (16 LDS reads of 16 bytes beside 400 other instructions a unit; 98-128 registers, 4 waves per
// SIMD, no spills -- with a block's operands ahead the four-group build spilled 30 and took 1.4 times as long).  What
// bounds it is its instruction issue (53-68 % of all cycles issue a vector instruction, at 1.9-2.1 GHz), then the start (16 MiB of first
// units) and the last unit's arithmetic.  28672x8192, 4 rows: 31.3 us, 3.8 TB/s; the LDS-staged kernel, whose 140-164
// registers leave 3 waves per SIMD and whose barriers line them up, 35.1.
// It replaces nothing in the reference, whose kernel is fixed to one activation row
// (gemv/threadblock/default_mma_core_simt.h:68-70); the dequantiser is the one of every kernel here
// (gemv/warp/warp_dequantizer.h:52-59, 86-92), the epilogue host/mixed_gemv.h:102-103.
// Dynamic LDS: waves x 8 activation rows (the stage each wave turns its operand round in, at the start; bf16: waves x
// m_batch rows, which stay) and
// tiles of the longest walk x 4 x m_batch x 17 x 16 bytes (the partial sums) -- one behind the other where
// both fit, else sharing the space, with a barrier between the two uses.  Static, bf16: kKStationaryZeroBytes of zeros.
// TAIL: m_batch rows that stay in either type, the zeros, and kKStationaryStagedBytes of words.
// ---------------------------------------------------------------------------------------------

// Where a wave keeps its activation operand: in registers, or in its stage.
template <int BITS, bool LDS_OPERAND>
struct KStatOperand { typedef MfmaActivations<BITS> type; };
template <int BITS>
struct KStatOperand<BITS, true> { typedef LdsActivations<BITS> type; };

// PROBE (measurement builds, wrong results): kProbeLoadsOnly keeps every load, the operand's way through LDS, the
// parking, the barrier and the combine, and replaces the arithmetic of a unit by taking its registers;
// kProbeComputeOnly requests only the first tile's unit and repeats its arithmetic for every tile of the walk.
// TAIL: the tiles that do not divide over the workgroups are split into parts, two or four workgroups to a tile: behind its walk a
// workgroup takes 16 / parts rows of one of them, and a wave a unit of `parts` k steps of those, mapped to the matrix operands as in
// the part-tile kernel.  A column of a product holds one k step's sums in the order of every other unit's, so the bits are the same.
// (Which launches, and what it is worth: left_over_parts.)
template <int BITS, int QOP, int GROUPS_PER_RUN, int ACT, int PROBE = kProbeNone, bool TAIL = false>
__global__ void __launch_bounds__(kWave * kMaxWavesPerWorkgroup)
gemv_mfma_kstat_kernel(const uint8_t* weights, const half_t* x, const half_t* scale, const half_t* zero_add, int n_out,
                       int k, uint32_t packed_steps, int workgroups, int num_groups, uint32_t packed_group,
                       GemvTail tail) {
  extern __shared__ float partials[];
  using G = Geometry<BITS>;
  constexpr bool kLdsOperand = ACT == kActBf16;
  Problem p;
  p.weights = weights;
  p.x = x;
  p.scale = scale;
  p.zero_add = zero_add;
  p.n_out = n_out;
  p.k = k;
  p.ksteps = (int)(packed_steps & 0xffffu);
  p.steps_per_wave = 1;
  p.workgroups = workgroups;
  p.wgs_per_xcd = (workgroups + kNumXcd - 1) / kNumXcd;
  p.group_size = (int)(packed_group & 0xffffffu);
  p.tiles_per_wg = 1;
  const long long batch = blockIdx.z;
  long long owner;
  if (!place_problem(p, tail, packed_group, owner)) return;  // whole workgroup, before any barrier
  const bool has_bias = tail.bias != nullptr;
  tail.bias += owner * tail.stride_bias;
  tail.y += batch * tail.stride_y;
  const int m_batch = tail.m_batch;

  const int wg = logical_workgroup(p);
  if (wg >= p.workgroups) return;  // whole workgroup leaves before the barrier

  const int lane = threadIdx.x % kWave;
  const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // this wave's k step
  const int slice = lane / kTileRows;
  // Byte offset of the first row of this lane's scale / zero groups; a tile's entries are its row further on.
  // Rows past n_out (padding of the last tile) read the last row's: never stored.
  // (It takes preloaded arguments only, so it is held here, under the load of the others: 4096x4096 at 4 rows without
  // zeros 4.64 us, 4.73 behind them.)
  int group_offset[GROUPS_PER_RUN];
  {
    const int k_run = kw * G::kStepK + slice * G::kRunK;
#pragma unroll
    for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) {
      const int grp = QOP == MGEMV_PER_COLUMN_SCALE_ONLY ? 0 : group_of<GROUPS_PER_RUN>(p, k_run + gi * (G::kRunK / GROUPS_PER_RUN));
      group_offset[gi] = grp * p.n_out * 2;
      asm volatile("" : "+v"(group_offset[gi]));
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  const int waves = p.ksteps;
  const WaveWork work = valu_wave_work(true, wg, 0, 0, 1, tail.seq_base, tail.seq_rem, 0, 1, 1);
  const int tile0 = work.tile_begin;
  const int my_tiles = work.tiles;  // >= 1 by the host's geometry
  const int m = lane % kTileRows;
  // This workgroup's part of a left-over tile, and this wave's unit of it: `parts` k steps of 16 / parts rows (the mapping of
  // the part-tile kernel).  Everything else about the part is worked out where it is needed.
  const int parts = TAIL ? tiles_per_wg_of(packed_group) : 1;
  const int tail_tile = TAIL ? tail.seq_base * p.workgroups + wg / parts : 0;
  const bool has_tail = TAIL && tail_tile * kTileRows < p.n_out;
  const int tail_unit = TAIL ? kstat_tail_unit(kw, waves) : 0;
  const int tail_units = TAIL ? (waves + parts - 1) / parts : 0;
  const bool computes_tail = has_tail && tail_unit < tail_units;
  const int part_rows = kTileRows / parts;
  const int tail_row0 = tail_tile * kTileRows + wg % parts * part_rows;

  const int tile_stride = p.ksteps * kUnitBytes;  // bytes from a unit to the same k step of the next tile
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(
      p.weights + ((size_t)tile0 * (size_t)p.ksteps + (size_t)kw) * (size_t)kUnitBytes,
      (uint32_t)(my_tiles - 1) * (uint32_t)tile_stride + (uint32_t)kUnitBytes);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(p.x, (uint32_t)m_batch * (uint32_t)p.k * 2u);
  ScaleTables tables;
  const uint32_t table_bytes = (uint32_t)num_groups * (uint32_t)p.n_out * 2u;
  tables.scale = make_rsrc(p.scale, table_bytes);
  tables.zero = make_rsrc(p.zero_add, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS ? table_bytes : 0u);

  // A tile past the walk (the loop requests one or two) is sent past the tables: such a load comes back at
  // once, where a real one would have to land before the combine may reuse its register.
  auto offsets_of_tile = [&](int i, int (&off)[GROUPS_PER_RUN]) {
    const int row = (tile0 + i) * kTileRows + m;
    const uint32_t row_bytes = (uint32_t)(row < p.n_out ? row : p.n_out - 1) * 2u + (i < my_tiles ? 0u : 0x40000000u);
#pragma unroll
    for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) off[gi] = (int)((uint32_t)group_offset[gi] + row_bytes);
  };

  MfmaWeights<BITS, GROUPS_PER_RUN> wa, wb;
  auto request_first_unit = [&]() {
    int off[GROUPS_PER_RUN];
    offsets_of_tile(0, off);
    load_unit_mfma<BITS, GROUPS_PER_RUN, true, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS, ACT>(wa, w_rsrc, tables, lane * kChunkBytes, [&](int gi) { return off[gi]; });
  };
  // A unit of the part meets the rows of several waves.  Each wave says when its own are in its stage, and the first time a part's
  // unit looks they have long been there; the words are cleared in front of a barrier that waits for nothing but the waves'
  // starts.  (A barrier behind the rows costs 0.8 us a launch, one behind the walk 0.5, the rows fetched once more, straight to the
  // LDS, 0.5-1.)
  __shared__ uint32_t staged[TAIL ? kMaxWavesPerWorkgroup : 1];
  auto clear_staged = [&]() {
    if constexpr (TAIL) {
      if (lane == 0) staged[kw] = 0;
      __syncthreads();
    }
  };
  auto say_staged = [&]() {
    if constexpr (TAIL) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      if (lane == 0) __hip_atomic_store(&staged[kw], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  // Unit i of the walk; the one behind it is this wave's unit of the workgroup's part.
  auto request_unit = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& to, int i) {
    int off[GROUPS_PER_RUN];
    if (TAIL && computes_tail && i == my_tiles) {
      const int kstep = tail_unit * parts;
      const int steps = waves - kstep < parts ? waves - kstep : parts;
      const __amdgpu_buffer_rsrc_t part_rsrc = make_rsrc(
          p.weights + ((size_t)tail_tile * (size_t)p.ksteps + (size_t)kstep) * (size_t)kUnitBytes, (uint32_t)steps * (uint32_t)kUnitBytes);
      const int l = lane_after_loop(), k_part = l % kTileRows / part_rows, row_in_part = l % part_rows;
      const int row_raw = tail_row0 + row_in_part;
      const int row = row_raw < p.n_out ? row_raw : p.n_out - 1;
      const int k_run = (kstep + k_part) * G::kStepK + l / kTileRows * G::kRunK;
#pragma unroll
      for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) {
        const int grp = QOP == MGEMV_PER_COLUMN_SCALE_ONLY ? 0 : group_of<GROUPS_PER_RUN>(p, k_run + gi * (G::kRunK / GROUPS_PER_RUN));
        off[gi] = (grp * p.n_out + row) * 2;
      }
      load_unit_mfma<BITS, GROUPS_PER_RUN, true, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS, ACT>(
          to, part_rsrc, tables, k_part * kUnitBytes + (l / kTileRows * kTileRows + wg % parts * part_rows + row_in_part) * kChunkBytes, [&](int gi) { return off[gi]; });
    } else {
      offsets_of_tile(i, off);
      load_unit_mfma<BITS, GROUPS_PER_RUN, true, QOP == MGEMV_FINEGRAINED_SCALE_AND_ZEROS, ACT>(to, w_rsrc, tables, i * tile_stride + lane * kChunkBytes, [&](int gi) { return off[gi]; });
    }
  };
  // The activation operand: rows of this wave's k step come in whole (one fully coalesced load per row) and pass
  // through a stage that belongs to this wave alone.
  // (Read straight from x in operand shape, every load instruction touches 64 cache lines for 16 bytes each.)
  using XS = XStage<BITS>;
  const int stage_rows = kLdsOperand || TAIL ? m_batch : 8;
  uint8_t* const stage = reinterpret_cast<uint8_t*>(partials) + kw * (stage_rows * XS::kRowStride);
  __shared__ u32x4 zeros[kLdsOperand || TAIL ? kKStationaryZeroBytes / 16 : 1];
  typename KStatOperand<BITS, kLdsOperand>::type xa;
  clear_staged();
  if constexpr (kLdsOperand) {
    // The stage stays.
    for (int first = 0; first < m_batch; first += 8) {
      const int rows_here = m_batch - first < 8 ? m_batch - first : 8;
      XRows<BITS, 8> rows;
      fetch_x_rows<BITS, 8>(rows, p, x_rsrc, kw, lane, first, 1, rows_here);
      if (first == 0) request_first_unit();
      __builtin_amdgcn_sched_barrier(0);
      park_x_rows<BITS, 8>(rows, stage, lane, first, 1, rows_here);
    }
    say_staged();
    // Lanes of rows that do not exist read zeros: their columns of a matrix product are never stored, but the matrix unit
    // multiplies them all the same, and a large launch runs at the clock the power limit leaves (28672x8192 at 4 rows 1.92
    // GHz, its loads alone 2.32).  With row 0 in the idle columns that launch took 30.3 us, with zeros 29.4; 128256x4096 at
    // 2 rows 66.3 / 63.6, 28672x8064 g96 at 4 rows 33.2 / 32.3; up to 13 us level.
    if (lane < kKStationaryZeroBytes / 16) zeros[lane] = u32x4{0u, 0u, 0u, 0u};  // every wave for itself: no barrier
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the LDS executes a wave's accesses in order
    __builtin_amdgcn_wave_barrier();
    xa.lane_base = m < m_batch ? stage + m * XS::kRowStride + slice * (G::kRunK * 2) : reinterpret_cast<const uint8_t*>(zeros);
  } else {
    // ... and are read back in operand shape -- lane (slice, m) takes the sixteen 16-byte pieces of row m that its
    // matrix instructions pair with its weights.
    // More than 8 rows: a second round for the lanes of rows 8-15.  Lanes of rows that do not exist keep zeros.
    const uint8_t* const mine = stage + (m & 7) * XS::kRowStride + slice * (G::kRunK * 2);
#pragma unroll
    for (int i = 0; i < kBlocksPerUnit; ++i)
#pragma unroll
      for (int j = 0; j < (BITS == 4 ? 4 : 2); ++j) xa.x[i][j] = u32x4{0u, 0u, 0u, 0u};
    // Rows 8-15 are requested with the others: they are in registers that the operand takes later.  (In front of their own
    // turn, a load latency more, 4096x4096 at 16 rows took 5.85 us / 5.25, 11008x4096 8.3 / 7.8, 8192x8192 g64 12.7 / 12.1.
    // int8, whose rows are half as long, gains nothing.)  Four groups per run leave no registers for them: eight rows at a time,
    // in their own turn, spill 48 registers of the build with zeros, four at a time 16 (4096x4032 g96 at 16 rows 9.4 us / 7.35,
    // 8192x8064 22.1 / 17.5, 28672x8064 42.6 / 38.5; at 12 rows 0.95 of the time, up to 9 rows 1.02).
    constexpr bool kAllRowsAhead = BITS == 4 && GROUPS_PER_RUN != 4;
    constexpr int kLateRows = BITS == 4 ? 4 : 8;  // rows 8-15 requested at once where they are not ahead
    const int rows_ahead = m_batch < 8 ? m_batch : 8;
    XRows<BITS, 8> rows, more;
    fetch_x_rows<BITS, 8>(rows, p, x_rsrc, kw, lane, 0, 1, rows_ahead);
    if (kAllRowsAhead && m_batch > 8) fetch_x_rows<BITS, 8>(more, p, x_rsrc, kw, lane, 8, 1, m_batch - 8);
    // The first unit of weights is requested behind the rows of x (an L2 hit, back long before it):
    // the operand is turned round while the weights are still on their way.
    request_first_unit();
    __builtin_amdgcn_sched_barrier(0);
    auto read_back = [&](int first, int rows_here) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the LDS executes a wave's accesses in order
      __builtin_amdgcn_wave_barrier();
      if (m >= first && m < first + rows_here) {
#pragma unroll
        for (int i = 0; i < kBlocksPerUnit; ++i)
#pragma unroll
          for (int j = 0; j < (BITS == 4 ? 4 : 2); ++j)
            xa.x[i][j] = *reinterpret_cast<const u32x4*>(mine + (i * G::kChunkK + j * 8) * 2);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    park_x_rows<BITS, 8>(rows, stage, lane, 0, 1, rows_ahead);
    say_staged();
    read_back(0, rows_ahead);
    if (m_batch > 8) {
      if constexpr (kAllRowsAhead) {
        park_x_rows<BITS, 8>(more, stage, lane, 0, 1, m_batch - 8);
      } else {
        for (int first = 8; first < 16; first += kLateRows) {
          if (kLateRows < 8 && first >= m_batch) break;
          const int rows_here = m_batch - first < kLateRows ? m_batch - first : kLateRows;
          XRows<BITS, kLateRows> late_rows;
          fetch_x_rows<BITS, kLateRows>(late_rows, p, x_rsrc, kw, lane, first, 1, rows_here);
          park_x_rows<BITS, kLateRows>(late_rows, stage, lane, first - 8, 1, rows_here);
        }
      }
      read_back(8, m_batch - 8);
    }
  }
  if constexpr (TAIL) {
    if (!kLdsOperand && lane < kKStationaryZeroBytes / 16) zeros[lane] = u32x4{0u, 0u, 0u, 0u};
  }
  const bool park_behind_stage = kLdsOperand || TAIL || (tail.flags & kParkBehindStage) != 0;
  if (!park_behind_stage) __syncthreads();  // the stages make room for the partial sums
  const bool short_allowed = (tail.flags & kExactIntegerFormOnly) == 0;
  const ConvertRegs c = make_convert_regs();

  // Partial sums in LDS: for every (tile of the walk, row group, batch row) a block of 4, 8 or 16 entries of four floats, as
  // few as there is one for each wave, and one to spare; entry w is written by wave w (the odd block length spreads the lanes
  // over the banks, and the launch has room for blocks of 17).  The lane that later sums a block finds its entries side by
  // side, at offsets known to the compiler.  Blocks of 16 for every launch, those of missing waves zero, took fp16 launches of
  // up to 4 k steps 1.1-1.15 times as long and of 5-8 1.02-1.04 (36400x2048 at 4 rows 10.7 us / 9.35, 11008x4096 7.37 / 7.24;
  // a fourth size, 12, gains nothing and the choice costs the others 0.5 %).
  const int pieces = waves <= 4 ? 4 : waves <= 8 ? 8 : 16;
  const int slots = pieces + 1;
  f32x4* const park = reinterpret_cast<f32x4*>(reinterpret_cast<uint8_t*>(partials) +
                                               (park_behind_stage ? waves * (stage_rows * XS::kRowStride) : 0));
  const int park_tile_stride = kKSlices * m_batch * slots;  // entries from a tile to the next
  f32x4* my_park = park + (slice * m_batch + m) * slots + kw;
  bool parks = m < m_batch;
  // The unit of a left-over part: its operand and its entries take the place of the walk's.
  // (Through the loop itself, as one more unit of the walk, bf16 and longer walks lose 1-2 % and short fp16 ones gain as much.)
  auto turn_to_part = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& f) {
    const int l = lane_after_loop(), slice = l / kTileRows, k_part = l % kTileRows / part_rows, row_in_part = l % part_rows;
    const int kstep = tail_unit * parts + k_part;
    const uint8_t* const base =
        row_in_part < m_batch && kstep < waves
            ? reinterpret_cast<const uint8_t*>(partials) + (kstep * stage_rows + row_in_part) * XS::kRowStride + slice * (G::kRunK * 2)
            : reinterpret_cast<const uint8_t*>(zeros);
    const int of = tail_unit * parts + l % parts;
    // (every wave of the workgroup says so in front of its walk, whatever the others do)
    while (__builtin_amdgcn_ballot_w64(__hip_atomic_load(&staged[of < waves ? of : kw], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u) != 0)
      __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    if constexpr (kLdsOperand) {
      xa.lane_base = base;
    } else {
      const LdsActivations<BITS> from{base};
#pragma unroll
      for (int i = 0; i < kBlocksPerUnit; ++i)
#pragma unroll
        for (int j = 0; j < (BITS == 4 ? 4 : 2); ++j) xa.x[i][j] = mfma_operand<BITS>(from, i, j);
    }
    // K steps that are not there must not make a NaN of an infinite scale.  (In the last one an infinite scale does, where it is short, as in
    // whole tiles.)
    finite_past_reduction<ACT>(f.s, f.z, kstep, 0, waves);
    // The product's rows 4 * slice .. + 3 are the part's at one of the unit's k steps; a column is a batch row at one of them.
    const int quads = part_rows / 4;
    parks = slice / quads == k_part && row_in_part < m_batch;
    my_park = park + ((slice % quads) * m_batch + row_in_part) * slots + kstep;
  };
  auto compute_and_park = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& f, int i) {
    f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    half2_t col_scale = half2_t{};
    bool short_ok = short_allowed;
    if constexpr (QOP == MGEMV_PER_COLUMN_SCALE_ONLY) {
      col_scale = splat_low(f.s[0]);
    }
    if constexpr (PROBE == kProbeLoadsOnly) {
      uint32_t t = xa.x[0][0][0];
#pragma unroll
      for (int b = 0; b < kBlocksPerUnit; ++b) t ^= f.w[b][0] ^ f.w[b][1] ^ f.w[b][2] ^ f.w[b][3];
#pragma unroll
      for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) t ^= f.s[gi] ^ f.z[gi];
      acc[0] += __builtin_bit_cast(float, t & 0x3fffffffu);
    } else {
      compute_unit_mfma<BITS, QOP, GROUPS_PER_RUN, ACT>(acc, f, xa, c, col_scale, short_ok);
    }
    if (TAIL ? parks : m < m_batch) my_park[i * park_tile_stride] = acc;
  };
  // arithmetic-only build: the next unit is the first one again; the compiler must assume its registers changed
  auto repeat_first_unit = [&](MfmaWeights<BITS, GROUPS_PER_RUN>& to, const MfmaWeights<BITS, GROUPS_PER_RUN>& from) {
    to = from;
#pragma unroll
    for (int b = 0; b < kBlocksPerUnit; ++b) asm volatile("" : "+v"(to.w[b]));
#pragma unroll
    for (int gi = 0; gi < GROUPS_PER_RUN; ++gi) asm volatile("" : "+v"(to.s[gi]), "+v"(to.z[gi]));
  };

  // The loop begins at a 64-byte line: where its head fell on the last bytes of a 32-byte fetch, the fp16 build with
  // zeros took 1.02 of the time (71496x1792, groups of 256, 4 rows 18.3 us / 17.9; 128256x2048 at 8 rows 35.0 / 34.4).
  asm volatile(".p2align 6");
  int i = 0;
  do {
    if constexpr (PROBE == kProbeComputeOnly) {
      repeat_first_unit(wb, wa);
    } else {
      request_unit(wb, i + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    compute_and_park(wa, i);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PROBE == kProbeComputeOnly) {
      repeat_first_unit(wa, wb);
    } else {
      request_unit(wa, i + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < my_tiles) compute_and_park(wb, i + 1);
    __builtin_amdgcn_sched_barrier(0);
    i += 2;
  } while (i < my_tiles);
  if constexpr (TAIL) {
    if (computes_tail) {
      if (my_tiles & 1) wa = wb;  // requested last
      turn_to_part(wa);
      compute_and_park(wa, my_tiles);
    }
  }

  // The combine.  Wave r sums tiles r, r + waves, ... of the walk; lane (slice, m) the four rows
  // 4 * slice .. + 3 of batch row m.  A wave that reaches the barrier waits for the slowest one, and behind
  // the barrier it is alone on its SIMD, where every instruction costs its full latency: whatever does not
  // need the other waves' sums -- addresses, the bias, zeros in the entries of waves that do not exist --
  // is done in front of it.
  const int summed_tiles = my_tiles + (has_tail ? 1 : 0);
  const bool sums = m < m_batch && kw < summed_tiles;
  f32x4* block = park + ((kw * kKSlices + slice) * m_batch + m) * slots;
  int n0 = (tile0 + kw) * kTileRows + 4 * slice;
  uint16_t* dst = reinterpret_cast<uint16_t*>(tail.y) + (size_t)m * (size_t)p.n_out + n0;
  // the part: lanes of the first slices, one for every four of its rows
  auto move_to_part = [&]() {
    n0 = slice * 4 < part_rows ? tail_row0 + 4 * slice : p.n_out;
    dst = reinterpret_cast<uint16_t*>(tail.y) + (size_t)m * (size_t)p.n_out + n0;
  };
  if (TAIL && has_tail && kw == my_tiles) move_to_part();
  float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  auto fetch_bias = [&]() {
    if (has_bias) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = n0 + v < p.n_out ? n0 + v : p.n_out - 1;
        if constexpr (ACT == kActBf16)
          bias[v] = bf16_low_to_f32(reinterpret_cast<const uint16_t*>(tail.bias)[n]);
        else
          bias[v] = (float)tail.bias[n];
      }
    }
  };
  if (sums) {
    fetch_bias();
    if (TAIL || waves < pieces)
      for (int t = kw; t < summed_tiles; t += waves)
        for (int w = TAIL && t == my_tiles ? tail_units * parts : waves; w < pieces; ++w)
          block[(t - kw) * park_tile_stride + w] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const size_t dst_step = (size_t)waves * kTileRows;  // outputs from a tile this wave sums to the next
  const bool wide_store = ((reinterpret_cast<uintptr_t>(tail.y) | (uintptr_t)((size_t)p.n_out * 2)) & 7u) == 0;

  __syncthreads();
  if (sums) {
    for (int t = kw; t < summed_tiles; t += waves) {
      f32x4 sum;
      auto sum_block = [&](auto count) {
        f32x4 piece[decltype(count)::value];
#pragma unroll
        for (int w = 0; w < count; ++w) piece[w] = block[w];
        sum = piece[0];
#pragma unroll
        for (int w = 1; w < count; ++w) sum += piece[w];  // ascending k
      };
      switch (pieces) {
        case 4: sum_block(std::integral_constant<int, 4>{}); break;
        case 8: sum_block(std::integral_constant<int, 8>{}); break;
        default: sum_block(std::integral_constant<int, 16>{});
      }
      // n_out is a multiple of 4 and so is n0: the four outputs of a lane are all inside or all outside, and
      // they are neighbours in y -- one 8-byte store where y allows it
      if (n0 < p.n_out) {
        float r[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = epilogue_value(tail, sum[v], has_bias, bias[v]);
        uint32_t lo, hi;
        if constexpr (ACT == kActBf16) {
          lo = pack_bf16(r[0], r[1]);
          hi = pack_bf16(r[2], r[3]);
        } else {
          lo = as_u32(half2_t{(half_t)r[0], (half_t)r[1]});
          hi = as_u32(half2_t{(half_t)r[2], (half_t)r[3]});
        }
        if (wide_store) {
          *reinterpret_cast<u32x2*>(dst) = u32x2{lo, hi};
        } else {
          dst[0] = (uint16_t)lo; dst[1] = (uint16_t)(lo >> 16); dst[2] = (uint16_t)hi; dst[3] = (uint16_t)(hi >> 16);
        }
      }
      // walks longer than the workgroup has waves: on to this wave's next tile
      block += waves * park_tile_stride;
      n0 += waves * kTileRows;
      dst += dst_step;
      if (TAIL && has_tail && t + waves == my_tiles) move_to_part();
      if (t + waves < summed_tiles) fetch_bias();
    }
  }
}

template <int BITS, int QOP, int GPR, int ACT, int PROBE = kProbeNone, bool TAIL = false>
hipError_t launch_mfma_kstat_kernel(const GemvLaunch& g) {
  if constexpr (!TAIL) {
    if (g.plan.parts != 0) {  // whole tiles only would leave the rest of the matrix out, in stages of another size
      if constexpr (PROBE == kProbeNone && kstat_has_left_over_parts(BITS, GPR, ACT))
        return launch_mfma_kstat_kernel<BITS, QOP, GPR, ACT, PROBE, true>(g);
      else
        return hipErrorInvalidValue;
    }
  }
  const auto kernel = gemv_mfma_kstat_kernel<BITS, QOP, GPR, ACT, PROBE, TAIL>;
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
                pack_steps(num_ksteps(g.k, BITS), 1), g.plan.workgroups, g.tail.num_groups,
                pack_group(g.group_size, TAIL ? g.plan.parts : 1, g.tail.stack != nullptr),
                g.tail);
}

template <int BITS, int QOP, int ACT>
hipError_t launch_mfma_kstat_gpr(const GemvLaunch& g, int gpr) {
  if constexpr (QOP == MGEMV_PER_COLUMN_SCALE_ONLY) {
    return launch_mfma_kstat_kernel<BITS, QOP, 1, ACT>(g);
  } else {
    switch (gpr) {
      case 1: return launch_mfma_kstat_kernel<BITS, QOP, 1, ACT>(g);
      case 2: return launch_mfma_kstat_kernel<BITS, QOP, 2, ACT>(g);
      default: return launch_mfma_kstat_kernel<BITS, QOP, 4, ACT>(g);
    }
  }
}

template <int ACT>
hipError_t launch_mfma_kstat_act(const GemvLaunch& g, int bits, int qop, int gpr) {
  if (bits == 4) {
    switch (qop) {
      case 1: return launch_mfma_kstat_gpr<4, 1, ACT>(g, gpr);
      case 2: return launch_mfma_kstat_gpr<4, 2, ACT>(g, gpr);
      default: return launch_mfma_kstat_gpr<4, 3, ACT>(g, gpr);
    }
  }
  switch (qop) {
    case 1: return launch_mfma_kstat_gpr<8, 1, ACT>(g, gpr);
    case 2: return launch_mfma_kstat_gpr<8, 2, ACT>(g, gpr);
    default: return launch_mfma_kstat_gpr<8, 3, ACT>(g, gpr);
  }
}

// Measurement builds exist for int4 scale-and-zero fp16 launches with one or two groups per lane run.
bool mfma_kstat_probe_exists(int bits, int qop, int gpr, int act) {
  return bits == 4 && qop == MGEMV_FINEGRAINED_SCALE_AND_ZEROS && (gpr == 1 || gpr == 2) && act == kActF16;
}

hipError_t launch_mfma_kstat_probe(const GemvLaunch& g, int gpr, int probe) {
  constexpr int kQ = MGEMV_FINEGRAINED_SCALE_AND_ZEROS;
  if (probe == kProbeLoadsOnly)
    return gpr == 1 ? launch_mfma_kstat_kernel<4, kQ, 1, kActF16, kProbeLoadsOnly>(g)
                    : launch_mfma_kstat_kernel<4, kQ, 2, kActF16, kProbeLoadsOnly>(g);
  return gpr == 1 ? launch_mfma_kstat_kernel<4, kQ, 1, kActF16, kProbeComputeOnly>(g)
                  : launch_mfma_kstat_kernel<4, kQ, 2, kActF16, kProbeComputeOnly>(g);
}

hipError_t launch_mfma_kstat(const GemvLaunch& g, int bits, int qop, int gpr, int act) {
  if (act == kActBf16) return launch_mfma_kstat_act<kActBf16>(g, bits, qop, gpr);
  return launch_mfma_kstat_act<kActF16>(g, bits, qop, gpr);
}

}  // namespace mgemv
