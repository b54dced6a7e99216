// Device-side numeric building blocks for gfx950: the biased-integer -> fp16 converters, the
// two-rounding dequantiser and the DPP-broadcast dot product.  Everything here is wave64
// VALU code; nothing in this file is shared with or derived from a CUDA path.
#ifndef MIXED_GEMV_AMD_DEVICE_MATH_H_
#define MIXED_GEMV_AMD_DEVICE_MATH_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

// The dequantiser is "fp16 multiply, then fp16 add", two separately rounded operations
// (gemv/warp/warp_dequantizer.h:52-59).  A contracted v_pk_fma_f16 rounds once and changes
// bits, so contraction is switched off for everything that includes this header (the build
// also passes -ffp-contract=off).
#pragma clang fp contract(off)

namespace mgemv {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ half2_t as_half2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }
__device__ __forceinline__ uint32_t as_u32(half2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ half2_t splat(half_t v) { return half2_t{v, v}; }

// Register-resident constants for the converters.  VOP3 encodings on this target take no
// 32-bit literal, so (w & mask) | magic only becomes a single v_and_or_b32 when mask and
// magic already sit in registers; the empty asm keeps the compiler from folding them back
// into literals (which would split the operation into v_and + v_or).
struct ConvertRegs {
  uint32_t mask7;     // 0x07800780   the 4-bit field at bits 7-10 of each 16-bit half
  uint32_t mask3;     // 0x00780078   the 4-bit field at bits 3-6 of each 16-bit half
  uint32_t magic;     // 0x64006400   fp16 1024.0 in both halves      (general form only)
  uint32_t minus136;  // 0xd840d840   fp16 -136.0 in both halves      (general form only)
  uint32_t sel_lo;    // v_perm selector: bytes 0,1 of a word into the low byte of each half
  uint32_t sel_hi;    // v_perm selector: bytes 2,3
};

__device__ __forceinline__ ConvertRegs make_convert_regs() {
  ConvertRegs c;
  c.mask7 = 0x07800780u;
  c.mask3 = 0x00780078u;
  c.magic = 0x64006400u;
  c.minus136 = 0xd840d840u;
  c.sel_lo = 0x04010400u;
  c.sel_hi = 0x04030402u;
  asm("" : "+s"(c.mask7));
  asm("" : "+s"(c.mask3));
  asm("" : "+s"(c.magic));     // parked in SGPRs; general_form_regs() moves them where they are needed
  asm("" : "+s"(c.minus136));
  asm("" : "+s"(c.sel_lo));
  asm("" : "+s"(c.sel_hi));
  return c;
}

// The general form needs its two packed constants in VGPRs (a VOP3 instruction reads at most
// one SGPR).  They are copied there at the start of each general-form unit instead of living
// in VGPRs for the whole kernel, where they would cost the short form a wave of occupancy.
__device__ __forceinline__ ConvertRegs general_form_regs(ConvertRegs c) {
  asm volatile("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3" : "=&v"(c.magic), "=v"(c.minus136) : "s"(c.magic), "s"(c.minus136));
  return c;
}

__device__ __forceinline__ uint32_t rotate_right_8(uint32_t w) { return __builtin_amdgcn_alignbit(w, w, 8); }

// int4, general form: one stored word (8 biased 4-bit fields in the order of tile_layout.h)
// -> 8 fp16 values, exact integers in [-8, 7], as 4 packed pairs in ascending k.
//   (v & 0x00780078) | 0x6400_6400  is the pair (1024 + 8 u, 1024 + 8 u');  * 1/8 - 136 -> u - 8
// for v = w >> 4, w, rotr(w, 12) and w >> 8.  Every step is exact in fp16.  This is the
// numeric contract of gemv/interleaved_numeric_conversion.h:232-291 (lop3 / sub.f16x2 /
// fma.rn.f16x2: biased nibble under a 1024.0 exponent, then an exact affine map) expressed
// in v_alignbit_b32, v_and_or_b32 and v_pk_fma_f16.  (It shares no intermediate with the
// short form below, so the compiler has nothing to hoist in front of the branch between them.)
__device__ __forceinline__ void convert_int4_word(uint32_t w, const ConvertRegs& c, half2_t (&q)[4]) {
  const half2_t h0 = as_half2(((w >> 4) & c.mask3) | c.magic);
  const half2_t h1 = as_half2((w & c.mask3) | c.magic);
  const half2_t h2 = as_half2((__builtin_amdgcn_alignbit(w, w, 12) & c.mask3) | c.magic);
  const half2_t h3 = as_half2(((w >> 8) & c.mask3) | c.magic);
  const half2_t k8th = splat((half_t)0.125f);
  const half2_t kn136 = as_half2(c.minus136);
  q[0] = __builtin_elementwise_fma(h0, k8th, kn136);
  q[1] = __builtin_elementwise_fma(h1, k8th, kn136);
  q[2] = __builtin_elementwise_fma(h2, k8th, kn136);
  q[3] = __builtin_elementwise_fma(h3, k8th, kn136);
}

// int4, short form for a positive scale s below 2^-5.  A masked half-word read as fp16 IS
// u * 2^-17 (field at bits 7-10) or u * 2^-21 (field at bits 3-6), exactly; with the scale
// pre-multiplied by 2^17 / 2^21 (exact: s * 2^21 <= 65504) a single fused multiply-add
//     fma(u * 2^-p, s * 2^p, -8 s)  =  rn16(u s - 8 s)  =  rn16((u - 8) * s)
// rounds the exact product once, which is bit for bit the rn16(q * s) of
// gemv/warp/warp_dequantizer.h:52-59; the additive zero then follows as its own rounded
// add.  8 s is exact, and for s > 0 a zero product is +0 on both routes.  Outside
// 0 < s < 2^-5 (large, zero, negative, NaN) the general form above is used instead.
struct ShortFormScale {
  half2_t s17;   // (s * 2^17, s * 2^17)
  half2_t s21;   // (s * 2^21, s * 2^21)
  half2_t m8s;   // (-8 s, -8 s)
};

// fp16 bit patterns of the scales for which the short form is exact: 0x0001 .. 0x27ff.
constexpr uint32_t kShortF16First = 0x0001, kShortF16Past = 0x2800;

__device__ __forceinline__ ShortFormScale make_short_form_scale(half2_t s2) {
  ShortFormScale f;
  const half2_t a = s2 * splat((half_t)32768.0f);  // 2^17 itself is not an fp16 value
  f.s17 = a * splat((half_t)4.0f);
  f.s21 = f.s17 * splat((half_t)16.0f);
  f.m8s = s2 * splat((half_t)-8.0f);
  return f;
}

template <bool HAS_ZERO>
__device__ __forceinline__ void dequant_int4_word_short(uint32_t w, const ConvertRegs& c, const ShortFormScale& f,
                                                        half2_t z2, half2_t (&d)[4]) {
  const uint32_t t = rotate_right_8(w);
  d[0] = __builtin_elementwise_fma(as_half2(w & c.mask7), f.s17, f.m8s);
  d[1] = __builtin_elementwise_fma(as_half2(w & c.mask3), f.s21, f.m8s);
  d[2] = __builtin_elementwise_fma(as_half2(t & c.mask7), f.s17, f.m8s);
  d[3] = __builtin_elementwise_fma(as_half2(t & c.mask3), f.s21, f.m8s);
  if (HAS_ZERO) {
#pragma unroll
    for (int h = 0; h < 4; ++h) d[h] = d[h] + z2;
  }
}

// int8: one stored word (4 biased bytes, natural order) -> 4 fp16 exact integers in
// [-128, 127] as 2 packed pairs.  v_perm_b32 drops each byte under a 0x64 high byte
// (1024 + u), then minus 1152 -> u - 128.  Bit-level contract of
// gemv/interleaved_numeric_conversion.h:62-81 (prmt / sub.f16x2).
__device__ __forceinline__ void convert_int8_word(uint32_t w, const ConvertRegs& c, half2_t (&q)[2]) {
  const uint32_t sixty_four = 0x64646464u;
  const half2_t h0 = as_half2(__builtin_amdgcn_perm(sixty_four, w, c.sel_lo));
  const half2_t h1 = as_half2(__builtin_amdgcn_perm(sixty_four, w, c.sel_hi));
  const half2_t k1152 = splat((half_t)1152.0f);
  q[0] = h0 - k1152;
  q[1] = h1 - k1152;
}

// Dequantise one packed pair: rn16(rn16(q * s) + z) or rn16(q * s).
// gemv/warp/warp_dequantizer.h:52-59 (with zero) and :86-92 (without).
template <bool HAS_ZERO>
__device__ __forceinline__ half2_t dequant_pair(half2_t q, half2_t s, half2_t z) {
  half2_t d = q * s;
  if (HAS_ZERO) d = d + z;
  return d;
}

// acc += d.lo * x.lo + d.hi * x.hi in fp32, where x is read from lane SRC of the caller's
// DPP row (16 lanes) instead of the caller's own register: v_dot2c_f32_f16 with a
// row_newbcast DPP control.  This replaces gemv/thread/mma.h:83-95 (one scalar fp32 FMA per
// weight) and the register broadcast of the activation fragment
// (gemv/threadblock/dq_mma_base.h:76-103).
//
// The x operand must come straight from a memory load: a VALU write followed within two
// instructions by a DPP read of the same register is a hazard that neither the assembler nor
// the compiler (which sees an opaque asm statement) pads.  Nothing in the sources can stop the
// register allocator from copying x or the accumulator at a bad place, so the build checks the
// compiled code instead: isa_lint.py walks the device assembly of every kernel and fails the
// build on a VALU write within two wait states in front of a DPP read, or a read of a dot
// result by any other kind of instruction within three behind it.
template <int SRC>
__device__ __forceinline__ void dot2_row_bcast(float& acc, uint32_t x, half2_t d) {
  static_assert(SRC >= 0 && SRC < 16, "source lane within a 16-lane DPP row");
  // Instructions of 8 bytes that lie across an 8-byte boundary are fetched late.  Most of a unit's are dots and multiply-adds of
  // 8 bytes, one run of them per block with a single one of 4 in between (a wait), so whole units lie well or badly by the
  // length of what is in front: the int8 loops had 25 to 76 % of theirs across a boundary.  Each block's first dot is aligned,
  // at the price of an s_nop where it was not: 16-36 % in int8, 44-47 % in int4, whose conversions mix both lengths.
  // Before / here: int8 walks of 3 and 4 rows 0.95 of the time, longer waves of 2-4 rows 0.98-0.985 (20000x8192 at 3 rows 30.2 us /
  // 29.3), int4 0.985-0.995 (7004x17408 at 2 rows 17.8 / 16.45, 5120x13824 13.4 / 13.2); means of 207 builds over 17500 fp16
  // launches 0.94-1.017.  Aligning every dot costs int4 2-4 % (121 s_nops a pair of units); bf16, whose conversions
  // are longer, gains in the loop and loses as much in the other builds.
  if constexpr (SRC % 4 == 0)
    asm(".p2align 3\n\tv_dot2c_f32_f16_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(acc)
        : "v"(x), "v"(d), "n"(SRC));
  else
    asm("v_dot2c_f32_f16_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(acc)
        : "v"(x), "v"(d), "n"(SRC));
}

// The same with x from lane SRC of the caller's four lanes.
template <int SRC>
__device__ __forceinline__ void dot2_quad_bcast(float& acc, uint32_t x, half2_t d) {
  static_assert(SRC >= 0 && SRC < 4, "source lane within four lanes");
  if constexpr (SRC == 0)
    asm(".p2align 3\n\tv_dot2c_f32_f16_dpp %0, %1, %2 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(d));
  else
    asm("v_dot2c_f32_f16_dpp %0, %1, %2 quad_perm:[%3,%3,%3,%3] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(d), "n"(SRC));
}

// The compiler does not know the asm above is a dot instruction, so it cannot pad the
// "dot result read by a different instruction" hazard of this target (3 wait states).
// Call this once after the last dot of a chain, before the accumulator is consumed.
__device__ __forceinline__ void settle_dot_chain(float& acc) { asm volatile("s_nop 4" : "+v"(acc)); }

// ---------------------------------------------------------------------------------------------
// bfloat16 activations / scales / outputs.
//
// The reference's bf16 converters (gemv/interleaved_numeric_conversion.h:130-183 for int8,
// :340-401 for int4) produce the exact integer q as a bf16, and its dequantiser
// (gemv/warp/warp_dequantizer.h:52-59) multiplies by the scale and adds the zero term, each
// rounded to bf16.  This target has no packed bf16 arithmetic, so both steps run in fp32, where
// q * s is exact (at most 8 x 8 significant bits), and v_cvt_pk_bf16_f32 rounds to nearest even;
// for the sum, rounding the fp32 sum to bf16 equals rounding the exact sum once (24 >= 2*8+2).
// Values are kept as packed pairs of bf16 bit patterns, (low, high) = ascending k.
//
// Two forms each, as for fp16:
//   short    int4: the products of the fp16 short form, exact in fp16, widened to fp32 by the matrix unit and rounded
//            (dequant_int4_words_bf16); int8: fma(u, s, -128 s), exact for 2^-100 <= s < 2^119;
//   general  (8u - 64) * (s/8) resp. (u - 128) * s: exact for every finite s, with the sign of
//            a zero product as the reference's multiply gives it.
// ---------------------------------------------------------------------------------------------
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kActF16 = 0;
constexpr int kActBf16 = 1;

__device__ __forceinline__ float bf16_low_to_f32(uint32_t bits) { return __builtin_bit_cast(float, bits << 16); }
__device__ __forceinline__ float bf16_high_to_f32(uint32_t bits) { return __builtin_bit_cast(float, bits & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2_t));
}
template <int BYTE>
__device__ __forceinline__ float byte_to_f32(uint32_t v) {
  return (float)((v >> (8 * BYTE)) & 0xffu);  // v_cvt_f32_ubyteN
}

// Which scales the short form takes, by bf16 bit pattern.
// int8: 2^-100 .. 2^119 -- positive, every product with an integer a normal number, -128 s finite.
// int4: the products q s have 11 significant bits and must not fall off either end of fp16: 2^-17 <= s < 2^-5, or 2^shift
// times that, any shift that is the same for the four lanes of a widening step (which takes it back).
constexpr uint32_t kShortBf16Int8First = 0x0d80, kShortBf16Int8Past = 0x7b00;
constexpr uint32_t kShortBf16Int4FirstExponent = 127 - 17, kShortBf16Int4Binades = 12;
constexpr uint32_t kShortBf16Int4First = kShortBf16Int4FirstExponent << 7;
constexpr uint32_t kShortBf16Int4Past = (kShortBf16Int4FirstExponent + kShortBf16Int4Binades) << 7;
constexpr int kShortBf16MinShift = -14, kShortBf16MaxShift = 15;  // 2^shift is a normal fp16 value

// A lane's int4 scale for the short bf16 form: s 2^-shift, and 2^shift twice, as fp16.
struct Int4ScaleBf16 {
  float s;
  uint32_t power;
};
constexpr uint32_t kNoShift = 0x3c003c00u;

// One lane's row of the 4x4 identity, as a mask on four packed 16-bit values: the operand of the widening steps below.
struct Identity4 {
  uint32_t lo, hi;
};
__device__ __forceinline__ Identity4 make_identity4() {
  const uint32_t row = threadIdx.x & 3u;  // lane i of each four holds row i
  const uint32_t half = (row & 1u) != 0 ? 0xffff0000u : 0x0000ffffu;
  return Identity4{row < 2 ? half : 0u, row < 2 ? 0u : half};
}

// v_mfma_f32_4x4x4_16b with the 4x4 identity as one operand gives every lane its own four 16-bit values back as fp32 --
// times the identity's value, plus the lane's accumulator operand: one instruction of 8 cycles on the otherwise idle
// matrix unit in place of four conversions (and four additions) of the vector unit.  Every instruction these kernels issue costs
// a wave about 4.3 cycles (measured with 4 waves per SIMD), so what counts is their number.
// The other three values of a lane's block meet zero factors: all of them must be finite.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 widen_f16(const u32x2& identity, half2_t a, half2_t b) {
  return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(half4_t, identity), __builtin_bit_cast(half4_t, u32x2{as_u32(a), as_u32(b)}),
                                            f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}
// Bf16 values plus the additive zero, rounded to bf16, PAIRS packed pairs at a time.  r + z carries at most 17 significant
// bits wherever it comes near the middle between two bf16 values, so its rounding to bf16 is that of the exact sum (checked
// on the device against the vector unit over 8e8 pairs, subnormal zeros included).
// A matrix instruction's result is there five issue slots later.  The barriers keep the compiler from lining up each
// instruction with its own conversions, where it would have to fill those slots with waits (100 of them a unit): first all
// instructions, then all conversions.
template <int PAIRS>
__device__ __forceinline__ void add_zero_bf16(uint32_t (&d)[PAIRS], const u32x2& identity, const f32x4& z) {
  f32x4 sum[PAIRS / 2];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < PAIRS / 2; ++i)
    sum[i] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, identity),
                                                    __builtin_bit_cast(s16x4, u32x2{d[2 * i], d[2 * i + 1]}), z, 0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < PAIRS / 2; ++i) {
    d[2 * i] = pack_bf16(sum[i][0], sum[i][1]);
    d[2 * i + 1] = pack_bf16(sum[i][2], sum[i][3]);
  }
}

struct Bf16Scale {
  float mul;              // int4, general: s/8; int8: s
  float add;              // int8, short: -128 s
  f32x4 z;                // additive zero, four times: the accumulator operand of add_zero_bf16
  ShortFormScale f16;     // int4, short: of s * 2^-shift
  u32x2 widen, identity;  // int4, short: 2^shift (fp16) and 1 (bf16) times the lane's row of the identity
};

// short4: int4 short form only (which does not read s_bits).
template <int BITS, bool SHORT>
__device__ __forceinline__ Bf16Scale make_bf16_scale(uint32_t s_bits, uint32_t z_bits, const Identity4& id, const Int4ScaleBf16& short4) {
  const float s = bf16_low_to_f32(s_bits), z = bf16_low_to_f32(z_bits);
  Bf16Scale f{};
  if constexpr (BITS == 4 && SHORT) {
    auto scaled = [&](float power) { return splat((half_t)(short4.s * power)); };  // exact
    f.f16.s17 = scaled(0x1p17f);
    f.f16.s21 = scaled(0x1p21f);
    f.f16.m8s = scaled(-8.0f);
    f.widen = u32x2{id.lo & short4.power, id.hi & short4.power};
  } else {
    f.mul = BITS == 4 ? s * 0.125f : s;
    f.add = s * -128.0f;
  }
  f.identity = u32x2{id.lo & 0x3f803f80u, id.hi & 0x3f803f80u};
  f.z = f32x4{z, z, z, z};
  return f;
}

// General form.  (a, b): the integers 8u (int4) or u (int8) of a k-adjacent pair -> packed bf16 pair of
// rn(rn(q s) + z) resp. rn(q s).  (The products may overflow, so the sum stays on the vector unit.)
template <int BITS, bool HAS_ZERO>
__device__ __forceinline__ uint32_t dequant_pair_bf16(float a, float b, const Bf16Scale& f) {
  constexpr float kBias = BITS == 4 ? 64.0f : 128.0f;
  uint32_t d = pack_bf16((a - kBias) * f.mul, (b - kBias) * f.mul);
  if constexpr (HAS_ZERO) d = pack_bf16(bf16_low_to_f32(d) + f.z[0], bf16_high_to_f32(d) + f.z[0]);
  return d;
}

// WORDS words of int4 (field positions: tile_layout.h), 8 WORDS weights, to packed bf16 pairs in ascending k.
// Short: 17 vector and 4 matrix instructions a word with a zero, 13 and 2
// without; 98 cycles a word and SIMD with the product's matrix instruction (4 waves; the scale applied in fp32, one field at
// a time, 122; v_dot2_f32_bf16 on packed pairs, with the zero, 35 instructions).
// General: a field masked at bits 3-6 of a byte converts to 8u.
template <bool HAS_ZERO, bool SHORT, int WORDS>
__device__ __forceinline__ void dequant_int4_words_bf16(const uint32_t (&words)[WORDS], const ConvertRegs& c, const Bf16Scale& f,
                                                        uint32_t (&d)[4 * WORDS]) {
  if constexpr (SHORT) {
    half2_t q[WORDS][4];
#pragma unroll
    for (int i = 0; i < WORDS; ++i) dequant_int4_word_short<false>(words[i], c, f.f16, half2_t{}, q[i]);  // q s 2^-shift, exact
    f32x4 p[2 * WORDS];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * WORDS; ++i) p[i] = widen_f16(f.widen, q[i / 2][2 * (i % 2)], q[i / 2][2 * (i % 2) + 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * WORDS; ++i) {
      d[2 * i] = pack_bf16(p[i][0], p[i][1]);
      d[2 * i + 1] = pack_bf16(p[i][2], p[i][3]);
    }
    if constexpr (HAS_ZERO) add_zero_bf16(d, f.identity, f.z);
  } else {
    uint32_t mask = c.mask3;  // a value of its own: shared masked words would be computed, and kept, in front of the branch between the forms
    asm("" : "+s"(mask));
#pragma unroll
    for (int i = 0; i < WORDS; ++i) {
      const uint32_t w = words[i];
      const uint32_t e01 = (w >> 4) & mask;
      const uint32_t e23 = w & mask;
      const uint32_t e45 = __builtin_amdgcn_alignbit(w, w, 12) & mask;
      const uint32_t e67 = w & 0x78007800u;
      d[4 * i + 0] = dequant_pair_bf16<4, HAS_ZERO>(byte_to_f32<0>(e01), byte_to_f32<2>(e01), f);
      d[4 * i + 1] = dequant_pair_bf16<4, HAS_ZERO>(byte_to_f32<0>(e23), byte_to_f32<2>(e23), f);
      d[4 * i + 2] = dequant_pair_bf16<4, HAS_ZERO>(byte_to_f32<0>(e45), byte_to_f32<2>(e45), f);
      d[4 * i + 3] = dequant_pair_bf16<4, HAS_ZERO>(byte_to_f32<1>(e67), byte_to_f32<3>(e67), f);
    }
  }
}

// WORDS words of int8: 4 biased bytes each in natural order.
template <bool HAS_ZERO, bool SHORT, int WORDS>
__device__ __forceinline__ void dequant_int8_words_bf16(const uint32_t (&words)[WORDS], const Bf16Scale& f, uint32_t (&d)[2 * WORDS]) {
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    const uint32_t w = words[i];
    if constexpr (SHORT) {
      d[2 * i] = pack_bf16(__builtin_fmaf(byte_to_f32<0>(w), f.mul, f.add), __builtin_fmaf(byte_to_f32<1>(w), f.mul, f.add));
      d[2 * i + 1] = pack_bf16(__builtin_fmaf(byte_to_f32<2>(w), f.mul, f.add), __builtin_fmaf(byte_to_f32<3>(w), f.mul, f.add));
    } else {
      d[2 * i] = dequant_pair_bf16<8, HAS_ZERO>(byte_to_f32<0>(w), byte_to_f32<1>(w), f);
      d[2 * i + 1] = dequant_pair_bf16<8, HAS_ZERO>(byte_to_f32<2>(w), byte_to_f32<3>(w), f);
    }
  }
  if constexpr (SHORT && HAS_ZERO) add_zero_bf16(d, f.identity, f.z);
}

// bf16 counterpart of dot2_row_bcast (same hazards, same settle_dot_chain afterwards).
template <int SRC>
__device__ __forceinline__ void dot2_row_bcast_bf16(float& acc, uint32_t x, uint32_t d) {
  static_assert(SRC >= 0 && SRC < 16, "source lane within a 16-lane DPP row");
  asm("v_dot2c_f32_bf16_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(x), "v"(d), "n"(SRC));
}

template <int SRC>
__device__ __forceinline__ void dot2_quad_bcast_bf16(float& acc, uint32_t x, uint32_t d) {
  static_assert(SRC >= 0 && SRC < 4, "source lane within four lanes");
  asm("v_dot2c_f32_bf16_dpp %0, %1, %2 quad_perm:[%3,%3,%3,%3] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(d), "n"(SRC));
}

// Raw buffer descriptor: base pointer + byte count; out-of-range lanes read zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

constexpr int kCacheDefault = 0;
constexpr int kCacheStream = 2;  // "nt": weights are read once, keep them from displacing x / scales

}  // namespace mgemv

#endif  // MIXED_GEMV_AMD_DEVICE_MATH_H_
