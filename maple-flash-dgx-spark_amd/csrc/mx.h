// Scaled 8-bit and 4-bit matrix instructions (gfx950) for the packed codes.
//
// v_mfma_scale_f32_16x16x128_f8f6f4 takes each operand in its own small float
// format with one power-of-two scale per 32 values of K, and this card reaches
// 4.3 PFLOP/s with it against 1.3 with v_mfma_f32_16x16x32_bf16 (eight
// independent accumulators a wave, both measured).  Two properties fit it to
// packed codes and bf16 activations:
//
//  * A code c in 0..3 as the bits of an FP4 (E2M1) number reads as c / 2, so a
//    packed ternary word becomes two operand registers with one shift and two
//    ANDs (expand_word needs 12 instructions for its 8 bf16 registers).  With
//    the weights' scale at 2 the product is sum c x, and the ternary product
//    is sum c x - sum x.
//  * A bf16 value has 8 significant bits and FP8 (E4M3) 4, so x = p0 + p1 / 16
//    exactly, p0 the nearest E4M3 number and p1 sixteen times what is left
//    (values 2^13 below their block's largest lose bits below 2^-20 of that
//    largest).  Each further piece takes 4 to 5 more bits: four carry a float32
//    product to 2^-19 of itself or 2^-29 of that largest.  The pieces cost what one
//    bf16 pass would at twice the rate; what is saved is the expansion.
//
// Lane layout of 16x16x128 (checked on the device; logical K index k):
//   FP4 A: lane l holds row l % 16, k = 32 (l / 16) + nibble (4 registers)
//   FP8 B: lane l holds col l % 16, byte i < 16: k = 16 (l / 16) + i,
//          i >= 16: k = 64 + 16 (l / 16) + i - 16 (8 registers)
//   scales: byte 0 of lane l's scale register is 2^(byte - 127) for k / 32 == l / 16
//   C: lane l holds col l % 16, rows 4 (l / 16) ..+3
//
// Row format of the activations ("mx rows"), NP pieces: per step of 128 values
// (8 packed words) NP runs of 128 bytes; word w of the step fills bytes 16 w
// ..+15 of each run with its even values, then its odd ones -- the order that
// the two ANDs above leave the codes in.  Beside them one uint32 per row and
// step: byte b is the exponent of the step's values 32 b ..+31.
#pragma once

#include "common.h"

namespace ma {

typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float mx_f32x4_t __attribute__((ext_vector_type(4)));
typedef float mx_f32x2_t __attribute__((ext_vector_type(2)));

constexpr int kMxStep = 128;  // values of K per step

// Scale byte of the weights against piece p: 2 (FP4 reads a code as c / 2) over 16^p.
constexpr int mx_piece_scale(int p) { return 128 - 4 * p; }

// acc += codes (FP4) x pieces (FP8), 16 x 16 x 128.
__device__ __forceinline__ mx_f32x4_t mx_mfma_fp4(const uint32_t (&a)[4], i32x8_t b, mx_f32x4_t acc, int sa, int sb) {
  const i32x8_t av = {static_cast<int>(a[0]), static_cast<int>(a[1]), static_cast<int>(a[2]), static_cast<int>(a[3]),
                      0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, b, acc, 4, 0, 0, sa, 0, sb);
}

// Keeps the products that form these sums before, and every load after, this
// point (left alone, the compiler issues a step's reads first and all of its
// products last, with the operands of the whole step in registers).
__device__ __forceinline__ void mx_pin(mx_f32x4_t& a, mx_f32x4_t& b, mx_f32x4_t& c, mx_f32x4_t& d) {
  asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d)::"memory");
}

// The FP8 operand of a lane: chunks g and 4 + g of its column's 128 bytes.
__device__ __forceinline__ i32x8_t mx_operand(uint4 lo, uint4 hi) {
  return i32x8_t{static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z), static_cast<int>(lo.w),
                 static_cast<int>(hi.x), static_cast<int>(hi.y), static_cast<int>(hi.z), static_cast<int>(hi.w)};
}

// The FP4 operand of two packed ternary words.
__device__ __forceinline__ void mx_expand2(uint2 w, uint32_t (&a)[4]) {
  a[0] = w.x & 0x33333333u;
  a[1] = (w.x >> 2) & 0x33333333u;
  a[2] = w.y & 0x33333333u;
  a[3] = (w.y >> 2) & 0x33333333u;
}

// The largest exponent field of some values (255 if one is not finite); taken
// over a block of 32, it gives the block's scale byte and the factor that
// brings the values under 2^8, where E4M3 (largest value 448) holds them after
// rounding.  255 stays 255, a NaN scale, so such a block's row becomes NaN.
__device__ __forceinline__ uint32_t mx_exponent(uint32_t e, float v) {
  const uint32_t f = (__float_as_uint(v) >> 23) & 255u;
  return f > e ? f : e;
}
__device__ __forceinline__ uint32_t mx_scale_byte(uint32_t e) { return e == 255u ? 255u : (e < 7u ? 0u : e - 7u); }
__device__ __forceinline__ float mx_factor(uint32_t e) {
  const uint32_t c = e < 7u ? 7u : e;
  return __uint_as_float((261u - c) << 23);
}

// Four scaled values as one register of E4M3 numbers; v becomes 16 times what
// they leave over.
__device__ __forceinline__ uint32_t mx_piece4(float (&v)[4]) {
  int p = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
  p = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], p, true);
  const mx_f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(p, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(p, true);
  v[0] = (v[0] - a[0]) * 16.f;
  v[1] = (v[1] - a[1]) * 16.f;
  v[2] = (v[2] - b[0]) * 16.f;
  v[3] = (v[3] - b[1]) * 16.f;
  return static_cast<uint32_t>(p);
}

// A word's 16 values (times the block's factor f) as NP pieces of 16 bytes.
template <int NP>
__device__ __forceinline__ void mx_word(const float (&v)[16], float f, uint4 (&out)[NP]) {
  float r[4][4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = 4 * d + i;  // byte b: even values first, then odd
      r[d][i] = v[b < 8 ? 2 * b : 2 * (b - 8) + 1] * f;
    }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    uint32_t q[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) q[d] = mx_piece4(r[d]);
    out[p] = make_uint4(q[0], q[1], q[2], q[3]);
  }
}

// The mx rows (two pieces) of bf16 tokens [tokens, 16 nwords] in the order of
// weights read 64 bytes of a row at a time (nwords % 16 == 0): of each 16 words,
// words 4 b and 4 b + 1 are block b of the even step, 4 b + 2 and 4 b + 3 of the
// odd one.  Token t's scale word of step k is xs[t * nwords / 8 + k]; xc[t] =
// (sum x, 1).
void launch_mx_prep_wide(const uint16_t* x, int64_t ldx, int64_t tokens, int64_t nwords, uint32_t* xq, uint32_t* xs,
                         float2* xc, hipStream_t s);

}  // namespace ma
