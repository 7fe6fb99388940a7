// Device helpers shared by the tiled (prefill) GEMM kernels: dequantisation
// of packed codes to bf16 pairs, the SwiGLU epilogue, small integer helpers.
#pragma once

#include "common.hpp"

namespace mlxr_moe {

// raw buffer resource word 3 (gfx9 family)
constexpr int kBufFlags = 0x00020000;
// XCDs of an MI355X (the workgroup numbering below assumes this many; any
// other count only changes which workgroups share an L2)
constexpr unsigned kXcds = 8;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_convertvector((f32x2_t){lo, hi}, bf16x2_t));
}
// a and b rounded to bf16 by one conversion (round to nearest even), as f32
__device__ __forceinline__ f32x2_t bf16_hw2(float a, float b) {
  const uint32_t p =
      __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
  return f32x2_t{__uint_as_float(p << 16), __uint_as_float(p & 0xffff0000u)};
}
// silu(g) * u of two elements with the reference's bf16 rounding points
// (crates/mlxr-lm/src/activations.rs:187-200), each rounding done for both at
// once; the sigmoid from the hardware exp2 and reciprocal (about 1 ulp each in
// f32; the bf16 rounding that follows hides that except next to a rounding
// boundary).  The results packed, the first in the low half.
__device__ __forceinline__ uint32_t swiglu_fast2(float g0_acc, float u0_acc, float g1_acc,
                                                 float u1_acc) {
  const f32x2_t g = bf16_hw2(g0_acc, g1_acc), u = bf16_hw2(u0_acc, u1_acc);
  const float e0 = __builtin_amdgcn_exp2f(-g.x * 1.4426950408889634f);
  const float e1 = __builtin_amdgcn_exp2f(-g.y * 1.4426950408889634f);
  const f32x2_t sg = bf16_hw2(__builtin_amdgcn_rcpf(1.0f + e0), __builtin_amdgcn_rcpf(1.0f + e1));
  const f32x2_t h = bf16_hw2(g.x * sg.x, g.y * sg.y);
  return __builtin_bit_cast(uint32_t,
                            __builtin_convertvector(f32x2_t{h.x * u.x, h.y * u.y}, bf16x2_t));
}
// a compile-time flag as a type (for generic lambdas)
template <bool B>
struct PfFlag {
  static constexpr bool value = B;
};
// n / d for 0 <= n < 2^31, 1 <= d <= 2^16, rd = 1.0f / d: a float estimate
// (off by up to 3 * 2^-24 of the quotient and one, as many as 385), another of
// what it leaves (off by one at most), and a correction either way.
__host__ __device__ __forceinline__ int div_small(int n, int d, float rd) {
  uint32_t q = (uint32_t)((float)n * rd);
  int r = (int)((uint32_t)n - q * (uint32_t)d);
  q += (uint32_t)(int)((float)r * rd);
  r = (int)((uint32_t)n - q * (uint32_t)d);
  return (int)q - (r < 0 ? 1 : 0) + (r >= d ? 1 : 0);
}

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
// x & m, opaque to the optimiser (it would otherwise turn the masks and the
// conversions below into bit-field extracts)
__device__ __forceinline__ uint32_t and_opaque(uint32_t x, uint32_t m) {
  uint32_t r;
  asm("v_and_b32 %0, %1, %2" : "=v"(r) : "v"(x), "s"(m));
  return r;
}
// 8 four-bit codes of one word (little end first) -> 4 words of bf16 pairs,
// each bf16(fmaf(code, s, b)).  A nibble alone in the low bits of an f16 half
// is the f16 subnormal code * 2^-24 (code * 2^-20 four bits up), and
// v_fma_mix_f32 multiplies it as it is by s * 2^24 (s * 2^20): the product is
// code * s exactly, so the sum is rounded once, as fmaf(code, s, b) is (for
// |s| < 2^104, where s * 2^24 is finite: a unit with a larger scale is done
// again by exact4_unit).  17 instructions a word against 23
// with a v_cvt_f32_ubyte per code: step of c3 T=4096 509 to 502 us, c4 T=2048
// 489 to 481, bit-identical.
__device__ __forceinline__ void dequant4(uint32_t w, float s24, float s20, float b,
                                         uint32_t* o) {
  const uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, w8 = w >> 8;
  // codes (0, 4), (1, 5), (2, 6), (3, 7)
  const f16x2_t c04 = __builtin_bit_cast(f16x2_t, and_opaque(w, m0));
  const f16x2_t c15 = __builtin_bit_cast(f16x2_t, and_opaque(w, m1));
  const f16x2_t c26 = __builtin_bit_cast(f16x2_t, and_opaque(w8, m0));
  const f16x2_t c37 = __builtin_bit_cast(f16x2_t, and_opaque(w8, m1));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    o[2 * j] = pack_bf16(__builtin_fmaf((float)c04[j], s24, b),
                         __builtin_fmaf((float)c15[j], s20, b));
    o[2 * j + 1] = pack_bf16(__builtin_fmaf((float)c26[j], s24, b),
                             __builtin_fmaf((float)c37[j], s20, b));
  }
}
// The same words by fmaf(code, s, b) as it stands, for scales of any size.
__device__ __forceinline__ void dequant4_any(uint32_t w, float s, float b, uint32_t* o) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = pack_bf16(__builtin_fmaf((float)((w >> (8 * j)) & 15u), s, b),
                     __builtin_fmaf((float)((w >> (8 * j + 4)) & 15u), s, b));
}
// 4 eight-bit codes -> 2 words of pairs
__device__ __forceinline__ void dequant8(uint32_t w, float s, float b,
                                         uint32_t* o) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
    o[j] = pack_bf16(__builtin_fmaf((float)((w >> (16 * j)) & 255u), s, b),
                     __builtin_fmaf((float)((w >> (16 * j + 8)) & 255u), s, b));
}

__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

}  // namespace mlxr_moe
