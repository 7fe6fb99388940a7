// MLX affine quantise / dequantise on gfx950.
//
// Replaces mlx_quantize / mlx_dequantize as called from
// crates/mlxr/src/ops/quantization.rs:47-70 and :118-146.  Layout
// (crates/mlxr-lm/src/attention/kernel_source.rs:30-35,96-107):
//   wq [rows, cols*bits/32] uint32, element k of a word at bits
//   [k*bits, (k+1)*bits); scales/biases [rows, cols/group] in w's dtype.
// Loading-time kernels, HBM-bound: consecutive lanes take consecutive 16-byte
// pieces of the rows (groups divide a row, so the flat element index gives the
// word, the group and the scale alike: no row arithmetic).
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace mlxr_moe {
namespace {

template <bool BF16>
__device__ __forceinline__ float ld(const void* p, int64_t i) {
  if constexpr (BF16)
    return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
  else
    return static_cast<const float*>(p)[i];
}
template <bool BF16>
__device__ __forceinline__ void st(void* p, int64_t i, float v) {
  if constexpr (BF16)
    static_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
  else
    static_cast<float*>(p)[i] = v;
}

// Elements per thread: a whole number of packed words, 16 bytes of bf16 where
// that gives one.
template <int BITS>
constexpr int kEpt = BITS == 2 ? 16 : 8;

// max / min over the LPG lanes of a group (2, 4, 8 or 16 neighbours of one
// DPP row); every lane gets the result.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ void group_max_min(int lpg, float& mx, float& mn) {
  mx = fmaxf(mx, dpp_f<0xB1>(mx)), mn = fminf(mn, dpp_f<0xB1>(mn));  // lane ^ 1
  if (lpg >= 4) mx = fmaxf(mx, dpp_f<0x4E>(mx)), mn = fminf(mn, dpp_f<0x4E>(mn));
  if (lpg >= 8) mx = fmaxf(mx, dpp_f<0x141>(mx)), mn = fminf(mn, dpp_f<0x141>(mn));
  if (lpg >= 16) mx = fmaxf(mx, dpp_f<0x140>(mx)), mn = fminf(mn, dpp_f<0x140>(mn));
}

// fp32 recipe of MLX's affine quantiser: scale = max((max-min)/n_bins, 1e-7)
// signed towards the edge of larger magnitude, snapped so that the edge is an
// exact code; codes use the unrounded scale and bias; scale and bias are
// stored in w's dtype.
// gs / kEpt neighbouring lanes hold a group (16-byte loads, whole cache lines
// per wave) and find its range by DPP moves; each lane then codes its own
// elements.  Against one thread per group (2-byte loads 128 bytes apart on
// neighbouring lanes): [128, 768, 2048] bf16 to 4 bits 7149 to 143 us (3.6 TB/s; a large copy
// reaches 4.7).
// VEC: w is 16-byte and wq 8-byte aligned; else loads and stores by element
// and word.
template <bool BF16, int BITS, bool VEC>
__global__ __launch_bounds__(256) void quantize_kernel(
    const void* __restrict__ w, int64_t n, int gs_log2, uint32_t* __restrict__ wq,
    void* __restrict__ scales, void* __restrict__ biases) {
  constexpr int EPT = kEpt<BITS>, WORDS = EPT * BITS / 32, PER = 32 / BITS;
  const int64_t e0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * EPT;
  if (e0 >= n) return;  // whole groups: gs divides n, and a group its wave
  float v[EPT];
  if constexpr (VEC && BF16) {
#pragma unroll
    for (int i = 0; i < EPT / 8; ++i) {
      const u32x4_t u =
          *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(w) + e0 + 8 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[8 * i + 2 * j] = __uint_as_float(u[j] << 16);
        v[8 * i + 2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
      }
    }
  } else if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < EPT / 4; ++i) {
      const f32x4_t u =
          *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(w) + e0 + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * i + j] = u[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < EPT; ++i) v[i] = ld<BF16>(w, e0 + i);
  }
  constexpr float n_bins = (float)((1 << BITS) - 1);
  float wmax = -INFINITY, wmin = INFINITY;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    wmax = fmaxf(wmax, v[j]);
    wmin = fminf(wmin, v[j]);
  }
  group_max_min((1 << gs_log2) / EPT, wmax, wmin);
  const bool neg_edge = fabsf(wmin) > fabsf(wmax);
  float scale = fmaxf((wmax - wmin) / n_bins, 1e-7f);
  scale = neg_edge ? scale : -scale;
  const float edge = neg_edge ? wmin : wmax;
  const float q0 = rintf(edge / scale);
  float bias = 0.0f;
  if (q0 != 0.0f) {
    scale = edge / q0;
    bias = edge;
  }
  uint32_t word[WORDS];
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    word[i] = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      float q = rintf((v[i * PER + k] - bias) / scale);
      q = fminf(fmaxf(q, 0.0f), n_bins);
      word[i] |= (uint32_t)q << (k * BITS);
    }
  }
  uint32_t* out = wq + e0 / PER;
  if constexpr (VEC && WORDS == 2) {
    *reinterpret_cast<u32x2_t*>(out) = u32x2_t{word[0], word[1]};
  } else {
#pragma unroll
    for (int i = 0; i < WORDS; ++i) out[i] = word[i];
  }
  if ((e0 & ((1 << gs_log2) - 1)) == 0) {
    st<BF16>(scales, e0 >> gs_log2, scale);
    st<BF16>(biases, e0 >> gs_log2, bias);
  }
}

// code * scale + bias as one fma, rounded once; 8 values per thread (16 bytes
// of bf16, 32 of f32).  One thread per packed word with 2-byte stores and
// 64-bit divisions before: [128, 768, 2048] 4 bits to bf16 167.8 to 113.3 us
// (4.6 TB/s).
// VEC: out is 16-byte and wq 8-byte aligned.
template <bool SB_BF16, bool OUT_BF16, int BITS, bool VEC>
__global__ __launch_bounds__(256) void dequantize_kernel(
    const uint32_t* __restrict__ wq, const void* __restrict__ scales,
    const void* __restrict__ biases, int64_t n, int gs_log2, void* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t e0 = i * 8;
  if (e0 >= n) return;
  uint32_t w[2] = {0u, 0u};
  if constexpr (BITS == 2) {
    w[0] = wq[i >> 1] >> (16 * (int)(i & 1));
  } else if constexpr (BITS == 4) {
    w[0] = wq[i];
  } else if constexpr (VEC) {
    const u32x2_t u = *reinterpret_cast<const u32x2_t*>(wq + 2 * i);
    w[0] = u.x, w[1] = u.y;
  } else {
    w[0] = wq[2 * i], w[1] = wq[2 * i + 1];
  }
  const float s = ld<SB_BF16>(scales, e0 >> gs_log2);
  const float b = ld<SB_BF16>(biases, e0 >> gs_log2);
  constexpr uint32_t mask = (1u << BITS) - 1u;
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t c = (w[k * BITS / 32] >> (k * BITS % 32)) & mask;
    v[k] = __builtin_fmaf((float)c, s, b);
  }
  if constexpr (VEC && OUT_BF16) {
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = (uint32_t)f32_to_bf16(v[2 * j]) | ((uint32_t)f32_to_bf16(v[2 * j + 1]) << 16);
    *reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(out) + e0) = o;
  } else if constexpr (VEC) {
    f32x4_t* o = reinterpret_cast<f32x4_t*>(static_cast<float*>(out) + e0);
    o[0] = f32x4_t{v[0], v[1], v[2], v[3]};
    o[1] = f32x4_t{v[4], v[5], v[6], v[7]};
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) st<OUT_BF16>(out, e0 + k, v[k]);
  }
}

// elements per launch (a grid holds under 2^32 threads)
constexpr int64_t kLaunchElems = (int64_t)1 << 34;

bool vec_aligned(const void* rows16, const uint32_t* wq) {
  return (reinterpret_cast<uintptr_t>(rows16) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(wq) & 7) == 0;
}

}  // namespace

// bits 2, 4 or 8; group_size 32, 64 or 128, dividing cols
hipError_t launch_quantize(const void* w, bool w_bf16, int64_t rows,
                           int64_t cols, int group_size, int bits, uint32_t* wq,
                           void* scales, void* biases, hipStream_t s) {
  const int64_t n = std::min(rows * cols, kLaunchElems);
  if (n == 0) return hipSuccess;
  const int64_t threads = n / (bits == 2 ? kEpt<2> : kEpt<4>);
  const dim3 grid((unsigned)((threads + 255) / 256));
  const int gl = __builtin_ctz((unsigned)group_size);
  const bool vec = vec_aligned(w, wq);
#define MLXR_Q2(BF, B)                                                              \
  do {                                                                              \
    if (vec)                                                                        \
      quantize_kernel<BF, B, true><<<grid, 256, 0, s>>>(w, n, gl, wq, scales, biases);  \
    else                                                                            \
      quantize_kernel<BF, B, false><<<grid, 256, 0, s>>>(w, n, gl, wq, scales, biases); \
  } while (0)
#define MLXR_Q(B)          \
  do {                     \
    if (w_bf16)            \
      MLXR_Q2(true, B);    \
    else                   \
      MLXR_Q2(false, B);   \
  } while (0)
  if (bits == 2)
    MLXR_Q(2);
  else if (bits == 4)
    MLXR_Q(4);
  else
    MLXR_Q(8);
#undef MLXR_Q
#undef MLXR_Q2
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || rows * cols == n) return e;
  const int64_t es = w_bf16 ? 2 : 4;  // the rest (n is whole groups): as one row
  return launch_quantize(static_cast<const char*>(w) + n * es, w_bf16, 1, rows * cols - n,
                         group_size, bits, wq + n / 32 * bits,
                         static_cast<char*>(scales) + n / group_size * es,
                         static_cast<char*>(biases) + n / group_size * es, s);
}

hipError_t launch_dequantize(const uint32_t* wq, const void* scales,
                             const void* biases, bool sb_bf16, int64_t rows,
                             int64_t cols, int group_size, int bits, void* out,
                             bool out_bf16, hipStream_t s) {
  const int64_t n = std::min(rows * cols, kLaunchElems);
  if (n == 0) return hipSuccess;
  const dim3 grid((unsigned)((n / 8 + 255) / 256));
  const int gl = __builtin_ctz((unsigned)group_size);
  const bool vec = vec_aligned(out, wq);
#define MLXR_DQ3(SB, OB, B)                                                             \
  do {                                                                                  \
    if (vec)                                                                            \
      dequantize_kernel<SB, OB, B, true><<<grid, 256, 0, s>>>(wq, scales, biases, n, gl, out);  \
    else                                                                                \
      dequantize_kernel<SB, OB, B, false><<<grid, 256, 0, s>>>(wq, scales, biases, n, gl, out); \
  } while (0)
#define MLXR_DQ2(SB, OB)      \
  do {                        \
    if (bits == 2)            \
      MLXR_DQ3(SB, OB, 2);    \
    else if (bits == 4)       \
      MLXR_DQ3(SB, OB, 4);    \
    else                      \
      MLXR_DQ3(SB, OB, 8);    \
  } while (0)
  if (sb_bf16 && out_bf16)
    MLXR_DQ2(true, true);
  else if (sb_bf16)
    MLXR_DQ2(true, false);
  else if (out_bf16)
    MLXR_DQ2(false, true);
  else
    MLXR_DQ2(false, false);
#undef MLXR_DQ2
#undef MLXR_DQ3
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || rows * cols == n) return e;
  const int64_t es = sb_bf16 ? 2 : 4;
  return launch_dequantize(wq + n / 32 * bits, static_cast<const char*>(scales) + n / group_size * es,
                           static_cast<const char*>(biases) + n / group_size * es, sb_bf16, 1,
                           rows * cols - n, group_size, bits,
                           static_cast<char*>(out) + n * (out_bf16 ? 2 : 4), out_bf16, s);
}

}  // namespace mlxr_moe
