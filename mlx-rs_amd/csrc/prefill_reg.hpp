// What the tiled GEMMs that dequantise in registers share (prefill_reg.hip:
// 64-row tiles, prefill_tall.hip: 128-row tiles).
#pragma once

#include "common.hpp"
#include "kernels.hpp"
#include "prefill_dev.hpp"

namespace mlxr_moe {

constexpr uint32_t kPastEnd = 0xFFFFFFF0u;  // out of range of every buffer

// Where the scales and biases of a weight step come from: single loads, one
// aligned vector per row, or chunks of several steps in LDS.
enum { kSbSingle, kSbVector, kSbLds };

// Workgroups of a problem of at most `tiles` M-tiles.
__host__ __device__ constexpr int reg_grid(int64_t tiles, int units_n) {
  return (int)((tiles + kXcds - 1) / kXcds * kXcds) * units_n;
}

// groups per weight step: one 128-byte line of every row
template <int BITS>
constexpr int kStepGroups = BITS == 4 ? 4 : BITS == 8 ? 2 : 1;

// The operands of one unit, chosen between the routed problem and the folded
// one field by field (scalar selects).
struct RegArgs {
  const uint16_t* x;
  int64_t x_ld;
  const int32_t *row_map, *sorted;
  int32_t row_div;
  bool x_by_slot, out_by_flat;
  QWeights w0, w1;
  int32_t e_rows, act;
  uint16_t* out;
  int64_t out_ld;
  uint32_t x_bytes;
};
__device__ __forceinline__ RegArgs pick_reg(bool q, const QGemmArgs& b, uint32_t b_bytes,
                                            const QGemmArgs& c, uint32_t c_bytes) {
  RegArgs r;
  r.x = q ? b.x : c.x;
  r.x_ld = q ? b.x_ld : c.x_ld;
  r.row_map = q ? b.row_map : c.row_map;
  r.sorted = q ? b.sorted : c.sorted;
  r.row_div = q ? b.row_div : c.row_div;
  r.x_by_slot = q ? b.x_by_slot : c.x_by_slot;
  r.out_by_flat = q ? b.out_by_flat : c.out_by_flat;
  r.w0 = QWeights{q ? b.w0.w : c.w0.w, q ? b.w0.scales : c.w0.scales,
                  q ? b.w0.biases : c.w0.biases};
  r.w1 = QWeights{q ? b.w1.w : c.w1.w, q ? b.w1.scales : c.w1.scales,
                  q ? b.w1.biases : c.w1.biases};
  r.e_rows = q ? b.e_rows : c.e_rows;
  r.act = q ? b.act : c.act;
  r.out = q ? b.out : c.out;
  r.out_ld = q ? b.out_ld : c.out_ld;
  r.x_bytes = q ? b_bytes : c_bytes;
  return r;
}

// One line of every row of a wave's two sides (gate and up channels, or the
// two 32-channel blocks of the down projection): four 16-byte loads per lane
// and side.  sb: the step's scales (lanes 0-31) and biases (lanes 32-63).
struct WStep {
  u32x4_t w[2][4];
  uint32_t sb[2][2];
};

__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// A pointer to device memory as one.  Chosen between two kernel arguments it
// would otherwise count as a pointer to anything, whose (flat) loads wait for
// every other load in flight.
template <class T>
using gptr = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gptr<T> as_global(const void* p) {
  return (gptr<T>)reinterpret_cast<uintptr_t>(p);
}

// Wave-private LDS hand-over.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace mlxr_moe
