// What the tiled GEMMs that dequantise in registers share (prefill_reg.hip:
// 64-row tiles, prefill_tall.hip: 128-row tiles).
#pragma once

#include "common.hpp"
#include "kernels.hpp"
#include "prefill_dev.hpp"

namespace mlxr_moe {

constexpr uint32_t kPastEnd = 0xFFFFFFF0u;  // out of range of every buffer

// Where the scales and biases of a weight step come from: rows of any length at
// any alignment, one aligned vector per row, or chunks of several steps in LDS.
enum { kSbAny, kSbVector, kSbLds };

// Workgroups of a problem of at most `tiles` M-tiles.
__host__ __device__ constexpr int reg_grid(int64_t tiles, int units_n) {
  return (int)((tiles + kXcds - 1) / kXcds * kXcds) * units_n;
}

// What the kernels are launched with: the routed problem and the folded one
// (which takes the first workgroups: tiles2 M-tiles of rows2 rows in token
// order, no dispatch); units_n units of ntl N-tiles, of tiles_n in all, per
// M-tile.
struct RegLaunch {
  QGemmArgs a;
  int32_t tiles_n, ntl, units_n;
  uint32_t x_bytes;
  QGemmArgs a2;
  int32_t tiles2, rows2;
  uint32_t x_bytes2;
};

// A workgroup's unit: rows [slot0, slot0 + rows) of expert e against N-tiles
// [nt0, nt1).  place() gives its M-tile and N-tiles, or false without one;
// find_rows() the rest, from the tile's record.  (Two steps, so that the record's
// loads and those of the kernel's arguments overlap: 1% of c4 T=2048 gate/up.)
// Workgroups go to the XCDs round robin (block % kXcds).  Each XCD takes an
// eighth of the M-tile list, in order, a tile's units one after another: they
// share the tile's x rows, and an expert's further tiles its weights, in that
// XCD's L2.  (Tiles dealt to the XCDs in turn: c5 T=512 step 679 us against
// 657, c3 T=512 177 against 168, c4 T=2048 428 against 427; a few tiles'
// units interleaved: 1-5% slower.)
template <int ROWS>
struct RegUnit {
  bool second;
  int tile, nt0, nt1;
  int e, slot0, rows;
  __device__ __forceinline__ bool place(const RegLaunch& L, int block) {
    const int grid2 = reg_grid(L.tiles2, L.units_n);
    second = block < grid2;
    const int b = second ? block : block - grid2;
    const int xcd = b % (int)kXcds, jx = b / (int)kXcds;
    const int n_tiles = second ? L.tiles2 : *L.a.num_tiles;
    tile = xcd * n_tiles / (int)kXcds + jx / L.units_n;
    if (tile >= (xcd + 1) * n_tiles / (int)kXcds) return false;
    nt0 = (jx - jx / L.units_n * L.units_n) * L.ntl;
    nt1 = min(nt0 + L.ntl, L.tiles_n);
    return true;
  }
  __device__ __forceinline__ void find_rows(const RegLaunch& L) {
    e = 0;
    slot0 = tile * ROWS;
    int end = L.rows2;
    if (!second) {
      const int2 trec = *reinterpret_cast<const int2*>(L.a.tiles + 2 * tile);
      e = __builtin_amdgcn_readfirstlane(trec.x);
      slot0 = __builtin_amdgcn_readfirstlane(trec.y);
      end = __builtin_amdgcn_readfirstlane(L.a.offsets[e + 1]);
    }
    rows = min(ROWS, end - slot0);
  }
};

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

// The scales (or biases) of a step of SG groups from g0 on, of row ch of an
// expert's N rows of G, two to a word; zeros past the row, so that a step's
// groups past it add nothing, whatever the row holds.  One load that needs no
// more than the elements' alignment, ending within the expert's rows (the rest
// is shifted out), and no branch around it: that would make the compiler wait
// for every load in flight.
template <int SG>
__device__ __forceinline__ void load_sb_any(gptr<const uint16_t> expert, int N, int G, int ch,
                                            int g0, uint32_t (&sb)[2]) {
  typedef uint64_t u64_a2 __attribute__((aligned(2)));
  typedef uint32_t u32_a2 __attribute__((aligned(2)));
  const uint32_t off = (uint32_t)(ch * G + g0), at = min(off, (uint32_t)(N * G - SG));
  const uint32_t sh = 16 * (off - at);
  const int left = G - g0;
  if constexpr (SG == 4) {
    const uint64_t mask = left < 4 ? (1ull << (16 * left)) - 1 : ~0ull;
    const uint64_t v = (*(gptr<const u64_a2>)(expert + at) >> sh) & mask;
    sb[0] = (uint32_t)v, sb[1] = (uint32_t)(v >> 32);
  } else {
    sb[0] = (*(gptr<const u32_a2>)(expert + at) >> sh) & (left < 2 ? 0xffffu : ~0u);
    sb[1] = 0u;
  }
}

// Wave-private LDS hand-over.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// For a wave whose sums are not all finite: whether its columns of its unit
// have a 4-bit scale of 2^104 or more.  dequant4's scaled forms overflow there,
// so that every weight of the group is an infinity or a NaN and no sum of its
// channel finite; then the columns are done once more, every sum in the same
// order, weights by fmaf(code, scale, bias) and operands straight from memory.
// (No weight of a trained model has such a scale: the units' loops pay nothing
// for it, and everything it needs is read again, from the kernel's arguments
// on, so that nothing is held for it.)
template <bool GATED, int ROWS>
__device__ __forceinline__ void exact4_unit(int waves) {
  uintptr_t args = reinterpret_cast<uintptr_t>(
      (const void*)__builtin_amdgcn_kernarg_segment_ptr());
  int block = blockIdx.x;
  asm volatile("" : "+s"(args), "+s"(block));
  const RegLaunch& L = *reinterpret_cast<const RegLaunch*>(args);
  RegUnit<ROWS> u;
  u.place(L, block);
  u.find_rows(L);
  const RegArgs a = pick_reg(u.second, L.a2, L.x_bytes2, L.a, L.x_bytes);
  const int N = L.a.N, K = L.a.K, e = u.e, slot0 = u.slot0, rows = u.rows;
  const int nt0 = u.nt0, nt1 = u.nt1;
  const int TC = GATED ? 32 * waves : 64 * waves, WC = TC / waves;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, h = lane >> 5, G = K >> 6;
  bool large = false;
  for (int nt = nt0; nt < nt1; ++nt)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int ch = nt * TC + wave * WC + (GATED ? 0 : 32 * s) + c;
      const gptr<const uint16_t> sp = as_global<const uint16_t>(GATED && s ? a.w1.scales
                                                                            : a.w0.scales) +
                                      ((int64_t)e * a.e_rows + min(ch, N - 1)) * G;
      for (int g = h; g < G; g += 2)
        large |= fabsf(__uint_as_float((uint32_t)sp[g] << 16)) >= 0x1p104f;
    }
  if (!__any(large)) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first results are out
#pragma nounroll
  for (int nt = nt0; nt < nt1; ++nt)
#pragma nounroll
    for (int r0 = 0; r0 < rows; r0 += 32) {
      int xrow = slot0 + min(r0 + c, rows - 1);
      if (!a.x_by_slot) {
        xrow = as_global<const int32_t>(a.sorted)[xrow];
        xrow = a.row_map ? as_global<const int32_t>(a.row_map)[xrow] : xrow / a.row_div;
      }
      const gptr<const uint16_t> xp = as_global<const uint16_t>(a.x) + (int64_t)xrow * a.x_ld;
      const int och0 = nt * TC + wave * WC;
      f32x16_t acc[2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[s][r] = 0.0f;
#pragma nounroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) {
          const bf16x8_t af =
              as_bf16x8(*(gptr<const u32x4_t>)(xp + 64 * g + 16 * kc + 8 * h));
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const QWeights& W = GATED && s ? a.w1 : a.w0;
            const int64_t row =
                (int64_t)e * a.e_rows + min(och0 + (GATED ? 0 : 32 * s) + c, N - 1);
            const float sc = __uint_as_float(
                (uint32_t)as_global<const uint16_t>(W.scales)[row * G + g] << 16);
            const float bi = __uint_as_float(
                (uint32_t)as_global<const uint16_t>(W.biases)[row * G + g] << 16);
            uint32_t o[4];
            dequant4_any(as_global<const uint32_t>(W.w)[(row * G + g) * 8 + 2 * kc + h], sc, bi,
                         o);
            acc[s] = mfma32x32x16(af, as_bf16x8(u32x4_t{o[0], o[1], o[2], o[3]}), acc[s]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int trow = r0 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (trow >= rows) continue;
        int64_t orow = slot0 + trow;
        if (!GATED && a.out_by_flat) orow = as_global<const int32_t>(a.sorted)[orow];
        const gptr<uint16_t> op = as_global<uint16_t>(a.out) + orow * a.out_ld + och0 + c;
        if constexpr (GATED) {
          const uint16_t v =
              a.act == kActGeglu
                  ? geglu_bf16(bf16_round(acc[0][r]), bf16_round(acc[1][r]))
                  : (uint16_t)swiglu_fast2(acc[0][r], acc[1][r], acc[0][r], acc[1][r]);
          if (och0 + c < N) op[0] = v;
        } else {
#pragma unroll
          for (int s = 0; s < 2; ++s)
            if (och0 + 32 * s + c < N)
              op[32 * s] = __builtin_bit_cast(uint16_t, (__bf16)acc[s][r]);
        }
      }
    }
}

}  // namespace mlxr_moe
