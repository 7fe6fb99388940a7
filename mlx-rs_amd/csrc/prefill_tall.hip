// Grouped quantised expert GEMM for many rows per expert: 128-row M-tiles,
// the weights dequantised in registers.
//
// Same operation and the same sums, in the same order, as the 64-row tiles
// (prefill_reg.hip).  A wave owns 32 gate and the same 32 up channels, or 64
// down channels, for up to 128 rows (its sums are half its registers), so a
// weight is dequantised half as often as with 64 rows, and the MFMAs bound the
// launch: per group 32 of them (1024 cycles of a SIMD) against about 600 of
// dequantisation, two waves a SIMD.  Keeping the dequantised weights out of LDS
// is what makes the room: through it, a 256 x 256 tile moves 256 KB per group
// and CU, as many cycles as its MFMAs take; here the x operand alone does, half
// as many.
//
// One line of every row is in flight in registers; once there it waits in the
// wave's own 8 KB of LDS and is read a group at a time.  x is staged one group
// ahead, a barrier per group, two workgroups per CU.
//
// c3 T=4096 (256 rows an expert on average, skewed) against 256 x 256 tiles
// through LDS, both from one run: step 509 to 446 us; first passes on new
// inputs, traced, gate/up 288 to 242, down 176 to 134.  A copy that only reads x
// and multiplies takes 174 us for gate/up.  The matrix cores
// are busy 39% of it, 35% of down.  No faster, against a step of 466 us then:
// the MFMAs of a chunk kept together, raised wave priority around them (519),
// one MFMA to every 4 or 5 VALU instructions by scheduling groups (489, 505),
// the order pinned instruction group by instruction group (475).
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "prefill_dev.hpp"
#include "prefill_reg.hpp"

namespace mlxr_moe {
namespace {

constexpr int kRows = 128;                  // rows per M-tile
constexpr int kWaves = 4, kNT = 64 * kWaves;
constexpr int kXBytes = kRows * 128;        // x stage: one group
constexpr int kLine = 4096;                 // per wave and side: a line of 32 rows
constexpr int kScratch = 2 * kLine;         // ... both sides; the epilogue's tile
constexpr int kSbChunk = 8;                 // groups of scales per LDS buffer
constexpr int kSbBytes = 2 * 32 * 2 * kSbChunk * 2;  // per wave: [side][32][s, b][8]
constexpr int tall_lds(int sbm) {
  return 2 * kXBytes + kWaves * (kScratch + (sbm == kSbLds ? 2 * kSbBytes : 0));
}
// two workgroups share a CU's 160 KB
static_assert(2 * tall_lds(kSbLds) <= 160 * 1024, "two workgroups per CU");

// The rows [slot0, slot0 + rows) of expert e against N-tiles [nt0, nt1).
// NMB: 32-row blocks that hold rows.  Returns (for the whole wave) whether a
// 4-bit scale may have been too large (exact4_unit).
template <int BITS, bool GATED, int SBM, int NMB>
__device__ __forceinline__ bool tall_unit(const RegArgs& a, int N, int K, int e, int slot0,
                                         int rows, int nt0, int nt1, char* smem) {
  constexpr int SG = kStepGroups<BITS>;  // groups per weight step
  constexpr int TC = GATED ? 32 * kWaves : 64 * kWaves;  // channels per N-tile
  constexpr int WC = TC / kWaves;                        // ... per wave
  constexpr int CS = kSbChunk / SG;                      // weight steps per scale chunk
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int G = K >> 6;                  // groups
  const int T = (G + SG - 1) / SG;       // weight steps per tile
  const int total = T * (nt1 - nt0);     // ... of this unit
  char* xl = smem;
  char* scratch = smem + 2 * kXBytes + wave * (kScratch + (SBM == kSbLds ? 2 * kSbBytes : 0));
  char* sbl = scratch + kScratch;

  // ---- weights: a buffer per side over the expert's rows
  const int64_t row_bytes = (int64_t)K * BITS / 8;
  const __amdgpu_buffer_rsrc_t wr0 = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(a.w0.w) + (int64_t)e * a.e_rows * (row_bytes / 4), 0,
      (int)(N * row_bytes), kBufFlags);
  const __amdgpu_buffer_rsrc_t wr1 = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(GATED ? a.w1.w : a.w0.w) +
          (int64_t)e * a.e_rows * (row_bytes / 4),
      0, (int)(N * row_bytes), kBufFlags);
  // first channel of a side of tile nt
  auto channel0 = [&](int nt, int side) {
    return nt * TC + wave * WC + (GATED ? 0 : 32 * side);
  };
  const int lrow = lane >> 3, lch = lane & 7;  // load i: row 8 i + lrow, 16-byte chunk lch
  const uint32_t lane_off = (uint32_t)(lrow * row_bytes + 16 * lch);
  const uint32_t row8 = (uint32_t)(8 * row_bytes);
  int pt = nt0, pw = 0;  // the next weight step to load: tile, step within it
  // The next step's loads.  Every step issues the same ones; those of bytes
  // past the row, channels past N and steps past the unit's are out of range
  // (zeros, no memory round trip).
  auto load_w = [&](WStep& W) {
    const bool on = pt < nt1;
    // bytes of the row from this step's line on
    const int left = (int)row_bytes - 128 * pw;
    const bool ok = on && 16 * lch < left;
    const uint32_t so = on && left > 0 ? 128 * pw : 0;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // (rows past N: out of range by the vector offset)
      const uint32_t v0 = lane_off + (uint32_t)(channel0(pt, s) * row_bytes);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        W.w[s][i] = __builtin_amdgcn_raw_buffer_load_b128(s ? wr1 : wr0,
                                                          ok ? v0 + i * row8 : kPastEnd, so, 0);
    }
    if constexpr (SBM != kSbLds) {
      const int g0 = on ? min(SG * pw, (G - 1) / SG * SG) : 0;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint16_t* sp = GATED && s ? a.w1.scales : a.w0.scales;
        const uint16_t* bp = GATED && s ? a.w1.biases : a.w0.biases;
        const int ch = min(channel0(on ? pt : nt0, s) + c, N - 1);
        const gptr<const uint16_t> p =
            as_global<const uint16_t>(h ? bp : sp) + (int64_t)e * a.e_rows * G;
        if constexpr (SBM == kSbVector && BITS == 4) {
          const u32x2_t v = *(gptr<const u32x2_t>)(p + (int64_t)ch * G + g0);
          W.sb[s][0] = v.x, W.sb[s][1] = v.y;
        } else if constexpr (SBM == kSbVector) {
          W.sb[s][0] = *(gptr<const uint32_t>)(p + (int64_t)ch * G + g0);
          W.sb[s][1] = 0u;
        } else {
          load_sb_any<SG>(p, N, G, ch, g0, W.sb[s]);
        }
      }
    }
    if (++pw == T) {
      pw = 0;
      ++pt;
    }
  };
  // A side's scales and biases of groups 8 k .. 8 k + 7 of tile nt: lane l
  // takes those of row l / 2, scales (even lanes) or biases (odd), 16 bytes.
  // (The array is chosen by arithmetic: a choice among the four fields becomes
  // one among their addresses, for which the compiler kept all of `a` in scratch
  // memory, and each K step waited, for every other load in flight too, until
  // the pointer was back.  Gate/up of c3 T=4096 248 us so, 238 without.)
  const auto addr = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
  const uintptr_t sb_w0 = addr(a.w0.scales), b_off0 = addr(a.w0.biases) - sb_w0;
  const uintptr_t up_s = GATED ? addr(a.w1.scales) - sb_w0 : 0;
  const uintptr_t up_b = GATED ? addr(a.w1.biases) - sb_w0 - b_off0 : 0;
  auto load_sp = [&](int nt, int k, int side) {
    const uintptr_t up = GATED ? side : 0, bias = lane & 1;
    const uintptr_t q = sb_w0 + up * up_s + bias * (b_off0 + up * (up_b - up_s));
    const int ch = channel0(nt, side) + (lane >> 1);
    return *(gptr<const u32x4_t>)(as_global<const uint16_t>(reinterpret_cast<const void*>(q)) +
                                  ((int64_t)e * a.e_rows + min(ch, N - 1)) * G + kSbChunk * k);
  };
  auto store_sp = [&](int buf, int side, u32x4_t v) {
    *reinterpret_cast<u32x4_t*>(sbl + buf * kSbBytes + side * (kSbBytes / 2) + 16 * lane) = v;
  };

  WStep W;  // the weight step in flight
  load_w(W);
  u32x4_t sp0[2];
  if constexpr (SBM == kSbLds) {
#pragma unroll
    for (int i = 0; i < 2; ++i) sp0[i] = load_sp(nt0, 0, i);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- x: thread -> 16-byte chunk tid % 8 of the group of rows tid / 8 +
  // 32 j; chunk cc of row r sits at cc ^ ((r >> 1) & 7)
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.x), 0, (int)a.x_bytes, kBufFlags);
  const int xrow0 = tid >> 3, xc = tid & 7;
  uint32_t aoff[NMB];
  {
    int xrow[NMB];
#pragma unroll
    for (int j = 0; j < NMB; ++j) xrow[j] = slot0 + min(xrow0 + 32 * j, rows - 1);
    if (!a.x_by_slot) {
#pragma unroll
      for (int j = 0; j < NMB; ++j) xrow[j] = as_global<const int32_t>(a.sorted)[xrow[j]];
      if (a.row_map) {
#pragma unroll
        for (int j = 0; j < NMB; ++j) xrow[j] = as_global<const int32_t>(a.row_map)[xrow[j]];
      } else {
        const float rdiv = 1.0f / (float)a.row_div;
#pragma unroll
        for (int j = 0; j < NMB; ++j) xrow[j] = div_small(xrow[j], a.row_div, rdiv);
      }
    }
#pragma unroll
    for (int j = 0; j < NMB; ++j)
      aoff[j] = xrow0 + 32 * j < rows ? (uint32_t)((int64_t)xrow[j] * a.x_ld * 2 + 16 * xc)
                                      : kPastEnd;
  }
  const int aw = xrow0 * 128 + 16 * (xc ^ swz(xrow0));
  u32x4_t xv[NMB];
  const int XS = T * SG;  // x stages per tile
  int px = 0, left_x = XS * (nt1 - nt0);
  // The next x stage (zeros past K and past the unit; rows past the tile are
  // out of range already)
  auto load_x = [&]() {
    const bool on = left_x > 0 && px < G;
#pragma unroll
    for (int j = 0; j < NMB; ++j)
      xv[j] = __builtin_amdgcn_raw_buffer_load_b128(xr, on ? aoff[j] : kPastEnd,
                                                    on ? 128 * px : 0, 0);
    px = px + 1 < XS ? px + 1 : 0;
    --left_x;
  };
  auto store_x = [&](int st) {
#pragma unroll
    for (int j = 0; j < NMB; ++j)
      *reinterpret_cast<u32x4_t*>(xl + st * kXBytes + aw + 4096 * j) = xv[j];
  };
  // the flat output rows of tile rows lane and lane + 64 (the down projection)
  int orow[2] = {slot0 + min(lane, rows - 1), slot0 + min(lane + 64, rows - 1)};
  if (!GATED && a.out_by_flat) {
#pragma unroll
    for (int i = 0; i < 2; ++i) orow[i] = as_global<const int32_t>(a.sorted)[orow[i]];
  }
  load_x();
  store_x(0);
  if constexpr (SBM == kSbLds) {
#pragma unroll
    for (int i = 0; i < 2; ++i) store_sp(0, i, sp0[i]);
  }
  __syncthreads();

  f32x16_t acc[NMB][2];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < NMB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  };
  clear();

  // ---- an arrived line into the wave's scratch: chunk cc of row r at
  // cc ^ (r & 7) of its 128 bytes
  const int tw = lrow * 128 + 16 * (lch ^ lrow);
  auto put = [&](const WStep& W) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<u32x4_t*>(scratch + s * kLine + 1024 * i + tw) = W.w[s][i];
    wave_sync();
  };
  // A side's codes of group gi of the line: lane (c, h) reads the half h of
  // channel c's, then the halves of the wave are swapped so that every
  // register (pair, at 8 bits) is one MFMA chunk's operand: chunk kc at 4 bits
  // is w[kWord4[kc]], at 8 bits w[kWord8[kc]] and the next.
  const char* tr = scratch + c * 128;
  const int tx = c & 7;
  auto take = [&](int s, int gi, uint32_t (&w)[8]) {
    const char* p = tr + s * kLine;
    if constexpr (BITS == 4) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p + 16 * ((2 * gi + h) ^ tx));
      w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
      swap32(w[0], w[1]);
      swap32(w[2], w[3]);
    } else {
      const u32x4_t u = *reinterpret_cast<const u32x4_t*>(p + 16 * ((4 * gi + 2 * h) ^ tx));
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p + 16 * ((4 * gi + 2 * h + 1) ^ tx));
      w[0] = u.x, w[1] = u.y, w[2] = u.z, w[3] = u.w;
      w[4] = v.x, w[5] = v.y, w[6] = v.z, w[7] = v.w;
      swap32(w[0], w[2]);
      swap32(w[1], w[3]);
      swap32(w[4], w[6]);
      swap32(w[5], w[7]);
    }
  };
  constexpr int kWord4[4] = {0, 2, 1, 3}, kWord8[4] = {0, 4, 2, 6};

  // scales and biases of the step's groups, two per register, on every lane
  auto scales = [&](const WStep& W, int buf, int g8, uint32_t (&sv)[2][2],
                    uint32_t (&bv)[2][2]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if constexpr (SBM == kSbLds) {
        const char* p = sbl + buf * kSbBytes + s * (kSbBytes / 2) + 32 * c + 2 * g8;
        if constexpr (BITS == 4) {
          const u32x2_t u = *reinterpret_cast<const u32x2_t*>(p);
          const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p + 16);
          sv[s][0] = u.x, sv[s][1] = u.y, bv[s][0] = v.x, bv[s][1] = v.y;
        } else {
          sv[s][0] = *reinterpret_cast<const uint32_t*>(p);
          bv[s][0] = *reinterpret_cast<const uint32_t*>(p + 16);
        }
      } else {
#pragma unroll
        for (int j = 0; j < SG / 2; ++j) {
          sv[s][j] = bv[s][j] = W.sb[s][j];
          swap32(sv[s][j], bv[s][j]);
        }
      }
    }
  };

  // ---- one 16-wide chunk: dequantised weights of both sides
  struct Scaled {
    float sc[2], s4[2], bi[2];
  };
  auto scaled = [&](const uint32_t (&sv)[2][2], const uint32_t (&bv)[2][2], int gi) {
    Scaled r;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      r.sc[s] = __uint_as_float(gi & 1 ? sv[s][gi / 2] & 0xffff0000u : sv[s][gi / 2] << 16);
      r.bi[s] = __uint_as_float(gi & 1 ? bv[s][gi / 2] & 0xffff0000u : bv[s][gi / 2] << 16);
      if constexpr (BITS == 4) {
        r.s4[s] = r.sc[s] * 0x1p20f;
        r.sc[s] *= 0x1p24f;
        // (kept, not recomputed for every word)
        asm("" : "+v"(r.sc[s]), "+v"(r.s4[s]));
      }
    }
    return r;
  };
  auto weights = [&](const uint32_t (&w)[2][8], const Scaled& q, int kc, bf16x8_t (&bf)[2]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint32_t o[4];
      if constexpr (BITS == 4) {
        dequant4(w[s][kWord4[kc]], q.sc[s], q.s4[s], q.bi[s], o);
      } else {
        dequant8(w[s][kWord8[kc]], q.sc[s], q.bi[s], o);
        dequant8(w[s][kWord8[kc] + 1], q.sc[s], q.bi[s], o + 2);
      }
      bf[s] = as_bf16x8(u32x4_t{o[0], o[1], o[2], o[3]});
    }
  };
  const int aswz = swz(c);
  auto read_a = [&](bf16x8_t (&af)[NMB], int st, int kc) {
    const char* A = xl + st * kXBytes + c * 128;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
      af[mb] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(
          A + 4096 * mb + 16 * ((2 * kc + h) ^ aswz)));
  };

  // ---- a finished tile: through the wave's scratch, 32 rows at a time, so
  // that every store is 16 bytes of a row
  uint16_t* O = reinterpret_cast<uint16_t*>(scratch);
  uint64_t nonfinite = 0;  // (a scale too large: not one sum of its channel is finite)
  auto epilogue = [&](int nt) {
    if constexpr (BITS == 4)
      nonfinite |= __ballot(!__builtin_isfinite(acc[0][0][0]) || !__builtin_isfinite(acc[0][1][0]));
    const int och0 = nt * TC + wave * WC;
    // (the lane anew, so that what the stores make of it is made here: kept
    // over the weight steps it was ten registers too many)
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int lane = lane_e, c = lane & 31, h = lane >> 5;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
      if constexpr (GATED) {
        auto rows_of = [&](auto geglu) {
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const int row = 8 * (r >> 2) + 4 * h + (r & 3);
            uint32_t v;
            if constexpr (decltype(geglu)::value)
              v = (uint32_t)geglu_bf16(bf16_round(acc[mb][0][r]), bf16_round(acc[mb][1][r])) |
                  ((uint32_t)geglu_bf16(bf16_round(acc[mb][0][r + 1]),
                                        bf16_round(acc[mb][1][r + 1]))
                   << 16);
            else
              v = swiglu_fast2(acc[mb][0][r], acc[mb][1][r], acc[mb][0][r + 1],
                               acc[mb][1][r + 1]);
            O[row * WC + c] = (uint16_t)v;
            O[(row + 1) * WC + c] = (uint16_t)(v >> 16);
          }
        };
        if (a.act == kActGeglu)
          rows_of(PfFlag<true>{});
        else
          rows_of(PfFlag<false>{});
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = 8 * (r >> 2) + 4 * h + (r & 3);
#pragma unroll
          for (int s = 0; s < 2; ++s)
            O[row * WC + 32 * s + c] = __builtin_bit_cast(uint16_t, (__bf16)acc[mb][s][r]);
        }
      }
      wave_sync();
      constexpr int CPR = WC / 8;  // 16-byte runs per row
#pragma unroll
      for (int i = 0; i < 32 * CPR / 64; ++i) {
        const int id = lane + 64 * i, row = id / CPR, cc = id % CPR;
        const int trow = 32 * mb + row;
        const int64_t orw = GATED ? slot0 + trow : __shfl(orow[mb >> 1], trow & 63, 64);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(O + row * WC + 8 * cc);
        if (trow < rows && och0 + 8 * cc < N)
          *(gptr<u32x4_t>)(as_global<uint16_t>(a.out) + orw * a.out_ld + och0 + 8 * cc) = v;
      }
      wave_sync();
    }
  };

  // ---- the weight steps.  Issue order within one: the next x stage, the
  // scales of the next chunk, then, once the line that arrived is in the
  // scratch, the next line.
  int nt = nt0, s = 0;  // tile, weight step within it
  int xst = 0;          // the x stage that is read next
  int ws = 0, ck = 0;   // weight step within its scale chunk, chunk within the tile
  int buf = 0;          // the LDS buffer of the current scale chunk
#pragma nounroll
  for (int q = 0; q < total; ++q) {
    load_x();
    u32x4_t sp;
    if constexpr (SBM == kSbLds) {
      // one side of the next chunk; stored when the x stage is
      const bool wrap = ck + 1 == G / kSbChunk;
      sp = load_sp(wrap ? min(nt + 1, nt1 - 1) : nt, wrap ? 0 : ck + 1, ws / (CS / 2));
    }
    __builtin_amdgcn_sched_barrier(0);
    put(W);
    uint32_t sv[2][2], bv[2][2];
    scales(W, buf, SBM == kSbLds ? SG * ws : 0, sv, bv);
    load_w(W);
    __builtin_amdgcn_sched_barrier(0);
    // Chunk by chunk; the next chunk's weights are dequantised between the
    // MFMAs of the current one (the compiler's order within a chunk; left free
    // across chunks: down 144 us, 136 so).
    uint32_t w[2][8];
    take(0, 0, w[0]);
    take(1, 0, w[1]);
    Scaled sq = scaled(sv, bv, 0);
    bf16x8_t bf[2][2];
    weights(w, sq, 0, bf[0]);
#pragma unroll
    for (int ci = 0; ci < 4 * SG; ++ci) {
      const int gi = ci / 4, kc = ci & 3;
      bf16x8_t af[NMB];
      read_a(af, xst, kc);
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
        for (int s = 0; s < 2; ++s)
          acc[mb][s] = mfma32x32x16(af[mb], bf[ci & 1][s], acc[mb][s]);
      if (ci + 1 < 4 * SG) {
        if (kc == 3) {
          take(0, gi + 1, w[0]);
          take(1, gi + 1, w[1]);
          sq = scaled(sv, bv, gi + 1);
        }
        weights(w, sq, (kc + 1) & 3, bf[(ci + 1) & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kc == 3) {
        store_x(xst ^ 1);
        if constexpr (SBM == kSbLds) {
          if (gi == 0) store_sp(buf ^ 1, ws / (CS / 2), sp);
        }
        __syncthreads();
        xst ^= 1;
        if (gi + 1 < SG) load_x();
      }
    }
    if constexpr (SBM == kSbLds) {
      if (++ws == CS) {
        ws = 0;
        buf ^= 1;
        if (++ck == G / kSbChunk) ck = 0;
      }
    }
    if (++s == T) {
      epilogue(nt);
      clear();
      s = 0;
      ++nt;
    }
  }
  return nonfinite != 0;
}

template <int BITS, bool GATED, int SBM>
__global__ __launch_bounds__(kNT, 2) void qgemm_prefill_tall_kernel(RegLaunch L) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  RegUnit<kRows> u;
  if (!u.place(L, blockIdx.x)) return;
  u.find_rows(L);
  const RegArgs r = pick_reg(u.second, L.a2, L.x_bytes2, L.a, L.x_bytes);
  bool nonfinite;
  if (u.rows > 96)
    nonfinite = tall_unit<BITS, GATED, SBM, 4>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows, u.nt0,
                                              u.nt1, smem);
  else if (u.rows > 64)
    nonfinite = tall_unit<BITS, GATED, SBM, 3>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows, u.nt0,
                                              u.nt1, smem);
  else if (u.rows > 32)
    nonfinite = tall_unit<BITS, GATED, SBM, 2>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows, u.nt0,
                                              u.nt1, smem);
  else
    nonfinite = tall_unit<BITS, GATED, SBM, 1>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows, u.nt0,
                                              u.nt1, smem);
  if constexpr (BITS == 4) {
    if (nonfinite) exact4_unit<GATED, kRows>(kWaves);
  }
}

}  // namespace

hipError_t launch_qgemm_prefill_tall(const QGemmArgs& a, int64_t x_rows, int64_t max_tiles,
                                     hipStream_t s, const char* profile,
                                     const QGemmArgs* shared, int64_t rows2) {
  if (a.bits != 4 && a.bits != 8) return hipErrorInvalidValue;
  const int64_t tiles2 = shared ? (rows2 + kRows - 1) / kRows : 0;
  if (max_tiles <= 0 && tiles2 <= 0) return hipSuccess;
  const QGemmArgs& b = shared ? *shared : a;
  const int cols = a.gated ? 32 * kWaves : 64 * kWaves;
  const int tiles_n = (a.N + cols - 1) / cols;
  const int G = a.K / 64;
  int ntl = 1;
  while (ntl < tiles_n && G * ntl < MLXR_PFR_GROUPS &&
         (max_tiles + tiles2) * ((tiles_n + 2 * ntl - 1) / (2 * ntl)) >= MLXR_PFR_MIN_UNITS)
    ntl *= 2;
  const int units_n = (tiles_n + ntl - 1) / ntl;
  const auto sb_bits = [](const QGemmArgs& q) {
    return reinterpret_cast<uintptr_t>(q.w0.scales) | reinterpret_cast<uintptr_t>(q.w0.biases) |
           (q.gated ? reinterpret_cast<uintptr_t>(q.w1.scales) |
                          reinterpret_cast<uintptr_t>(q.w1.biases)
                    : 0);
  };
  const uintptr_t sb_addr = sb_bits(a) | sb_bits(b);
  // 8-group chunks load as aligned 16-byte pieces, a step's groups as one
  // aligned vector; anything else by element
  const bool sb_lds = G % kSbChunk == 0 && (sb_addr & 15) == 0;
  const bool sb_vec = a.bits == 4 ? G % 4 == 0 && (sb_addr & 7) == 0
                                  : G % 2 == 0 && (sb_addr & 3) == 0;
  const dim3 grid((unsigned)(reg_grid(max_tiles, units_n) + reg_grid(tiles2, units_n)));
  const RegLaunch L{a, tiles_n, ntl, units_n, (uint32_t)(x_rows * a.x_ld * 2),
                    b, (int32_t)tiles2, (int32_t)rows2, (uint32_t)(rows2 * b.x_ld * 2)};
  ProfileScope prof(profile, s);
#define MLXR_PT(B, G_, V)                                                        \
  qgemm_prefill_tall_kernel<B, G_, V><<<grid, kNT, tall_lds(V), s>>>(L)
#define MLXR_PT_V(B, V)       \
  do {                        \
    if (a.gated)              \
      MLXR_PT(B, true, V);    \
    else                      \
      MLXR_PT(B, false, V);   \
  } while (0)
#define MLXR_PT_S(B)            \
  do {                          \
    if (sb_lds)                 \
      MLXR_PT_V(B, kSbLds);     \
    else if (sb_vec)            \
      MLXR_PT_V(B, kSbVector);  \
    else                        \
      MLXR_PT_V(B, kSbAny);  \
  } while (0)
  if (a.bits == 4)
    MLXR_PT_S(4);
  else
    MLXR_PT_S(8);
#undef MLXR_PT_S
#undef MLXR_PT_V
#undef MLXR_PT
  return hipGetLastError();
}

}  // namespace mlxr_moe
