// Grouped quantised expert GEMM for a few tens of rows per expert: 64-row
// M-tiles, the weights dequantised in registers.
//
// Same operation and the same sums, in the same order, as the LDS-tiled
// kernels of prefill.hip (v_mfma_f32_32x32x16_bf16 over each 64-wide group in
// four 16-wide chunks, groups ascending): the outputs do not depend on which
// of them runs.
//
// At these sizes a tile dequantises every weight for 64 rows or fewer, so the
// dequantisation and what is done with its result bound the launch, not the
// MFMAs.  The LDS-tiled form writes each dequantised group to LDS, waits at a
// barrier, and reads it back; here a wave owns its columns (32 gate and the
// same 32 up channels, or 64 down channels) for all the tile's rows, so the
// MFMA's B operand goes from the dequantisation straight into the MFMA.  Only
// x goes through LDS, 256 inputs at a time: one barrier per four groups, none
// once x is whole in LDS (K <= 512).
//
// Weight loads are whole 128-byte lines (eight lanes a row, four groups of
// it at 4 bits, two at 8), turned to the operand layout -- lane l holds
// channel l % 32 -- through the wave's own 4 KB of LDS; the line after is in
// flight while a line is multiplied, also across the N-tiles of one unit (a
// unit is one M-tile and ntl N-tiles, so short input dims do not pay a
// prologue per tile).  An MFMA chunk wants consecutive pieces of one group on
// the two halves of the wave: v_permlane32_swap_b32 turns two registers into
// the operands of two chunks.  Scales and biases of long rows are copied to
// LDS 32 groups at a time: fetched step by step their lines, 64 groups long,
// would have left the L2 between uses.  Short rows (K <= 1024) share a few
// lines and are read where they are used.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "prefill_dev.hpp"
#include "prefill_reg.hpp"

namespace mlxr_moe {
namespace {

constexpr int kRows = 64;                   // rows per M-tile
constexpr int kWaves = 4, kNT = 64 * kWaves;
constexpr int kGroupBytes = kRows * 128;    // one group of x in LDS
constexpr int kXBytes = 2 * kGroupBytes;    // x stage: two groups
constexpr int kScratch = 4096;              // per wave: line turn, epilogue
constexpr int kSbChunk = 32;                // groups of scales in LDS at a time
constexpr int kSbArray = 32 * kSbChunk * 2;  // per wave: [side][s, b] of these
constexpr int kSbBytes = 4 * kSbArray;
constexpr int kSbMinGroups = 17;            // fewer: read from memory
constexpr int kResGroups = 8;               // x whole in LDS up to here

constexpr int reg_lds(int sbm, bool res) {
  return (res ? kResGroups * kGroupBytes : 2 * kXBytes) +
         kWaves * (kScratch + (sbm == kSbLds ? kSbBytes : 0));
}
// two workgroups share a CU's 160 KB
static_assert(2 * reg_lds(kSbLds, false) <= 160 * 1024 &&
                  2 * reg_lds(kSbVector, true) <= 160 * 1024,
              "two workgroups per CU");

// groups per macro step: whole weight steps and whole x stages
template <int BITS>
constexpr int kMacroGroups = BITS == 4 ? 4 : 2;

// The rows [slot0, slot0 + rows) of expert e against N-tiles [nt0, nt1).
// NMB: 32-row blocks that hold rows.  RES: x whole in LDS.  Returns (for the
// whole wave) whether a 4-bit scale may have been too large (exact4_unit).
template <int BITS, bool GATED, int SBM, bool RES, int NMB>
__device__ __forceinline__ bool reg_unit(const RegArgs& a, int N, int K, int e, int slot0,
                                         int rows, int nt0, int nt1, char* smem) {
  constexpr int SG = kStepGroups<BITS>, MG = kMacroGroups<BITS>;
  constexpr int TC = GATED ? 32 * kWaves : 64 * kWaves;  // channels per N-tile
  constexpr int WC = TC / kWaves;                        // ... per wave
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int G = K >> 6;                  // groups
  const int S = (G + MG - 1) / MG;       // macro steps per tile
  const int T = S * (MG / SG);           // weight steps per tile
  const int total = S * (nt1 - nt0);     // macro steps of this unit
  char* xl = smem;
  char* scratch = smem + (RES ? kResGroups * kGroupBytes : 2 * kXBytes) +
                  wave * (kScratch + (SBM == kSbLds ? kSbBytes : 0));
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
    if constexpr (BITS != 16 && SBM != kSbLds) {
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
  // The scales and biases of groups 32 k .. of tile nt into LDS, as
  // [side][s, b][32 rows][n groups], n = min(G, 32).  Rows of up to 32 groups
  // follow each other in memory as they do here; of longer ones (G % 8 == 0)
  // each gives 64 bytes.  All loads are issued before the first store.
  const int sbn = min(G, kSbChunk);
  u32x4_t sp[8];
  auto load_sp = [&](int nt, int k) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int arr = i >> 1, id = lane + 64 * (i & 1);  // 16-byte piece id
      const bool up = GATED && (arr & 2);
      const uint16_t* q = arr & 1 ? (up ? a.w1.biases : a.w0.biases)
                                  : (up ? a.w1.scales : a.w0.scales);
      const int ch0 = channel0(nt, arr >> 1);
      const int64_t row0 = (int64_t)e * a.e_rows + ch0;
      const int valid = N - ch0;  // rows below N
      int64_t off;                // elements; pieces past the copy repeat its last
      if (G <= kSbChunk)
        off = row0 * G + 8 * max(0, min(id, min(32, valid) * G / 8 - 1));
      else
        off = (row0 + min(id >> 2, valid - 1)) * G + kSbChunk * k + 8 * (id & 3);
      if (valid <= 0) off = 0;
      // (groups of the row's last, partial chunk: up to its end)
      if (G > kSbChunk && kSbChunk * k + 8 * (id & 3) >= G) off = 0;
      sp[i] = *(gptr<const u32x4_t>)(as_global<const uint16_t>(q) + off);
    }
  };
  auto store_sp = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int arr = i >> 1, id = lane + 64 * (i & 1);
      if (8 * id < 32 * sbn)
        *reinterpret_cast<u32x4_t*>(sbl + arr * kSbArray + 16 * id) = sp[i];
    }
  };

  WStep W0, W1;
  load_w(W0);
  if constexpr (SBM == kSbLds) load_sp(nt0, 0);
  __builtin_amdgcn_sched_barrier(0);

  // ---- x: thread -> 16-byte chunk tid % 16 (of the stage's 256) of rows
  // tid / 16 + 16 j; chunk cc of row r of a group sits at cc ^ ((r >> 1) & 7)
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.x), 0, (int)a.x_bytes, kBufFlags);
  constexpr int XC = 2 * NMB;  // rows per thread
  const int xrow0 = tid >> 4, xc = tid & 15;
  uint32_t aoff[XC];
  {
    int xrow[XC];
#pragma unroll
    for (int j = 0; j < XC; ++j) xrow[j] = slot0 + min(xrow0 + 16 * j, rows - 1);
    if (!a.x_by_slot) {
#pragma unroll
      for (int j = 0; j < XC; ++j) xrow[j] = as_global<const int32_t>(a.sorted)[xrow[j]];
      if (a.row_map) {
#pragma unroll
        for (int j = 0; j < XC; ++j) xrow[j] = as_global<const int32_t>(a.row_map)[xrow[j]];
      } else {
        const float rdiv = 1.0f / (float)a.row_div;
#pragma unroll
        for (int j = 0; j < XC; ++j) xrow[j] = div_small(xrow[j], a.row_div, rdiv);
      }
    }
#pragma unroll
    for (int j = 0; j < XC; ++j)
      aoff[j] = xrow0 + 16 * j < rows ? (uint32_t)((int64_t)xrow[j] * a.x_ld * 2 + 16 * xc)
                                      : kPastEnd;
  }
  const int aw = (xc >> 3) * kGroupBytes + xrow0 * 128 + 16 * ((xc & 7) ^ swz(xrow0));
  u32x4_t xv[XC];
  // x stages per tile: two groups each (rows of kSbAny: up to K's end)
  const int XS = BITS == 4 && SBM == kSbAny ? (G + 1) / 2 : S * (MG / 2);
  int px = 0, left_x = XS * (nt1 - nt0);
  auto load_x = [&]() {  // the next x stage (zeros past K and past the unit)
    const bool ok = left_x > 0 && 128 * px + 8 * xc < K;
#pragma unroll
    for (int j = 0; j < XC; ++j)
      xv[j] = __builtin_amdgcn_raw_buffer_load_b128(
          xr, ok && aoff[j] != kPastEnd ? aoff[j] + 256 * px : kPastEnd, 0, 0);
    px = px + 1 < XS ? px + 1 : 0;
    --left_x;
  };
  auto store_x = [&](int st) {
#pragma unroll
    for (int j = 0; j < XC; ++j)
      *reinterpret_cast<u32x4_t*>(xl + st * kXBytes + aw + 2048 * j) = xv[j];
  };
  // the flat output row of tile row `lane` (the down projection)
  int orow = slot0 + min(lane, rows - 1);
  if (!GATED && a.out_by_flat) orow = as_global<const int32_t>(a.sorted)[orow];
  load_x();
  store_x(0);
  if constexpr (RES) {
    for (int st = 1; st < XS; ++st) {
      load_x();
      store_x(st);
    }
  }
  if constexpr (SBM == kSbLds) store_sp();
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

  // ---- a loaded line to the operand layout: lane (c, h) gets the bytes
  // [64 h, 64 h + 64) of channel c's line (bf16 weights: chunks 2 i + h),
  // then halves are swapped so that each register is one chunk's operand.
  // (One wave's LDS operations execute in order.)
  const int tw = lrow * 128 + 16 * (lch ^ lrow);
  const int tr = c * 128;
  auto turn = [&](WStep& W) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<u32x4_t*>(scratch + 1024 * i + tw) = W.w[s][i];
      wave_sync();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = BITS == 16 ? 2 * i + h : 4 * h + i;
        W.w[s][i] =
            *reinterpret_cast<const u32x4_t*>(scratch + tr + 16 * (p ^ (c & 7)));
      }
      wave_sync();
    }
    if constexpr (BITS != 16) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t w[4] = {W.w[s][i].x, W.w[s][i].y, W.w[s][i].z, W.w[s][i].w};
          swap32(w[0], w[BITS == 4 ? 1 : 2]);
          swap32(w[BITS == 4 ? 2 : 1], w[3]);
          W.w[s][i] = u32x4_t{w[0], w[1], w[2], w[3]};
        }
    }
  };
  // scales and biases of the step's groups, two per register, on every lane
  auto scales = [&](const WStep& W, int g0, uint32_t (&sv)[2][2],
                    uint32_t (&bv)[2][2]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if constexpr (SBM == kSbLds) {
        const char* p = sbl + 2 * s * kSbArray + 2 * (c * sbn + g0);
        if constexpr (BITS == 4) {
          const u32x2_t u = *reinterpret_cast<const u32x2_t*>(p);
          const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p + kSbArray);
          sv[s][0] = u.x, sv[s][1] = u.y, bv[s][0] = v.x, bv[s][1] = v.y;
        } else {
          sv[s][0] = *reinterpret_cast<const uint32_t*>(p);
          bv[s][0] = *reinterpret_cast<const uint32_t*>(p + kSbArray);
        }
      } else if constexpr (BITS != 16) {
#pragma unroll
        for (int j = 0; j < (SG + 1) / 2; ++j) {
          sv[s][j] = bv[s][j] = W.sb[s][j];
          swap32(sv[s][j], bv[s][j]);
        }
      }
    }
  };

  // ---- x operand of chunk kc of group gx of x stage st
  const int aswz = swz(c);
  auto read_a = [&](bf16x8_t (&af)[NMB], int st, int gx, int kc) {
    const char* A = xl + st * kXBytes + gx * kGroupBytes + c * 128;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
      af[mb] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(
          A + 4096 * mb + 16 * ((2 * kc + h) ^ aswz)));
  };
  // ---- groups gi0 .. gi0 + n - 1 of a weight step times those of x stage st
  // from group gx on; the x operand is read a chunk ahead
  auto multiply = [&](const WStep& W, const uint32_t (&sv)[2][2], const uint32_t (&bv)[2][2],
                      int gi0, int n, int st, int gx) {
    bf16x8_t af[2][NMB];
    read_a(af[0], st, gx, 0);
#pragma unroll
    for (int g = 0; g < n; ++g) {
      const int gi = gi0 + g;
      float sc[2], s4[2], bi[2];
      if constexpr (BITS != 16) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          sc[s] = __uint_as_float(gi & 1 ? sv[s][gi / 2] & 0xffff0000u : sv[s][gi / 2] << 16);
          bi[s] = __uint_as_float(gi & 1 ? bv[s][gi / 2] & 0xffff0000u : bv[s][gi / 2] << 16);
          if constexpr (BITS == 4) {
            s4[s] = sc[s] * 0x1p20f;
            sc[s] *= 0x1p24f;
            // (kept, not recomputed for every word)
            asm("" : "+v"(sc[s]), "+v"(s4[s]));
          }
        }
      }
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) {
        const int ci = 4 * g + kc;
        if (ci + 1 < 4 * n) read_a(af[(ci + 1) & 1], st, gx + (ci + 1) / 4, (kc + 1) & 3);
        bf16x8_t bf[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          uint32_t o[4];
          if constexpr (BITS == 16) {
            bf[s] = as_bf16x8(W.w[s][kc]);
          } else {
            if constexpr (BITS == 4) {
              // group gi: loads 2 (gi & 1) + {0, 1}, words 2 kc + (gi >> 1) of the eight
              const int k = 2 * kc + (gi >> 1);
              dequant4(W.w[s][2 * (gi & 1) + k / 4][k % 4], sc[s], s4[s], bi[s], o);
            } else {
              dequant8(W.w[s][kc][2 * gi], sc[s], bi[s], o);
              dequant8(W.w[s][kc][2 * gi + 1], sc[s], bi[s], o + 2);
            }
            bf[s] = as_bf16x8(u32x4_t{o[0], o[1], o[2], o[3]});
          }
        }
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int s = 0; s < 2; ++s)
            acc[mb][s] = mfma32x32x16(af[ci & 1][mb], bf[s], acc[mb][s]);
      }
    }
  };

  // ---- a finished tile: through the wave's scratch, 32 rows at a time, so
  // that every store is 16 bytes of a row
  uint16_t* O = reinterpret_cast<uint16_t*>(scratch);
  uint64_t nonfinite = 0;  // (a scale too large: not one sum of its channel is finite)
  auto epilogue = [&](int nt) {
    if constexpr (BITS == 4)
      nonfinite |= __ballot(!__builtin_isfinite(acc[0][0][0]) || !__builtin_isfinite(acc[0][1][0]));
    const int och0 = nt * TC + wave * WC;
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
        const int64_t orw = GATED ? slot0 + trow : __shfl(orow, trow, 64);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(O + row * WC + 8 * cc);
        if (trow < rows && och0 + 8 * cc < N)
          *(gptr<u32x4_t>)(as_global<uint16_t>(a.out) + orw * a.out_ld + och0 + 8 * cc) = v;
      }
      wave_sync();
    }
  };

  // ---- the macro steps.  Issue order within one: the next x stage, the next
  // weight step (a wait for x leaves the weights in flight), then the
  // multiplies.
  int nt = nt0, s = 0;      // tile, macro step within it
  int xst = 0;              // the x stage that is read next
  int g32 = 0, ck = 0;      // group within its scale chunk, chunk within the tile
  auto macro = [&](WStep& A, WStep& B) {
#pragma unroll
    for (int u = 0; u < MG / SG; ++u) {
      WStep& cur = u & 1 ? B : A;
      WStep& nxt = u & 1 ? A : B;
      if (!RES && u % (2 / (SG < 2 ? SG : 2)) == 0) load_x();
      __builtin_amdgcn_sched_barrier(0);
      load_w(nxt);
      __builtin_amdgcn_sched_barrier(0);
      turn(cur);
      uint32_t sv[2][2], bv[2][2];
      if constexpr (SBM == kSbLds) {
        scales(cur, g32, sv, bv);
        g32 += SG;
      } else {
        scales(cur, 0, sv, bv);
      }
#pragma unroll
      for (int gi = 0; gi < SG; gi += 2) {
        multiply(cur, sv, bv, gi, SG == 1 ? 1 : 2, xst, SG == 1 ? u : 0);
        if (SG == 1 && u == 0) continue;  // the stage's second group follows
        // (RES: the tile's stages follow each other in LDS)
        if constexpr (RES) {
          ++xst;
        } else {
          store_x(xst ^ 1);
          __syncthreads();
          xst ^= 1;
        }
        if (BITS == 4 && SBM == kSbAny && SG * s + gi + 2 >= G) break;  // K's end
        if (!RES && gi + 2 < SG) load_x();
      }
      if constexpr (SBM == kSbLds) {
        if (g32 >= min(kSbChunk, G - kSbChunk * ck)) {
          g32 = 0;
          if (++ck * kSbChunk >= G) ck = 0;
          const int lt = ck ? nt : nt + 1;
          if (lt < nt1) {
            load_sp(lt, ck);
            store_sp();
            wave_sync();
          }
        }
      }
    }
    if (++s == S) {
      epilogue(nt);
      clear();
      s = 0;
      ++nt;
      if (RES) xst = 0;
    }
  };
  if constexpr (MG == SG) {
    int q = 0;
#pragma nounroll
    for (; q + 1 < total; q += 2) {
      macro(W0, W1);
      macro(W1, W0);
    }
    if (q < total) macro(W0, W1);
  } else {
#pragma nounroll
    for (int q = 0; q < total; ++q) macro(W0, W1);
  }
  return nonfinite != 0;
}

template <int BITS, bool GATED, int SBM, bool RES>
__global__ __launch_bounds__(kNT, 2) void qgemm_prefill_reg_kernel(RegLaunch L) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  RegUnit<kRows> u;
  if (!u.place(L, blockIdx.x)) return;
  u.find_rows(L);
  const RegArgs r = pick_reg(u.second, L.a2, L.x_bytes2, L.a, L.x_bytes);
  bool nonfinite;
  if (u.rows > 32)
    nonfinite = reg_unit<BITS, GATED, SBM, RES, 2>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows,
                                                  u.nt0, u.nt1, smem);
  else
    nonfinite = reg_unit<BITS, GATED, SBM, RES, 1>(r, L.a.N, L.a.K, u.e, u.slot0, u.rows,
                                                  u.nt0, u.nt1, smem);
  if constexpr (BITS == 4) {
    if (nonfinite) exact4_unit<GATED, kRows>(kWaves);
  }
}

}  // namespace

hipError_t launch_qgemm_prefill_reg(const QGemmArgs& a, int64_t x_rows, int64_t max_tiles,
                                    hipStream_t s, const char* profile, const QGemmArgs* shared,
                                    int64_t rows2) {
  const int64_t tiles2 = shared ? (rows2 + kRows - 1) / kRows : 0;
  if (max_tiles <= 0 && tiles2 <= 0) return hipSuccess;
  const QGemmArgs& b = shared ? *shared : a;
  const int cols = a.gated ? 32 * kWaves : 64 * kWaves;
  const int tiles_n = (a.N + cols - 1) / cols;
  const int G = a.K / 64;
  // N-tiles per unit: at least 2048 inputs' worth of groups where the grid
  // stays large
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
  // 32-group chunks load as aligned 16-byte pieces and are read a step's
  // groups at a time; one aligned vector per step; anything else by element
  const bool sb_lds = G >= kSbMinGroups && G % (a.bits == 4 ? 4 : 2) == 0 &&
                      (G <= kSbChunk || G % 8 == 0) && (sb_addr & 15) == 0;
  const bool sb_vec = a.bits == 4 ? G % 4 == 0 && (sb_addr & 7) == 0
                                  : G % 2 == 0 && (sb_addr & 3) == 0;
  const bool res = G <= kResGroups;
  const dim3 grid((unsigned)(reg_grid(max_tiles, units_n) + reg_grid(tiles2, units_n)));
  const RegLaunch L{a, tiles_n, ntl, units_n, (uint32_t)(x_rows * a.x_ld * 2),
                    b, (int32_t)tiles2, (int32_t)rows2, (uint32_t)(rows2 * b.x_ld * 2)};
  ProfileScope prof(profile, s);
#define MLXR_PR(B, G_, V, R)                                                               \
  qgemm_prefill_reg_kernel<B, G_, V, R><<<grid, kNT, reg_lds(V, R), s>>>(L)
  // (a gated launch of K <= 512 takes the general form: one instance less)
#define MLXR_PR_V(B, V)            \
  do {                             \
    if (a.gated)                   \
      MLXR_PR(B, true, V, false);  \
    else if (res && V != kSbLds)   \
      MLXR_PR(B, false, (V == kSbLds ? kSbVector : V), true); \
    else                           \
      MLXR_PR(B, false, V, false); \
  } while (0)
#define MLXR_PR_S(B)            \
  do {                          \
    if (sb_lds)                 \
      MLXR_PR_V(B, kSbLds);     \
    else if (sb_vec)            \
      MLXR_PR_V(B, kSbVector);  \
    else                        \
      MLXR_PR_V(B, kSbAny);  \
  } while (0)
  if (a.bits == 16)
    MLXR_PR_V(16, kSbAny);
  else if (a.bits == 4)
    MLXR_PR_S(4);
  else
    MLXR_PR_S(8);
#undef MLXR_PR_S
#undef MLXR_PR_V
#undef MLXR_PR
  return hipGetLastError();
}

}  // namespace mlxr_moe
