// The streaming decode GEMM's device code, shared by its kernels over 8-row
// work items (qgemm.hip) and over 16-row ones (qgemm_wide.hip), and its launch
// shape.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace mlxr_moe {

// Launch shape of the streaming kernel: (experts x 16-channel blocks) from
// which it runs, waves per workgroup, super-steps of loads in flight at 4-
// and 8-bit.
// (measured at T = 1..4: the streaming kernel's time is nearly flat in the
// blocks there, ~11.8 us for c2/c4 gate/up, while the split-K kernel's
// grows with the bytes: 10.1 us at 8 experts x 512 channels (288 blocks),
// 13.7 at 10 x 512 (352) and 8 x 768 (432))
#ifndef MLXR_STREAM_MIN_BLOCKS
#define MLXR_STREAM_MIN_BLOCKS 320
#endif
#ifndef MLXR_STREAM_WAVES
#define MLXR_STREAM_WAVES 4
#endif
#ifndef MLXR_STREAM_DEPTH4
#define MLXR_STREAM_DEPTH4 1
#endif
#ifndef MLXR_STREAM_DEPTH8
#define MLXR_STREAM_DEPTH8 1
#endif
// ... of the 8-token form (half the bytes per super-step: twice the depth)
#ifndef MLXR_STREAM_DEPTH4_TT8
#define MLXR_STREAM_DEPTH4_TT8 (2 * MLXR_STREAM_DEPTH4)
#endif
#ifndef MLXR_STREAM_DEPTH8_TT8
#define MLXR_STREAM_DEPTH8_TT8 (2 * MLXR_STREAM_DEPTH8)
#endif
// ... and of the gated kernels (gate and up: two rows of loads per step).
// The 4-bit gated 8-token form keeps three super-steps in flight: a ring
// of four slots divides its 16 super-steps at K = 2048 (with three slots two
// zero steps follow the last one).  Measured (event means, c2 T=8/32/64,
// c4 T=64, c6 T=64): gate/up 0.3-1% faster; depth 3 for the 4-token form
// was 2-12% slower.
#ifndef MLXR_STREAM_DEPTH4G
#define MLXR_STREAM_DEPTH4G MLXR_STREAM_DEPTH4
#endif
#ifndef MLXR_STREAM_DEPTH4G_TT8
#define MLXR_STREAM_DEPTH4G_TT8 3
#endif
#ifndef MLXR_STREAM_DEPTH8G
#define MLXR_STREAM_DEPTH8G MLXR_STREAM_DEPTH8
#endif
#ifndef MLXR_STREAM_DEPTH8G_TT8
#define MLXR_STREAM_DEPTH8G_TT8 (2 * MLXR_STREAM_DEPTH8G)
#endif
#ifndef MLXR_SCHED_BARRIER
#define MLXR_SCHED_BARRIER() __builtin_amdgcn_sched_barrier(0)
#endif

constexpr int64_t kStreamMinBlocks = MLXR_STREAM_MIN_BLOCKS;
#ifndef MLXR_STREAM_SLOTS
#define MLXR_STREAM_SLOTS 512
#endif
// workgroups resident at once (2 per CU on 256 CUs)
constexpr int64_t kStreamSlots = MLXR_STREAM_SLOTS;

// Reorder 8 consecutive bf16 x values to the code order that unpack4 emits:
// element j of the fragment holds x[perm(j)], perm = 0,4,1,5,2,6,3,7.
__device__ __forceinline__ u32x4_t perm4(u32x4_t v) {
  u32x4_t r;
  r.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
  r.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
  r.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
  r.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
  return r;
}

// 8 nibbles -> bf16 (1 + code/16): nibble k moves to mantissa bits 6..3 of
// its half; pairs (n0,n4) (n1,n5) (n2,n6) (n3,n7).  Written as one shift and
// one v_and_or_b32 per output: a VOP3 op takes one scalar operand here, so
// the mask rides in an SGPR and the bf16 1.0 pair in a VGPR (`one`).
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t m,
                                           uint32_t one) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(m), "v"(one));
  return r;
}
__device__ __forceinline__ u32x4_t unpack4(uint32_t w, uint32_t one) {
  const uint32_t m = 0x00780078u;
  u32x4_t r;
  r.x = and_or(w << 3, m, one);
  r.y = and_or(w >> 1, m, one);
  r.z = and_or(w >> 5, m, one);
  r.w = and_or(w >> 9, m, one);
  return r;
}
__device__ __forceinline__ u32x4_t unpack4(uint32_t w) {
  return unpack4(w, 0x3F803F80u);
}

// 8 bytes (two words) -> bf16 codes in natural order.  Integers <= 255 are
// exact in bf16, so the top half of the exact f32 is the bf16 value.
__device__ __forceinline__ uint32_t pack_hi(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo),
                               0x07060302u);
}
__device__ __forceinline__ u32x4_t unpack8(uint32_t w0, uint32_t w1) {
  u32x4_t r;
  r.x = pack_hi((float)(w0 & 0xffu), (float)((w0 >> 8) & 0xffu));
  r.y = pack_hi((float)((w0 >> 16) & 0xffu), (float)(w0 >> 24));
  r.z = pack_hi((float)(w1 & 0xffu), (float)((w1 >> 8) & 0xffu));
  r.w = pack_hi((float)((w1 >> 16) & 0xffu), (float)(w1 >> 24));
  return r;
}

// sc * P + cb * X terms of one group from its bf16 scale and bias bits.
template <int BITS>
__device__ __forceinline__ void group_terms(uint32_t s16, uint32_t b16,
                                            float& sc, float& cb) {
  const float sf = __uint_as_float(s16 << 16);
  const float bf = __uint_as_float(b16 << 16);
  if constexpr (BITS == 4) {
    sc = 16.0f * sf;
    cb = __builtin_fmaf(-16.0f, sf, bf);
  } else {
    sc = sf;
    cb = bf;
  }
}

// The unit of workgroup blockIdx.x: a work item of the routed problem `a`
// (its record, fetched whole: header and flat rows), or, from units1 on,
// an item of a folded second problem -- the block's shared expert, every
// token's row once: item i is rows 8i..8i+7 (16i..16i+15 of wide items) of
// `rows2` in token order, its record made here (expert 0, the rows' own slots,
// no dispatch).  Returns false for an idle workgroup (past the routed problem's
// items).
struct Unit {
  const int32_t* rec;
  int4 wk, fr0, fr1;
  int tile;
  bool shared;
};
template <int WR = kWorkRows>  // rows per item, or 0: a.work_rows
__device__ __forceinline__ bool decode_unit(const QGemmArgs& a, int tiles_n,
                                            int units1, int items1, int rows2,
                                            Unit& u) {
  u.shared = (int)blockIdx.x >= units1;
  const int v = u.shared ? (int)blockIdx.x - units1 : (int)blockIdx.x;
  const int ai = v / tiles_n;
  u.tile = v - ai * tiles_n;
  // (the routed record is read unconditionally, item 0's for a shared
  // unit)
  const int wr = WR ? WR : a.work_rows;
  u.rec = a.work + (int64_t)kWorkInts * (u.shared ? 0 : min(ai, items1 - 1));
  u.wk = *reinterpret_cast<const int4*>(u.rec);
  u.fr0 = *reinterpret_cast<const int4*>(u.rec + 4);
  u.fr1 = *reinterpret_cast<const int4*>(u.rec + 8);
  const int n_act = *a.num_work;
  if (u.shared) {
    const int r0 = wr * ai;
    u.wk = make_int4(0, r0, min(wr, rows2 - r0), rows2);
    u.fr0 = make_int4(r0, r0 + 1, r0 + 2, r0 + 3);
    u.fr1 = make_int4(r0 + 4, r0 + 5, r0 + 6, r0 + 7);
    return true;
  }
  return ai < n_act;
}

// Streaming decode GEMM for many (work item, channel tile) units.  One
// workgroup = `waves` waves = one work item (at most 8 rows of one expert)
// x one tile of waves*nb*16 output channels; wave w owns nb 16-channel
// blocks over the whole input dim, so no partial sums cross waves.  The
// workgroup stages the item's x rows (bf16, in the MFMA operand order) and
// the per-group token sums X in LDS once; each wave then streams its
// blocks' packed weights with D super-steps of loads in flight (a register
// ring) and reads x from LDS.
//
// Prologue order: the work record (one scalar load: the expert and the flat
// row of each slot, so the x rows need no further lookup), then the first D
// weight super-steps, the wave's scales and biases and the x rows are all
// issued before the first LDS store, so the weight stream starts one memory
// round trip after the workgroup does.
//
// Block-diagonal MFMA: the 16 rows of the A operand are TT tokens x GG
// groups (GG = 16 / TT).  Lane quarter q (l/16) supplies the codes of group
// q*GG/4 of the super-step, and the x operand row (group j, token t) is
// non-zero only on the lanes of group j, so one v_mfma_f32_16x16x32_bf16
// yields the partial sums of GG groups at once and every lane applies the
// scale and bias of a single group.  A super-step covers GG groups; each
// lane loads 16*GG codes of its group (16 B per load).  Lanes that feed
// zeros read a zero block in LDS.  The GG partial sums of a token meet by
// cross-lane adds at the end.
template <int BITS, bool GATED, int TT, int D, int NB, int KS>
__device__ __forceinline__ void stream_body(const QGemmArgs& a,
                                            const int32_t* rec, int4 wk,
                                            int4 fr0, int4 fr1, int tile,
                                            char* smem, int ltid, int lthreads,
                                            uint16_t* yl, int yrow_off) {
  constexpr int nb = NB;
  constexpr int NM = GATED ? 2 : 1;
  constexpr int NA = 2 * NM;            // scale and bias arrays
  constexpr int GG = 16 / TT;           // groups per MFMA
  constexpr int LPG = 4 / GG;           // lane quarters per group
  constexpr int CPL = 64 / LPG;         // codes per lane per super-step
  constexpr int NL = CPL * BITS / 128;  // 16-byte loads per lane
  constexpr int NMF = CPL / 8;          // MFMAs per super-step
  constexpr int WPG = 2 * BITS;         // packed words per row and group
  // KS waves share each set of blocks, one K-slice each (KS > 1 for small
  // grids: more, shorter waves); their sums meet in LDS at the end
  const int waves = (lthreads >> 6) / KS;  // channel waves
  // items of experts with at most 4 rows run with TT = 4, the others with
  // TT = 8 (wide items of more than 8 rows in stream16_body): an item is
  // always one pass
  const int e = wk.x, row0 = wk.y, nt = min(wk.z, TT);
  const int lane = ltid & 63, wave_id = ltid >> 6;
  const int wave = wave_id / KS, kq = wave_id % KS;  // channel wave, K-slice
  const int n = lane & 15, q = lane >> 4;
  const int gq = q / LPG, sq = q % LPG;  // this lane's group, its part
  const int K = a.K, groups = K >> 6;
  const int ssteps = groups / GG;  // the host runs this kernel when GG | groups
  const int ssk = ssteps / KS;     // ... and KS | ssteps: steps per slice
  const int s0 = kq * ssk;         // this wave's first step of each block
  const int total = nb * ssk;      // super-steps of this wave, all blocks
  // LDS: x [TT][K + 8] bf16 (rows padded 16 B), 16 B zero block,
  // X [groups][TT] f32, then per wave its scales and biases
  const int xs = K + 8;
  uint16_t* xl = reinterpret_cast<uint16_t*>(smem);
  char* zero_blk = smem + (size_t)TT * xs * 2;
  float* Xl = reinterpret_cast<float*>(zero_blk + 16);
  char* sb_base =
      smem + (((size_t)TT * xs * 2 + 16 + (size_t)groups * TT * 4 + 15) & ~size_t(15));
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const u32x4_t zq = {0u, 0u, 0u, 0u};
  // this wave's blocks: nb consecutive 16-channel blocks from ch0
  const int ch0 = ((tile * waves + wave) * nb) * 16 + n;
  const int64_t wrow0 = (int64_t)e * a.e_rows + ch0;
  // A operand row of this lane: (group m / TT, token m % TT), m = l % 16
  const int arow_g = n / TT, arow_t = n % TT;

  // ring of R = D + 1 slots: global super-step gs lives in slot gs % R; the
  // load for gs + D goes into the slot that gs - 1 freed, so nothing is
  // copied, and the ring runs on across block boundaries
  constexpr int R = D + 1;
  struct Ring {
    u32x4_t w[NM][NL];
  };
  const uint32_t* wb[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const QWeights& W = m == 0 ? a.w0 : a.w1;
    wb[m] = W.w + (wrow0 * groups + gq) * WPG + sq * (CPL * BITS / 32);
  }
  const int64_t blk_rows = (int64_t)16 * groups;  // row stride of a block
  auto load = [&](Ring& r, int gs) {
    const int bi = gs / ssk, ss = s0 + gs - bi * ssk;
    const int64_t go = bi * blk_rows + ss * GG;  // group offset
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const u32x4_t* wp = reinterpret_cast<const u32x4_t*>(wb[m] + go * WPG);
#pragma unroll
      for (int i = 0; i < NL; ++i) r.w[m][i] = wp[i];
    }
  };
  // Prologue.  Loads retire in issue order, so what the staging waits for
  // is issued first: the x rows (L2 hits, shared by every tile of the
  // item), then the wave's scales and biases, then the first D weight
  // super-steps.  Staging x waits for the x loads alone, the barrier
  // follows, and the weights' memory round trip overlaps both.  Every load
  // is issued by every thread (indices clamped, the extra copies dropped):
  // a load under a branch would make the compiler's wait counts cover the
  // loads issued after it as well.

  // x rows of the item's tokens, from the record's flat rows (fetched with
  // its header; a row_map lookup issues every load before the first use)
  int64_t xr[TT];
  {
    const int fl[8] = {fr0.x, fr0.y, fr0.z, fr0.w, fr1.x, fr1.y, fr1.z, fr1.w};
    int32_t rm[TT];
    if (!a.x_by_slot && a.row_map) {
#pragma unroll
      for (int t = 0; t < TT; ++t) rm[t] = a.row_map[t < nt ? fl[t] : fl[0]];
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      int64_t r = 0;
      if (t < nt)
        r = a.x_by_slot ? row0 + t : (a.row_map ? rm[t] : fl[t] / a.row_div);
      xr[t] = r;
    }
  }
  // thread k8 holds elements 8*k8..8*k8+7 of every token; the token sums X
  // of each 64-wide group come from the 8 threads sharing it
  const int per_row = K >> 3;
  // (only the item's nt rows are read: the padding rows of the MFMA form
  // stage zeros.  The branch is uniform, and these are the first loads of
  // the workgroup, so every later wait counts only loads issued after them)
  auto load_x = [&](int k8, u32x4_t (&v)[TT]) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      v[t] = zq;
      if (t < nt) v[t] = *reinterpret_cast<const u32x4_t*>(a.x + xr[t] * a.x_ld + 8 * k8);
    }
  };
  auto stage_x = [&](int k8, const u32x4_t (&v)[TT]) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const u32x4_t vt = t < nt ? v[t] : zq;
      float sx = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sx += __uint_as_float(vt[j] << 16) + __uint_as_float(vt[j] & 0xffff0000u);
      sx += __shfl_xor(sx, 1, 64);
      sx += __shfl_xor(sx, 2, 64);
      sx += __shfl_xor(sx, 4, 64);
      if ((k8 & 7) == 0) Xl[(k8 >> 3) * TT + t] = sx;
      u32x4_t w = vt;
      if constexpr (BITS == 4) w = perm4(w);
      *reinterpret_cast<u32x4_t*>(xl + (size_t)t * xs + 8 * k8) = w;
    }
  };
  const int k8 = ltid;
  const bool x_in = k8 < per_row;
  u32x4_t xv[TT];
  load_x(min(k8, per_row - 1), xv);
  MLXR_SCHED_BARRIER();  // issue order is retire order: x first

  // Scales and biases of this wave's blocks: 16 rows x groups bf16 per
  // block and array, contiguous in memory, copied to the wave's own LDS
  // region with 16-byte loads (the hot loop then reads its two values per
  // step from LDS): a per-step 2-byte load per lane would touch 16 cache
  // lines for 128 useful bytes.
  const int sbn = nb * 16 * groups;  // bf16 per array
  const int sbv = sbn >> 3;          // 16-byte vectors per array
  uint16_t* sbl = reinterpret_cast<uint16_t*>(sb_base) + (size_t)wave_id * NA * sbn;
  const uint16_t* sbsrc[NA];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const QWeights& W = m == 0 ? a.w0 : a.w1;
    sbsrc[2 * m] = W.scales + (wrow0 - n) * groups;
    sbsrc[2 * m + 1] = W.biases + (wrow0 - n) * groups;
  }
  u32x4_t sv[NA];
  const bool s_in = lane < sbv;
  const int sl = min(lane, sbv - 1);
#pragma unroll
  for (int i = 0; i < NA; ++i)
    sv[i] = *reinterpret_cast<const u32x4_t*>(sbsrc[i] + 8 * sl);
  MLXR_SCHED_BARRIER();

  Ring ring[R];
#pragma unroll
  for (int j = 0; j < D; ++j) load(ring[j], min(j, total - 1));
  MLXR_SCHED_BARRIER();

  if (x_in) stage_x(k8, xv);  // per_row is a multiple of 8: whole octets
  // the rest of x (input dims above 64 * 8 * waves)
  for (int c8 = k8 + lthreads; c8 < per_row; c8 += lthreads) {
    u32x4_t v[TT];
    load_x(c8, v);
    stage_x(c8, v);
  }
  if (ltid == 0) *reinterpret_cast<u32x4_t*>(zero_blk) = zq;
  __syncthreads();
  // the scales (issued before the weights) -> this wave's region; only
  // this wave reads it
  if (s_in) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      *reinterpret_cast<u32x4_t*>(sbl + i * sbn + 8 * lane) = sv[i];
  }
  for (int i = lane + 64; i < sbv; i += 64) {
#pragma unroll
    for (int j = 0; j < NA; ++j)
      *reinterpret_cast<u32x4_t*>(sbl + j * sbn + 8 * i) =
          *reinterpret_cast<const u32x4_t*>(sbsrc[j] + 8 * i);
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // The loop issues the same loads every super-step (past the end they
  // repeat the last step, a cache hit) and holds no stores, so the
  // compiler can wait for exactly the oldest ring slot.  Steps past the
  // end multiply zeros.  With several blocks per wave each block's sums
  // move to done[block] when its last step is done (selects, so the
  // accumulators stay in registers).
  constexpr int ND = NB > 1 ? NB - 1 : 1;
  f32x4_t acc[NM], done[ND][NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    acc[m] = zero;
#pragma unroll
    for (int b = 0; b < ND; ++b) done[b][m] = zero;
  }
  const uint32_t one_v = 0x3F803F80u;
  // x operand source of this lane: its row's token chunk in its group's
  // codes, or the zero block off the diagonal / past the tokens
  const bool diag = arow_g == gq && arow_t < nt;
  const char* xsrc = smem + ((size_t)arow_t * xs + sq * CPL) * 2;
  for (int gs0 = 0; gs0 < total; gs0 += R) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int gs = gs0 + j;
      load(ring[(j + D) % R], min(gs + D, total - 1));
      const Ring& cur = ring[j];
      const bool live = gs < total;
      const int bi = gs / ssk, ls = gs - bi * ssk, ss = s0 + ls;
      const int g = ss * GG + gq;
      const bool on = diag && live;
      const char* xp = on ? xsrc + (size_t)(64 * g) * 2 : zero_blk;
      const int xstep = on ? 16 : 0;
      // all x fragments of the step are read before the first MFMA, so
      // the MFMA chain waits on LDS once per step, not once per MFMA
      bf16x8_t xa[NMF];
#pragma unroll
      for (int i = 0; i < NMF; ++i)
        xa[i] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(xp + xstep * i));
      // X of this lane's output rows: group (4q+r)/TT, tokens (4q+r)%TT
      const int og = ss * GG + (4 * q) / TT;
      f32x4_t X = *reinterpret_cast<const f32x4_t*>(Xl + og * TT + (4 * q) % TT);
      if (!live) X = zero;
      MLXR_SCHED_BARRIER();
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        f32x4_t P = zero;
#pragma unroll
        for (int i = 0; i < NMF; ++i) {
          u32x4_t u;
          if constexpr (BITS == 4) {
            u = unpack4(cur.w[m][i / 4][i % 4], one_v);
          } else {
            const u32x4_t wv = cur.w[m][i / 2];
            u = (i & 1) ? unpack8(wv.z, wv.w) : unpack8(wv.x, wv.y);
          }
          P = mfma16x16x32(xa[i], as_bf16x8(u), P);
        }
        // scale/bias of this lane's output group og (channel n)
        const int si = ((live ? bi : 0) * 16 + n) * groups + min(og, groups - 1);
        const uint32_t sc_bits = sbl[(m * 2) * sbn + si];
        const uint32_t bi_bits = sbl[(m * 2 + 1) * sbn + si];
        float sc, cb;
        group_terms<BITS>(sc_bits, bi_bits, sc, cb);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[m][r] = __builtin_fmaf(sc, P[r], __builtin_fmaf(cb, X[r], acc[m][r]));
      }
      if constexpr (NB > 1) {
        const bool last = live && ls == ssk - 1 && bi < NB - 1;
#pragma unroll
        for (int b = 0; b < NB - 1; ++b) {
          const bool fin = last && bi == b;
#pragma unroll
          for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) done[b][m][r] = fin ? acc[m][r] : done[b][m][r];
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][r] = last ? 0.0f : acc[m][r];
      }
    }
  }
  // Each token's GG group partials sit on lanes 16*(TT/4) apart: a
  // butterfly over those lanes sums them, and lanes q < TT/4 write tokens
  // 4q..4q+3 of channel n.  With K-slices the KS waves' sums of a block
  // meet in LDS (after the x region is no longer read) and the slice-0
  // wave adds them in slice order.
  f32x4_t* red = reinterpret_cast<f32x4_t*>(
      sb_base + (((size_t)(lthreads >> 6) * NA * nb * 16 * groups * 2 + 15) & ~size_t(15)));
  if constexpr (KS > 1) {
#pragma unroll
    for (int bi = 0; bi < NB; ++bi)
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        f32x4_t t = acc[m];
#pragma unroll
        for (int b = 0; b < NB - 1; ++b) t = bi == b ? done[b][m] : t;
        red[((wave_id * NB + bi) * NM + m) * 64 + lane] = t;
      }
    __syncthreads();
    if (kq != 0) return;
  }
#pragma unroll
  for (int bi = 0; bi < NB; ++bi) {
    f32x4_t tot[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      tot[m] = acc[m];
#pragma unroll
      for (int b = 0; b < NB - 1; ++b) tot[m] = bi == b ? done[b][m] : tot[m];
      if constexpr (KS > 1) {
#pragma unroll
        for (int k = 1; k < KS; ++k)
          tot[m] += red[(((wave_id + k) * NB + bi) * NM + m) * 64 + lane];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (TT == 4) tot[m][r] += __shfl_xor(tot[m][r], 16, 64);
        tot[m][r] += __shfl_xor(tot[m][r], 32, 64);
      }
    }
    if (q < TT / 4) {
      const int ch = ch0 + bi * 16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 4 * q + r;
        if (t < nt) {
          const int slot = row0 + t;
          if constexpr (GATED) {
            a.out[(int64_t)slot * a.out_ld + ch] =
                gated_act_bf16(a.act, bf16_round(tot[0][r]), bf16_round(tot[1][r]));
          } else {
            const int64_t orow = a.out_by_flat ? rec[4 + t] : slot;
            if (yl)  // the single-token down + combine: rows stay in LDS
              yl[(orow + yrow_off) * 16 + n] = f32_to_bf16(tot[0][r]);
            else
              a.out[orow * a.out_ld + ch] = f32_to_bf16(tot[0][r]);
          }
        }
      }
    }
  }
}

// Launch shape of the streaming kernel: 16-channel blocks per wave (nb),
// K-slices (ks), channel tiles per item and the LDS of one workgroup.
struct StreamShape {
  int nb, ks, tiles_n;
  size_t lds;
};
// The wide items' x stages: whole up to kWideWhole inputs, else kWideSlice at
// a time.
constexpr int kWideWhole = 1536, kWideSlice = 1024;
// The streaming kernel over wide items (qgemm_wide.hip); arguments as
// launch_qgemm's.
hipError_t launch_stream_wide(const QGemmArgs& a, const QGemmArgs& b, int64_t max_items,
                              int64_t items2, int64_t shared_rows, const char* profile,
                              hipStream_t s);

}  // namespace mlxr_moe
