// The streaming decode GEMM over work items of up to 16 rows (work_rows_for).
//
// A translation unit, and so a code object, of its own: with these kernels in
// qgemm.hip's the down projection and the launch after it ran slower at a few
// tokens, by the same instructions (layer tail of c6 at T = 7 from a graph:
// 59.9 us, 59.3 without them).
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "qgemm_stream.hpp"

namespace mlxr_moe {
namespace {

// The wide form: an item of 9 to 16 rows (of an expert of more than 8), so
// that an expert's weights are read once per 16 rows where the 8-token form
// reads them per 8.  A wave loads the same bytes per super-step (two groups of
// its 16 channels) as there; the MFMA's 16 A rows are 16 tokens, so all lanes
// must hold one group's codes: v_permlane32_swap_b32 turns two words of a
// lane, of group A on lanes 0-31 and B on 32-63, into a word of A and one of B
// on every lane.  Lane quarter q then supplies codes 16 i + 32 (q & 1) +
// 8 (q >> 1) .. + 7 of the group to MFMA i of two, and receives tokens
// 4 q .. 4 q + 3 of channel l % 16: no sums cross lanes.  The sums are those
// of the 8-token form, bit for bit: an MFMA adds its lane quarters' products
// quarter by quarter, so MFMA i here is MFMAs 2 i and 2 i + 1 there, and the
// groups A and the groups B are summed apart (acc[0], acc[1]) and joined at a
// block's end, as its two halves of the wave are.  x is staged whole up
// to kWideWhole inputs, else kWideSlice at a time, NB = 1 then: three
// workgroups share a CU up to K = 2048 (above, the 8-token form, which stages
// all of K, and the scales leave room for two at K = 3072 and for one at 4096).
// The gated 4-bit kernel keeps one register pair in scratch across its 4-token
// loop; no loop reads it.
// 12 rows an expert of c7 (T = 190): gate/up 83 us in 8-row items, 72 in these,
// down 59 and 44.  Steps of c2 at 8, 10 and 14 rows an expert (T = 128, 160,
// 224): 128, 151, 186 us and 117, 130, 154; c5 at 6 (T = 200) 893 and 810.
template <int BITS, bool GATED, int NB>
__device__ __forceinline__ void stream16_body(const QGemmArgs& a, int4 wk, int tile,
                                              char* smem) {
  constexpr int TT = 16, D = 3, R = D + 1;
  constexpr int NM = GATED ? 2 : 1, NA = 2 * NM;
  constexpr int NL = BITS / 4;     // 16-byte loads per lane and super-step
  constexpr int WPG = 2 * BITS;    // packed words per row and group
  const int e = wk.x, row0 = wk.y, nt = min(wk.z, TT);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, q = lane >> 4;
  const int K = a.K, groups = K >> 6, ssteps = groups >> 1;
  const int KS = K <= kWideWhole ? K : kWideSlice;  // inputs of x staged at once
  const int slices = K / KS, sps = ssteps / slices;  // super-steps per slice
  const int total = NB * ssteps;
  // LDS as stream_body: x [16][KS + 8], X [KS / 64][16], the waves' scales
  const int xs = KS + 8;
  uint16_t* xl = reinterpret_cast<uint16_t*>(smem);
  float* Xl = reinterpret_cast<float*>(smem + (size_t)TT * xs * 2);
  char* sb_base = smem + (size_t)TT * xs * 2 + (size_t)(KS >> 6) * TT * 4;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const u32x4_t zq = {0u, 0u, 0u, 0u};
  const int ch0 = ((tile * MLXR_STREAM_WAVES + wave) * NB) * 16 + n;
  const int64_t wrow0 = (int64_t)e * a.e_rows + ch0;

  struct Ring {
    u32x4_t w[NM][NL];
  };
  const uint32_t* wb[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const QWeights& W = m == 0 ? a.w0 : a.w1;
    wb[m] = W.w + (wrow0 * groups + (q >> 1)) * WPG + (q & 1) * BITS;
  }
  const int64_t blk_rows = (int64_t)16 * groups;
  auto load = [&](Ring& r, int gs) {
    const int bi = gs / ssteps, ss = gs - bi * ssteps;
    const int64_t go = bi * blk_rows + 2 * ss;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const u32x4_t* wp = reinterpret_cast<const u32x4_t*>(wb[m] + go * WPG);
#pragma unroll
      for (int i = 0; i < NL; ++i) r.w[m][i] = wp[i];
    }
  };
  // x: thread -> 16-byte chunks tid % 128, + 128, .. of rows 8 (tid / 128) + t
  const int k8 = tid & 127, rh = 8 * (tid >> 7), rows_h = nt - rh;
  int64_t xr[8];
  {
    int32_t fl[8], rm[8];
    if (!a.x_by_slot) {
#pragma unroll
      for (int t = 0; t < 8; ++t) fl[t] = a.sorted[row0 + min(rh + t, nt - 1)];
    }
    if (!a.x_by_slot && a.row_map) {
#pragma unroll
      for (int t = 0; t < 8; ++t) rm[t] = a.row_map[fl[t]];
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      int64_t r = 0;
      if (t < rows_h)
        r = a.x_by_slot ? row0 + rh + t : (a.row_map ? rm[t] : fl[t] / a.row_div);
      xr[t] = r;
    }
  }
  const int per_row = KS >> 3;
  auto load_x = [&](int k, u32x4_t (&v)[8]) {  // chunk k of all of K's
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      v[t] = zq;
      if (t < rows_h) v[t] = *reinterpret_cast<const u32x4_t*>(a.x + xr[t] * a.x_ld + 8 * k);
    }
  };
  auto stage_x = [&](int kl, const u32x4_t (&v)[8]) {  // ... chunk kl of the slice
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      float sx = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sx += __uint_as_float(v[t][j] << 16) + __uint_as_float(v[t][j] & 0xffff0000u);
      sx += __shfl_xor(sx, 1, 64);
      sx += __shfl_xor(sx, 2, 64);
      sx += __shfl_xor(sx, 4, 64);
      if ((kl & 7) == 0) Xl[(kl >> 3) * TT + rh + t] = sx;
      u32x4_t w = v[t];
      if constexpr (BITS == 4) w = perm4(w);
      *reinterpret_cast<u32x4_t*>(xl + (size_t)(rh + t) * xs + 8 * kl) = w;
    }
  };
  // issue order as stream_body: x, scales and biases, weights
  u32x4_t xv[8];
  load_x(min(k8, per_row - 1), xv);
  MLXR_SCHED_BARRIER();
  const int sbn = NB * 16 * groups, sbv = sbn >> 3;
  uint16_t* sbl = reinterpret_cast<uint16_t*>(sb_base) + (size_t)wave * NA * sbn;
  const uint16_t* sbsrc[NA];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const QWeights& W = m == 0 ? a.w0 : a.w1;
    sbsrc[2 * m] = W.scales + (wrow0 - n) * groups;
    sbsrc[2 * m + 1] = W.biases + (wrow0 - n) * groups;
  }
  u32x4_t sv[NA];
  const int sl = min(lane, sbv - 1);
#pragma unroll
  for (int i = 0; i < NA; ++i) sv[i] = *reinterpret_cast<const u32x4_t*>(sbsrc[i] + 8 * sl);
  MLXR_SCHED_BARRIER();
  Ring ring[R];
#pragma unroll
  for (int j = 0; j < D; ++j) load(ring[j], min(j, total - 1));
  MLXR_SCHED_BARRIER();
  if (k8 < per_row) stage_x(k8, xv);  // per_row is a multiple of 8: whole octets
  for (int c8 = k8 + 128; c8 < per_row; c8 += 128) {
    u32x4_t v[8];
    load_x(c8, v);
    stage_x(c8, v);
  }
  __syncthreads();
  if (lane < sbv) {
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

  constexpr int ND = NB > 1 ? NB - 1 : 1;
  f32x4_t acc[2][NM], done[ND][NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    acc[0][m] = acc[1][m] = zero;
#pragma unroll
    for (int b = 0; b < ND; ++b) done[b][m] = zero;
  }
  const uint32_t one_v = 0x3F803F80u;
  const char* xsrc = smem + ((size_t)n * xs + 32 * (q & 1) + 8 * (q >> 1)) * 2;
  for (int s = 0; s < slices; ++s) {
    if (s > 0) {
      // the next slice of x (kWideSlice inputs: one chunk per thread)
      u32x4_t v[8];
      load_x(s * per_row + k8, v);
      __syncthreads();
      stage_x(k8, v);
      __syncthreads();
    }
    const int end = slices == 1 ? total : (s + 1) * sps;
    for (int gs0 = s * sps; gs0 < end; gs0 += R) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int gs = gs0 + j;
        load(ring[(j + D) % R], min(gs + D, total - 1));
        MLXR_SCHED_BARRIER();
        if (gs >= end) continue;  // (uniform; the loads above run on)
        const int bi = gs / ssteps, ss = gs - bi * ssteps;
        uint32_t w[NM][4 * NL];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
#pragma unroll
          for (int i = 0; i < 4 * NL; ++i) w[m][i] = ring[j].w[m][i / 4][i % 4];
          // pairs of words (4-bit) or of word pairs (8-bit)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < NL; ++h) {
              uint32_t &lo = w[m][2 * NL * i + h], &hi = w[m][2 * NL * i + NL + h];
              const auto r = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
              lo = r[0];
              hi = r[1];
            }
        }
#pragma unroll
        for (int g2 = 0; g2 < 2; ++g2) {
          const int g = 2 * ss + g2, gl = g - s * (KS >> 6);
          bf16x8_t xa[2];
#pragma unroll
          for (int i = 0; i < 2; ++i)
            xa[i] = as_bf16x8(
                *reinterpret_cast<const u32x4_t*>(xsrc + (size_t)(64 * gl + 16 * i) * 2));
          const f32x4_t X = *reinterpret_cast<const f32x4_t*>(Xl + gl * TT + 4 * q);
#pragma unroll
          for (int m = 0; m < NM; ++m) {
            f32x4_t P = zero;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const int b = 2 * NL * i + NL * g2;
              u32x4_t u;
              if constexpr (BITS == 4)
                u = unpack4(w[m][b], one_v);
              else
                u = unpack8(w[m][b], w[m][b + NL - 1]);
              P = mfma16x16x32(xa[i], as_bf16x8(u), P);
            }
            const int si = (bi * 16 + n) * groups + g;
            float sc, cb;
            group_terms<BITS>(sbl[(m * 2) * sbn + si], sbl[(m * 2 + 1) * sbn + si], sc, cb);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              acc[g2][m][r] =
                  __builtin_fmaf(sc, P[r], __builtin_fmaf(cb, X[r], acc[g2][m][r]));
          }
        }
        if constexpr (NB > 1) {
          const bool last = ss == ssteps - 1 && bi < NB - 1;
#pragma unroll
          for (int b = 0; b < NB - 1; ++b) {
            const bool fin = last && bi == b;
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                done[b][m][r] = fin ? acc[0][m][r] + acc[1][m][r] : done[b][m][r];
          }
#pragma unroll
          for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              acc[0][m][r] = last ? 0.0f : acc[0][m][r];
              acc[1][m][r] = last ? 0.0f : acc[1][m][r];
            }
        }
      }
    }
  }
#pragma unroll
  for (int bi = 0; bi < NB; ++bi) {
    f32x4_t tot[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      tot[m] = acc[0][m] + acc[1][m];
#pragma unroll
      for (int b = 0; b < NB - 1; ++b) tot[m] = bi == b ? done[b][m] : tot[m];
    }
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
          const int64_t orow = a.out_by_flat ? a.sorted[slot] : slot;
          a.out[orow * a.out_ld + ch] = f32_to_bf16(tot[0][r]);
        }
      }
    }
  }
}

// The same over wide items (16 rows): an item of an expert of more than 8 rows
// runs in the wide form.
template <int BITS, bool GATED, int D, int D8, int NB>
__global__ __launch_bounds__(64 * MLXR_STREAM_WAVES, 3) void qgemm_stream_wide_kernel(
    QGemmArgs a, int tiles_n, QGemmArgs a2, int units1, int items1, int rows2) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  Unit u;
  if (!decode_unit<kWorkRowsWide>(a, tiles_n, units1, items1, rows2, u)) return;
  const QGemmArgs& A = u.shared ? a2 : a;
  if (u.wk.w <= kStreamTT4Rows)
    stream_body<BITS, GATED, 4, D, NB, 1>(A, u.rec, u.wk, u.fr0, u.fr1, u.tile, smem,
                                          threadIdx.x, blockDim.x, nullptr, 0);
  else if (u.wk.w <= kWorkRows)
    stream_body<BITS, GATED, 8, D8, NB, 1>(A, u.rec, u.wk, u.fr0, u.fr1, u.tile, smem,
                                           threadIdx.x, blockDim.x, nullptr, 0);
  else
    stream16_body<BITS, GATED, NB>(A, u.wk, u.tile, smem);
}

// ... of the wide items' kernel: no K-slices (work_rows_for); LDS for the
// larger of the 8- and the 16-token form.
StreamShape stream_wide_shape(const QGemmArgs& a, int64_t all_items) {
  constexpr int kWaves = MLXR_STREAM_WAVES;
  const int groups = a.K / 64;
  const int64_t per_tile = a.N / (16 * kWaves);
  int nb = 1;
  if (!a.gated && a.K <= kWideWhole && per_tile % 2 == 0 &&
      all_items * (per_tile / 2) >= kStreamSlots)
    nb = 2;
  const size_t sb_lds = (size_t)kWaves * (a.gated ? 2 : 1) * 2 * nb * 16 * groups * 2;
  const size_t ks = a.K <= kWideWhole ? a.K : kWideSlice;
  const size_t lds8 =
      ((size_t)8 * (a.K + 8) * 2 + 16 + (size_t)groups * 8 * 4 + 15) & ~size_t(15);
  const size_t lds16 = (size_t)16 * (ks + 8) * 2 + ks / 64 * 16 * 4;
  return StreamShape{nb, 1, (int)(per_tile / nb),
                     std::max(lds8, lds16) + ((sb_lds + 15) & ~size_t(15))};
}

}  // namespace

hipError_t launch_stream_wide(const QGemmArgs& a, const QGemmArgs& b, int64_t max_items,
                              int64_t items2, int64_t shared_rows, const char* profile,
                              hipStream_t s) {
  constexpr int kWaves = MLXR_STREAM_WAVES;
  const StreamShape sh = stream_wide_shape(a, max_items + items2);
  const int items1 = (int)max_items, units1 = (int)(max_items * sh.tiles_n);
  const dim3 grid((unsigned)(units1 + items2 * sh.tiles_n));
  ProfileScope prof(profile, s);
#define MLXR_QW(B, G, D, D8, NB)                                    \
  qgemm_stream_wide_kernel<B, G, D, D8, NB>                         \
      <<<grid, 64 * kWaves, sh.lds, s>>>(a, sh.tiles_n, b, units1, items1, (int)shared_rows)
  if (a.bits == 4) {
    if (a.gated)
      MLXR_QW(4, true, MLXR_STREAM_DEPTH4G, MLXR_STREAM_DEPTH4G_TT8, 1);
    else if (sh.nb == 2)
      MLXR_QW(4, false, MLXR_STREAM_DEPTH4, MLXR_STREAM_DEPTH4_TT8, 2);
    else
      MLXR_QW(4, false, MLXR_STREAM_DEPTH4, MLXR_STREAM_DEPTH4_TT8, 1);
  } else {
    if (a.gated)
      MLXR_QW(8, true, MLXR_STREAM_DEPTH8G, MLXR_STREAM_DEPTH8G_TT8, 1);
    else if (sh.nb == 2)
      MLXR_QW(8, false, MLXR_STREAM_DEPTH8, MLXR_STREAM_DEPTH8_TT8, 2);
    else
      MLXR_QW(8, false, MLXR_STREAM_DEPTH8, MLXR_STREAM_DEPTH8_TT8, 1);
  }
#undef MLXR_QW
  return hipGetLastError();
}

}  // namespace mlxr_moe
