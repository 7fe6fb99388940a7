// Grouped quantised expert GEMM for many rows per expert (prefill): an
// LDS-tiled bf16 MFMA GEMM that dequantises each weight tile once per
// workgroup.  The same kernel runs dense bf16 expert weights (gather_mm,
// bits = 16: the weight tile is staged as it is).
//
// Same operation as the decode kernels (gather_qmm with transpose = true,
// crates/mlxr/src/ops/quantization.rs:171-221, as called by
// QuantizedSwitchLinear::apply, crates/mlxr-lm/src/nn/switch.rs:148-167):
//   out[p, n] = sum_k x[row(p), k] * bf16(code[e, n, k] * scale + bias)
// over the sorted slots p of expert e.  Here the rows of an expert come in
// M-tiles (the dispatch lists them), and the work is compute-bound, so the
// weights are dequantised -- exactly the oracle's
// bf16(fmaf(code, scale, bias)) -- into LDS, where every wave of the
// workgroup reuses them.
//
// Workgroup: kWM x kWN waves (2 x 4, or 2 x 2 in the narrow form); tile
// kBM rows x kBN = 64 kWN columns (the gated kernel's columns are gate
// channels then the same up channels, so each wave holds matching gate and
// up sums for the SwiGLU epilogue).  Tile heights 256 and, for dense weights,
// 128 rows (prefill_tile.inc is built once per shape; 64-row tiles are
// prefill_reg.hip's): each wave 128 x 64 or 64 x 64 outputs as blocks of
// v_mfma_f32_32x32x16_bf16 (K = 16 per instruction, four per group).  A tall
// tile spreads the dequantisation (the VALU cost, about two instructions per
// weight) over more rows; waves whose rows lie past the expert's last row
// skip their MFMAs.  Global loads are raw buffer loads with the K step in the
// scalar offset: no per-step address arithmetic.
// K advances one quantisation group (64) per step.  Register buffers hold
// the loads of the next groups in flight, and LDS stages hold dequantised
// tiles: while the waves multiply stage s, the group loaded a step earlier
// is dequantised into the next stage, interleaved with the MFMAs.  One
// barrier per step.  When K has 16 or more groups, each tile's scales and
// biases are copied to LDS once (coalesced) instead of loaded every step:
// a step's per-column scale loads put a different cache line on every lane.
//
// LDS rows are 64 bf16 (128 bytes) with the eight 16-byte chunks of row r
// stored at chunk ^ ((r >> 1) & 7), which keeps the 16-byte operand reads of
// a wave on distinct banks.  The epilogue goes through LDS so that every
// output store is 16 bytes.
#include "common.hpp"
#include "kernels.hpp"
#include "prefill_dev.hpp"

namespace mlxr_moe {
namespace {

// The tile shapes.  Tall tiles (256 x 256, waves of 128 x 64) dequantise
// each weight group for more rows and read fewer LDS bytes per MFMA.
// prefill_tile_rows picks one per call, and the dispatch cuts the M-tiles to
// match.
namespace tile256 {
#define MLXR_PF_TILE_ROWS 256
#define MLXR_PF_MBLOCKS 4
#define MLXR_PF_WAVES_N 4
#define MLXR_PF_REGBUF 2
#include "prefill_tile.inc"
#undef MLXR_PF_TILE_ROWS
#undef MLXR_PF_MBLOCKS
#undef MLXR_PF_WAVES_N
#undef MLXR_PF_REGBUF
}  // namespace tile256
// 128 rows of dense bf16 weights: 128 columns, 4 waves of 64 x 64, two stages
// in 64 KB of LDS, so that two workgroups share a CU and one's barrier waits
// and staging overlap the other's MFMAs (c8 T=2048 gate/up 237 us with 256
// columns and 8 waves, 232 so).  Quantised weights run the 64-row tiles of
// prefill_reg.hip up to the 256-row ones.
namespace tile128n {
#define MLXR_PF_TILE_ROWS 128
#define MLXR_PF_MBLOCKS 2
#define MLXR_PF_WAVES_N 2
#define MLXR_PF_REGBUF 2
#define MLXR_PF_STAGES 2
#define MLXR_PF_DENSE_ONLY
#include "prefill_tile.inc"
#undef MLXR_PF_DENSE_ONLY
#undef MLXR_PF_STAGES
#undef MLXR_PF_TILE_ROWS
#undef MLXR_PF_MBLOCKS
#undef MLXR_PF_WAVES_N
#undef MLXR_PF_REGBUF
}  // namespace tile128n
}  // namespace

int prefill_tile_rows(int64_t rows, int64_t experts, int bits) {
  const int64_t e = experts > 0 ? experts : 1;
  if (rows >= (int64_t)MLXR_PREFILL_TALL_ROWS * e) return tile256::kBM;
  if (bits == 16 && rows >= (int64_t)MLXR_PREFILL_DENSE_ROWS * e) return tile128n::kBM;
  return kPrefillMinTileRows;
}

bool prefill_supported(const QGemmArgs& a, int64_t x_rows) {
  // buffer offsets are 32-bit: x, and one expert's weights, under 2 GB
  // outputs leave as 16-byte runs of a row
  const bool out16 = (reinterpret_cast<uintptr_t>(a.out) & 15) == 0 && a.out_ld % 8 == 0;
  return (a.bits == 4 || a.bits == 8 || a.bits == 16) && a.K % 64 == 0 && a.N % 64 == 0 &&
         a.sorted != nullptr && out16 && a.row_div >= 1 && a.row_div <= 65536 &&
         x_rows * a.x_ld * 2 < ((int64_t)1 << 31) &&
         (int64_t)a.N * a.K * a.bits / 8 < ((int64_t)1 << 31);
}

hipError_t launch_qgemm_prefill(const QGemmArgs& a, int64_t x_rows,
                                int tile_rows, int64_t max_tiles,
                                hipStream_t s, const char* profile,
                                const QGemmArgs* shared, int64_t shared_rows) {
  if (tile_rows == tile256::kBM)
    return tile256::launch(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  if (tile_rows == tile128n::kBM && a.bits == 16)
    return tile128n::launch(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  if (tile_rows == kPrefillMinTileRows)
    return launch_qgemm_prefill_reg(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  return hipErrorInvalidValue;
}

}  // namespace mlxr_moe
