// Grouped expert GEMM of dense bf16 weights (gather_mm) for many rows per
// expert (prefill): an LDS-tiled bf16 MFMA GEMM; and the choice of tiles for
// every width (quantised weights: prefill_reg.hip, prefill_tall.hip).
//
// Same operation as the decode kernels, with bf16 weights
// (SwitchLinear::apply, crates/mlxr-lm/src/nn/switch.rs:84-93):
//   out[p, n] = sum_k x[row(p), k] * w[e, n, k]
// over the sorted slots p of expert e, whose rows come in M-tiles (the
// dispatch lists them).
//
// Workgroup: kWM x kWN waves (2 x 4, or 2 x 2 in the narrow form); tile
// kBM rows x kBN = 64 kWN columns (the gated kernel's columns are gate
// channels then the same up channels, so each wave holds matching gate and
// up sums for the SwiGLU epilogue).  Tile heights 256 and 128 rows
// (prefill_tile.inc is built once per shape; shorter tiles are
// prefill_reg.hip's): each wave 128 x 64 or 64 x 64 outputs as blocks of
// v_mfma_f32_32x32x16_bf16 (K = 16 per instruction, four per group); waves
// whose rows lie past the expert's last row skip their MFMAs.  Global loads
// are raw buffer loads with the K step in the scalar offset: no per-step
// address arithmetic.
// K advances one group (64) per step.  Register buffers hold the loads of the
// next groups in flight, and LDS stages hold tiles: while the waves multiply
// stage s, the group loaded a step earlier is staged, interleaved with the
// MFMAs.  One barrier per step.
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

// The tile shapes.  prefill_tile_rows picks one per call, and the dispatch
// cuts the M-tiles to match.
namespace tile256 {
#define MLXR_PF_TILE_ROWS 256
#define MLXR_PF_MBLOCKS 4
#define MLXR_PF_WAVES_N 4
#include "prefill_tile.inc"
#undef MLXR_PF_TILE_ROWS
#undef MLXR_PF_MBLOCKS
#undef MLXR_PF_WAVES_N
}  // namespace tile256
// 128 rows of dense bf16 weights: 128 columns, 4 waves of 64 x 64, two stages
// in 64 KB of LDS, so that two workgroups share a CU and one's barrier waits
// and staging overlap the other's MFMAs (c8 T=2048 gate/up 237 us with 256
// columns and 8 waves, 232 so).
namespace tile128n {
#define MLXR_PF_TILE_ROWS 128
#define MLXR_PF_MBLOCKS 2
#define MLXR_PF_WAVES_N 2
#include "prefill_tile.inc"
#undef MLXR_PF_TILE_ROWS
#undef MLXR_PF_MBLOCKS
#undef MLXR_PF_WAVES_N
}  // namespace tile128n
}  // namespace

int prefill_tile_rows(int64_t rows, int64_t experts, int bits) {
  const int64_t e = experts > 0 ? experts : 1;
  if (bits != 16) return rows >= kPrefillMinTileRows * e ? 128 : kPrefillMinTileRows;
  if (rows >= (int64_t)MLXR_PREFILL_TALL_ROWS * e) return tile256::kBM;
  if (rows >= (int64_t)MLXR_PREFILL_DENSE_ROWS * e) return tile128n::kBM;
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
  if (tile_rows == kPrefillMinTileRows)
    return launch_qgemm_prefill_reg(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  if (a.bits != 16)
    return launch_qgemm_prefill_tall(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  if (tile_rows == tile256::kBM)
    return tile256::launch(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  if (tile_rows == tile128n::kBM)
    return tile128n::launch(a, x_rows, max_tiles, s, profile, shared, shared_rows);
  return hipErrorInvalidValue;
}

}  // namespace mlxr_moe
