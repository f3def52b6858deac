// Kernel variants of the dense layers and the launchers between their source files (host side only).
#pragma once

#include "kernels.h"

namespace lc0mi {

// (the numbers are those of SetGemmVariantOverride; 8 is no kernel: the answer of a choice that finds none)
enum GemmVariant { kDma256x256, kDma256x192, kDma256x128, kTile128, kTile64, kDma128x128, kRowPanel, kDma128x64, kNoVariant,
                   kDma128x32, kDma64x64, kResident };

// Direct-to-LDS tiles (gemm_dma_half.hip, gemm_dma_bf16.hip, gemm_dma_f8.hip). The folded layer-norm fields of
// GemmArgs are served by the half instances only.
void LaunchGemmDmaHalf(GemmVariant v, const GemmArgs& a, hipStream_t stream);
void LaunchGemmDmaBf16(GemmVariant v, const GemmArgs& a, hipStream_t stream);
void LaunchGemmDmaF8(GemmVariant v, const GemmF8Args& a, hipStream_t stream);
// As a value of GemmArgs::out_stores that no longer depends on the size (for the parts of a product).
int ResolvedOutStores(const GemmArgs& a);

// The order of a launch's tiles. Workgroups go to the eight XCDs in turn, and each XCD's L2 fetches every operand row that one of its
// tiles reads. In the order of the grid an XCD has tiles of all rows and of all columns, unless the row tiles are a multiple of
// eight. Neighbouring row tiles per XCD cut the activations fetched to an eighth: from 2048 rows (us of a 15x1024 pass
// with the tiles chosen now, fp16 36 positions 1733 -> 1756, 77 dense 2740 -> 2645, 150 3913 -> 3815, 300 7661 -> 7032, 1000 21300 -> 20768; e4m3 77
// 2091 -> 1987, 300 5495 -> 5044, 350 7019 -> 6140). With fewer rows the weights, which come
// from memory, are the larger part: in halves neighbouring column tiles up to 1024 rows (1 position 779 -> 761, 4 968 -> 947, 16 1204 ->
// 1196, but 20 1386 -> 1395), in e4m3, with half the bytes, for row panels only (5 positions on tiles 826 -> 841, 16 928 -> 939).
inline TileOrder PickTileOrder(int M, int columns_max_rows, const dim3& grid) {
  TileOrder o;
  const unsigned tiles = grid.x * grid.y;
  o.columns = M <= columns_max_rows;
  const unsigned d = o.columns ? grid.x : grid.y;
  if (grid.z != 1 || tiles < 16 || tiles > 65536 || (!o.columns && (M < 2048 || grid.x % 8 == 0))) return o;
  if (d > 1) o.inverse = 0xFFFFFFFFu / d + 1;   // (exact division while tiles * d < 2^32)
  return o;
}

// Row panels (gemm_rowpanel.hip): panels of 16 rt x 16 ct outputs, and how many of them cover a problem.
struct RowPanelShape { int rt, ct; };
constexpr RowPanelShape kRowPanelShapes[] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {4, 2}};
constexpr long long kRowPanelWorkgroups = 256;   // one per CU
inline long long RowPanelWorkgroups(int M, int N, int batch, const RowPanelShape& c) {
  return (long long)((M + 16 * c.rt - 1) / (16 * c.rt)) * ((N + 16 * c.ct - 1) / (16 * c.ct)) * batch;
}
void LaunchGemmRowPanel(const GemmArgs& a, hipStream_t stream);
void LaunchGemmF8RowPanel(const GemmF8Args& a, hipStream_t stream);

// Batched products with the weights of one product in the LDS of a CU (gemm_resident.hip). Workgroups per product; 0 where
// the kernel does not serve the arguments: K = N = 256, 16-bit output without bias and activation, whole 16-byte vectors.
inline int GemmResidentWorkgroups(const GemmArgs& a) {
  const bool vectors = a.lda % 8 == 0 && a.ldw % 8 == 0 && a.ldc % 8 == 0 && a.strideA % 8 == 0 && a.strideW % 8 == 0 &&
                       a.strideC % 8 == 0;
  if (a.K != 256 || a.N != 256 || a.M < 1 || a.batch < 1 || a.batch > 256 || a.out_f32 || a.split_k != 1 ||
      a.bias != nullptr || a.act != 3 || a.skip != nullptr || a.row_stats != nullptr || !vectors) {
    return 0;
  }
  const int blocks = (a.M + 127) / 128, share = 256 / a.batch;
  return blocks < share ? blocks : share;
}
void LaunchGemmResident(const GemmArgs& a, hipStream_t stream);

}  // namespace lc0mi
