// Direct-to-LDS tiles of gemm_dma.h for e4m3 operands.
#include "gemm_dma.h"

namespace lc0mi {

namespace {
template <int BM, int BN, int WAVES_M, int WAVES_N, int BKB = 128, int NSTAGES = 2, bool ALONE = false>
void LaunchGemmDmaF8Tile(const GemmF8Args& args, hipStream_t stream) {
  GemmF8Args a = args;
  dim3 grid((a.M + BM - 1) / BM, (a.N + BN - 1) / BN + (a.N2 + BN - 1) / BN);
  a.tile_order = PickTileOrder(a.M, 0, grid);
  const dim3 block(WAVES_M * WAVES_N * 64);
  if constexpr (BM == 256) {
    const int stores = OutputStores(a.out_stores, a.M, a.N, 1, a.out_f8 ? 1 : 2);
    auto launch = [&](auto stores_tag) {
      constexpr int S = decltype(stores_tag)::value;
      if (a.out_f8) {
        hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BKB, WAVES_M, WAVES_N, GemmF8Args, uint8_t, S>), grid, block, 0,
                           stream, a);
      } else {
        hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BKB, WAVES_M, WAVES_N, GemmF8Args, half_t, S>), grid, block, 0,
                           stream, a);
      }
    };
    if (stores == 1) return launch(std::integral_constant<int, 1>{});
    if (stores == 2) return launch(std::integral_constant<int, 2>{});
  }
  if constexpr (BM < 256) {
    if (a.N2 > 0) {
      hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BKB, WAVES_M, WAVES_N, GemmF8Args, half_t, 0, 0, NSTAGES,
                                          half_t, ALONE, true>), grid, block, 0, stream, a);
      return;
    }
  }
  if (a.out_f8) {
    hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BKB, WAVES_M, WAVES_N, GemmF8Args, uint8_t, 0, 0, NSTAGES,
                                        half_t, ALONE>), grid, block, 0, stream, a);
  } else {
    hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BKB, WAVES_M, WAVES_N, GemmF8Args, half_t, 0, 0, NSTAGES,
                                        half_t, ALONE>), grid, block, 0, stream, a);
  }
}

// Stage count by the launch's workgroup count, as LaunchGemmDmaStaged does for fp16 operands.
template <int BM, int BN, int WAVES_M, int WAVES_N>
void LaunchGemmDmaF8Staged(const GemmF8Args& a, hipStream_t stream) {
  constexpr int kStage = (BM + BN) * 128, kCus = 256;
  constexpr int kFour = WorkgroupsPerCu(4, kStage), kThree = WorkgroupsPerCu(3, kStage);
  constexpr bool kAlone = BM * BN <= 128 * 64;
  const long long wgs = (long long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN + (a.N2 + BN - 1) / BN);
  if constexpr (kAlone) {
    if (wgs <= kCus) return LaunchGemmDmaF8Tile<BM, BN, WAVES_M, WAVES_N, 128, 4, true>(a, stream);
  }
  if constexpr (kFour > (kAlone ? 1 : 0)) {
    if (wgs <= kCus * kFour) return LaunchGemmDmaF8Tile<BM, BN, WAVES_M, WAVES_N, 128, 4>(a, stream);
  }
  if constexpr (kThree > kFour) {
    if (wgs <= kCus * kThree) return LaunchGemmDmaF8Tile<BM, BN, WAVES_M, WAVES_N, 128, 3>(a, stream);
  }
  LaunchGemmDmaF8Tile<BM, BN, WAVES_M, WAVES_N, 128, 2>(a, stream);
}
}  // namespace

void LaunchGemmDmaF8(GemmVariant v, const GemmF8Args& a, hipStream_t stream) {
  switch (v) {
    case kDma256x256: LaunchGemmDmaF8Tile<256, 256, 2, 4>(a, stream); break;
    case kDma256x192: LaunchGemmDmaF8Tile<256, 192, 4, 2>(a, stream); break;
    case kDma256x128: LaunchGemmDmaF8Tile<256, 128, 4, 2>(a, stream); break;
    case kDma128x64: LaunchGemmDmaF8Staged<128, 64, 2, 2>(a, stream); break;
    case kDma64x64: LaunchGemmDmaF8Staged<64, 64, 2, 2>(a, stream); break;
    default: LaunchGemmDmaF8Staged<128, 128, 2, 2>(a, stream); break;
  }
}

}  // namespace lc0mi
