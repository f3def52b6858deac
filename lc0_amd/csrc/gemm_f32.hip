// fp32 matrix products of the dense layers (the float configuration): FullyConnectedLayer::Forward1D
// (blas/fully_connected_layer.cc:49-106) and the winograd-domain products of a float residual tower.
#include "kernel_common.h"
#include "row_panel.h"

#include <algorithm>
#include <stdexcept>

namespace lc0mi {

// ---------------------------------------------------------------------------
// C = act(scale * A.W^T + bias) on fp32 operands with v_mfma_f32_16x16x4_f32 (fp32 products, fp32 accumulation).
//
// A wave owns RT x CT accumulator tiles of 16x16 over its share of the reduction and takes its operand rows straight
// from global memory (row_panel.h); the four values of a 16-byte chunk feed four matrix instructions. A workgroup is
// WM x WN such waves by KS shares of the reduction; the KS partial tiles are added through LDS in wave order, so
// results do not depend on timing. ONE_STEP: K <= 64 KS, a wave has one step of 64 values at most and holds one set of
// operands instead of two (56 registers instead of 96: eight waves per SIMD).
//
// What bounds it: a CU multiplies 256 fp32 values per cycle and takes 64 bytes of operands per cycle, so even a 32x32
// tile (0.125 bytes per operation) leaves the matrix cores the slower side and no LDS staging is needed, provided that
// the loads run at that rate. The form before this one (32x32x2 instructions, 32 bytes of 32 rows per load) got a
// quarter of it. us per launch between two events, before -> now: 1280x256x256 12.6 -> 8.4, 1280x1024x256 27.5 -> 17.0,
// 1280x256x1024 25.3 -> 15.8, 32x1858x2048 25.2 -> 11.0, 36 x 128x64x64 10.0 -> 6.8, 36 x 4000x64x64 47.3 -> 26.1,
// 16384x256x1024 180 -> 104.
//
// Rounding: a 16x16 tile adds the 64 products of a step in eight (ONE_STEP) or four sums and pairs those. One sum over a
// wave's whole share rounds a longer chain: relative error of the result in the 2-norm at K = 64 / 256 / 1024, random
// operands, 1.4e-7 / 1.5e-7 / 2.9e-7, now 7.2e-8 / 8.2e-8 / 1.0e-7 (the form before: 7.8e-8 / 1.2e-7 / 2.1e-7). The large
// tile keeps one sum per quarter of K (K = 1024 2.9e-7, the form before 4.1e-7): its registers are used up.
// ---------------------------------------------------------------------------
namespace {
// The workgroup's tile from row m0 and column n0 of product z; part: the waves' sums in LDS, KS times kTileFloats.
template <int RT, int CT, int WM, int WN> constexpr int kTileFloats = 16 * RT * WM * (16 * CT * WN + 4);   // (rows stay 16-byte aligned)
template <int RT, int CT, int WM, int WN, int KS, bool ONE_STEP>
__device__ __forceinline__ void Tile(const GemmArgsF32& p, int m0, int n0, int z, float (*part)[kTileFloats<RT, CT, WM, WN>]) {
  constexpr int ROWS = 16 * RT * WM, COLS = 16 * CT * WN, NT = 64 * WM * WN * KS;
  constexpr int LD = COLS + 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = wave % KS, wn = (wave / KS) % WN, wm = wave / (KS * WN);
  const int r = lane & 15, g = lane >> 4;
  const int M = p.M, N = p.N, K = p.K;
  const char* A = reinterpret_cast<const char*>(p.A + (long long)z * p.strideA + (long long)m0 * p.lda);
  const char* W = reinterpret_cast<const char*>(p.W + (long long)z * p.strideW + (long long)n0 * p.ldw);
  TileOffsets ta[RT], tw[CT];
#pragma unroll
  for (int t = 0; t < RT; t++) ta[t].Set(16 * (wm * RT + t), M - m0, 4 * p.lda);
#pragma unroll
  for (int c = 0; c < CT; c++) tw[c].Set(16 * (wn * CT + c), N - n0, 4 * p.ldw);
  floatx4 acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  auto op = [](const intx4 (&w)[4], const intx4 (&a)[4], floatx4& c) {   // the products of one step
    constexpr int SUMS = RT * CT > 1 ? 1 : ONE_STEP ? 8 : 4;
    floatx4 sum[SUMS] = {};
    if constexpr (SUMS == 1) sum[0] = c;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int l = 0; l < 4; l++) {
        // (four sums: one per chunk, so that neighbouring instructions do not wait for each other)
        const int j = SUMS == 4 ? l : i, e = SUMS == 4 ? i : l, n = SUMS == 4 ? j : (4 * j + e) % SUMS;
        const floatx4 fw = __builtin_bit_cast(floatx4, w[j]), fa = __builtin_bit_cast(floatx4, a[j]);
        sum[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[e], fa[e], sum[n], 0, 0, 0);
      }
#pragma unroll
    for (int n = SUMS / 2; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; i++) sum[i] += sum[i + n];
    if constexpr (SUMS == 1 || ONE_STEP) c = sum[0];
    else c += sum[0];
  };
  // A contiguous share of the steps per wave.
  const int steps = (4 * K + kStepBytes - 1) / kStepBytes;
  if constexpr (ONE_STEP) {   // (K <= 64 KS)
    if (ks < steps) {
      OneStep<RT, CT>(A + ks * kStepBytes, ta, W + ks * kStepBytes, tw, 4 * K - ks * kStepBytes, acc, op);
    }
  } else {
    const int per_wave = (steps + KS - 1) / KS;
    const int s_begin = min(steps, ks * per_wave), s_end = min(steps, s_begin + per_wave);
    PanelProducts<RT, CT>(A, ta, W, tw, 4 * K, s_begin, s_end, acc, op);
  }
  // Accumulator lane (r, g) of tile (t, c): row 16 t + r, columns 16 c + 4 g + e.
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++)
      *reinterpret_cast<floatx4*>(&part[ks][(16 * (wm * RT + t) + r) * LD + 16 * (wn * CT + c) + 4 * g]) = acc[t][c];
  __syncthreads();
  float* C = p.C + (long long)z * p.strideC;
  DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
    for (int i = 0; i < (ROWS * COLS + NT - 1) / NT; i++) {
      const int idx = tid + NT * i;        // consecutive threads along n
      const int row = idx / COLS, col = idx % COLS;
      const int m = m0 + row, n = n0 + col;
      if (row < ROWS && m < M && n < N) {
        float x = part[0][row * LD + col];
#pragma unroll
        for (int w = 1; w < KS; w++) x += part[w][row * LD + col];
        x *= p.scale;
        if (p.bias != nullptr) x += p.bias[n];
        C[(long long)m * p.ldc + n] = act_fn(x);
      }
    }
  });
}

template <int RT, int CT, int WM, int WN, int KS, bool ONE_STEP>
__global__ __launch_bounds__(64 * WM * WN * KS, RT * CT == 1 ? 5 : 1) void gemm_f32_mfma_kernel(GemmArgsF32 p) {
  __shared__ __attribute__((aligned(16))) float part[KS][kTileFloats<RT, CT, WM, WN>];
  Tile<RT, CT, WM, WN, KS, ONE_STEP>(p, blockIdx.x * 16 * RT * WM, blockIdx.y * 16 * CT * WN, blockIdx.z, part);
}

// Up to three independent products in one launch, in 16x16 tiles: the heads of a float network, whose layers are small and whose
// chains of dependent launches take 5 to 10 us a launch whatever is in it. Workgroup first[i] is the first of product i.
struct GroupArgs {
  GemmArgsF32 p[kGemmF32Group];
  int first[kGemmF32Group];
};
template <int KS>
__global__ __launch_bounds__(64 * KS, 5) void gemm_f32_group_kernel(GroupArgs a) {
  __shared__ __attribute__((aligned(16))) float part[KS][kTileFloats<1, 1, 1, 1>];
  int which = 0;
#pragma unroll
  for (int i = 1; i < kGemmF32Group; i++) which = (int)blockIdx.x >= a.first[i] ? i : which;
  const GemmArgsF32& p = a.p[which];
  const unsigned t = blockIdx.x - a.first[which], rows = (p.M + 15) / 16, cols = (p.N + 15) / 16;
  const unsigned q = t / rows, z = q / cols;
  const int m0 = 16 * (t - q * rows), n0 = 16 * (q - z * cols);
  if (KS <= 2 || p.K <= 64 * KS) Tile<1, 1, 1, 1, KS, true>(p, m0, n0, z, part);
  else Tile<1, 1, 1, 1, KS, false>(p, m0, n0, z, part);
}

template <int RT, int CT, int WM, int WN, int KS, bool ONE_STEP = false>
void LaunchTile(const GemmArgsF32& a, hipStream_t stream) {
  dim3 grid((a.M + 16 * RT * WM - 1) / (16 * RT * WM), (a.N + 16 * CT * WN - 1) / (16 * CT * WN), a.batch);
  hipLaunchKernelGGL((gemm_f32_mfma_kernel<RT, CT, WM, WN, KS, ONE_STEP>), grid, dim3(64 * WM * WN * KS), 0, stream, a);
}
}  // namespace

namespace {
long long Tiles(const GemmArgsF32& a, int size) { return (long long)((a.M + size - 1) / size) * ((a.N + size - 1) / size) * a.batch; }
}  // namespace

// Where a launch of its own would take 16x16 tiles for every product, up to 14 tiles for every CU in all: us of a pass, one by one ->
// together, 6x64 tower 1 position 129 -> 122, 32 142 -> 136, 100 189 -> 184; 10x256 1 355 -> 336, 20 451 -> 437, 40 619 -> 604, from 64 on level.
bool GemmF32Grouped(const GemmArgsF32* a, int count) {
  if (count < 2 || count > kGemmF32Group) return false;
  long long all = 0;
  for (int i = 0; i < count; i++) {
    if (a[i].M <= 0 || a[i].N <= 0 || a[i].K <= 0 || a[i].batch <= 0 || Tiles(a[i], 64) >= 400) return false;
    if (a[i].K <= 128 && Tiles(a[i], 16) >= 2048) return false;
    all += Tiles(a[i], 16);
  }
  return all <= 14 * 256;
}

void LaunchGemmF32Group(const GemmArgsF32* a, int count, hipStream_t stream) {
  if (!GemmF32Grouped(a, count)) throw std::runtime_error("LaunchGemmF32Group: not products for one launch");
  GroupArgs g;
  long long tiles = 0;
  int k = 0;
  for (int i = 0; i < kGemmF32Group; i++) {
    g.first[i] = (int)tiles;   // (beyond the last product: past the grid)
    if (i >= count) continue;
    g.p[i] = a[i];
    tiles += Tiles(a[i], 16);
    k = std::max(k, a[i].K);
  }
  const dim3 grid((unsigned)tiles);
  // (the waves that share a reduction as for one product of the longest one)
  if (k <= 64) hipLaunchKernelGGL(gemm_f32_group_kernel<1>, grid, dim3(64), 0, stream, g);
  else if (k <= 128) hipLaunchKernelGGL(gemm_f32_group_kernel<2>, grid, dim3(128), 0, stream, g);
  else if (k <= 256 || tiles > 256) hipLaunchKernelGGL(gemm_f32_group_kernel<4>, grid, dim3(256), 0, stream, g);
  else hipLaunchKernelGGL(gemm_f32_group_kernel<8>, grid, dim3(512), 0, stream, g);
}

void LaunchGemmF32(const GemmArgsF32& a, hipStream_t stream) {
  if (a.M <= 0 || a.N <= 0 || a.batch <= 0) return;
  // The tile is a matter of filling the CUs: at small sizes many 16x16 tiles balance them best, at large ones operand
  // traffic decides (16384x256x1024: 103 us on 64x64 tiles, 143 on 16x16 ones; 1280x256x1024: 25 against 13).
  const long long tiles16 = Tiles(a, 16), tiles64 = Tiles(a, 64);
  if (tiles64 >= 400 && a.K >= 512) {
    // Two waves share every operand row in both; a long reduction is worth splitting (16384x1024x256: 125 us unsplit
    // against 137; 16384x256x1024: 117 against 103).
    LaunchTile<4, 2, 1, 2, 4>(a, stream);
  } else if (a.K <= 128) {
    // One step for each of one or two waves. 32-row workgroups once there are several for every CU; before, a few more or
    // less than one per CU decide (a 6x64 tower at 32 positions, 1152 tiles of 36 x 128x64x64: 207 us a pass in single
    // tiles, 219 in 288 workgroups of 32x32; at 64 positions 239 in 32x32, with four waves per tile 242).
    if (a.K <= 64) {
      if (tiles16 < 2048) LaunchTile<1, 1, 1, 1, 1, true>(a, stream);
      else LaunchTile<1, 1, 2, 2, 1, true>(a, stream);
    } else if (tiles64 >= 400) {
      LaunchTile<1, 1, 2, 2, 1>(a, stream);
    } else {
      if (tiles16 < 2048) LaunchTile<1, 1, 1, 1, 2, true>(a, stream);
      else LaunchTile<1, 1, 2, 1, 2, true>(a, stream);
    }
  } else if (tiles64 >= 400) {
    LaunchTile<1, 1, 2, 2, 1>(a, stream);
  } else if (tiles16 <= 256 && a.K >= 1024) {
    // One workgroup per CU at most: eight waves share a long reduction (32x1858x2048: 8.4 us against 10.2 with four).
    LaunchTile<1, 1, 1, 1, 8>(a, stream);
  } else if (a.K <= 256) {
    LaunchTile<1, 1, 1, 1, 4, true>(a, stream);
  } else {
    LaunchTile<1, 1, 1, 1, 4>(a, stream);
  }
}

}  // namespace lc0mi
