// Hand-written gfx950 (CDNA4, wave64) matrix-product kernels of the dense layers.
//
// What each kernel replaces in the reference CPU backend (file:line):
//   gemm_kernel, gemm_dma_kernel, gemm_rowpanel_kernel, gemm_f32_mfma_kernel
//                         FullyConnectedLayer::Forward1D  blas/fully_connected_layer.cc:49-106
//                         (+ bias/activation of shared/activation.cc:102-164), the per-sample
//                         Q.K^T sgemm of the attention policy (blas/network_blas.cc:850-872) and the
//                         winograd-domain products of WinogradConvolution3 (blas/winograd_convolution3.cc:47-324)
#include "gemm_variants.h"
#include "kernel_common.h"

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>
#include <utility>

namespace lc0mi {

namespace {

// ---------------------------------------------------------------------------
// GEMM  C[m][n] = act(scale * sum_k A[m][k] W[n][k] + bias[n])
//
// 256 threads = 4 waves laid out WAVES_M x WAVES_N over a BM x BN block tile;
// each wave owns (BM/WAVES_M) x (BN/WAVES_N) as 32x32 MFMA tiles
// (v_mfma_f32_32x32x16_f16). The weight rows are the MFMA "A" operand and the
// activation rows the "B" operand, so a lane ends up holding 4 consecutive n
// for one m and stores 8 bytes at a time. Global tiles are fetched as 16-byte
// vectors into registers one k-tile ahead and staged through padded LDS.
// ---------------------------------------------------------------------------
// ET: type of the operands (half_t or bf16_t); OutT: float, or ET.
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, typename OutT, typename ET = half_t>
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs p) {
  using ev8 = typename Vec16<ET>::v8;
  static_assert(WAVES_M * WAVES_N == 4, "four waves per block");
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int LDS_STRIDE = BK + 8;  // halves; 16-byte rows shifted by 4 banks per row
  constexpr int VEC_PER_ROW = BK / 8;
  constexpr int A_VECS = BM * VEC_PER_ROW / 256;
  constexpr int W_VECS = BN * VEC_PER_ROW / 256;
  static_assert(A_VECS >= 1 && W_VECS >= 1, "tile too small for 256 threads");

  __shared__ __attribute__((aligned(16))) half_t As[BM * LDS_STRIDE];
  __shared__ __attribute__((aligned(16))) half_t Ws[BN * LDS_STRIDE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int zb = blockIdx.z / p.split_k, zs = blockIdx.z - zb * p.split_k;
  const half_t* A = p.A + (long long)zb * p.strideA;
  const half_t* W = p.W + (long long)zb * p.strideW;
  const int M = p.M, N = p.N;
  // This workgroup's slice of the reduction dimension.
  const int k_slice = ((p.K + p.split_k - 1) / p.split_k + BK - 1) / BK * BK;
  const int k_begin = zs * k_slice;
  const int K = min(p.K, k_begin + k_slice);

  uint4 ra[A_VECS], rw[W_VECS];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_VECS; i++) {
      int v = tid + i * 256;
      int row = v / VEC_PER_ROW, kv = v % VEC_PER_ROW;
      int gm = min(m0 + row, M - 1), k = k0 + kv * 8;
      ra[i] = k < K ? *reinterpret_cast<const uint4*>(A + (long long)gm * p.lda + k) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < W_VECS; i++) {
      int v = tid + i * 256;
      int row = v / VEC_PER_ROW, kv = v % VEC_PER_ROW;
      int gn = min(n0 + row, N - 1), k = k0 + kv * 8;
      rw[i] = k < K ? *reinterpret_cast<const uint4*>(W + (long long)gn * p.ldw + k) : make_uint4(0, 0, 0, 0);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int i = 0; i < A_VECS; i++) {
      int v = tid + i * 256;
      int row = v / VEC_PER_ROW, kv = v % VEC_PER_ROW;
      *reinterpret_cast<uint4*>(&As[row * LDS_STRIDE + kv * 8]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < W_VECS; i++) {
      int v = tid + i * 256;
      int row = v / VEC_PER_ROW, kv = v % VEC_PER_ROW;
      *reinterpret_cast<uint4*>(&Ws[row * LDS_STRIDE + kv * 8]) = rw[i];
    }
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  const int nk = K > k_begin ? (K - k_begin + BK - 1) / BK : 0;
  const int frag_row = lane & 31, frag_k = (lane >> 5) * 8;
  if (nk > 0) load_tile(k_begin);
  for (int kt = 0; kt < nk; kt++) {
    store_tile();
    __syncthreads();
    if (kt + 1 < nk) load_tile(k_begin + (kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) {
      ev8 af[TM], wf[TN];
#pragma unroll
      for (int i = 0; i < TM; i++)
        af[i] = *reinterpret_cast<const ev8*>(&As[(wm * WM + i * 32 + frag_row) * LDS_STRIDE + ks * 16 + frag_k]);
#pragma unroll
      for (int j = 0; j < TN; j++)
        wf[j] = *reinterpret_cast<const ev8*>(&Ws[(wn * WN + j * 32 + frag_row) * LDS_STRIDE + ks * 16 + frag_k]);
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = Mfma32(wf[j], af[i], acc[i][j]);
    }
    __syncthreads();
  }

  // Epilogue. Accumulator element e of a tile: n = 8*(e/4) + 4*(lane/32) + e%4, m = lane%32.
  OutT* C = reinterpret_cast<OutT*>(p.C) + (long long)zb * p.strideC;
  if constexpr (sizeof(OutT) == 4) {
    if (p.split_k > 1) {
      // Every slice stores its own partial sums (no atomics: the consumer adds the
      // slices in a fixed order, so results do not depend on scheduling).
      C += (long long)zs * p.split_stride;
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
          const int n = n0 + wn * WN + j * 32 + blk * 8 + (lane >> 5) * 4;
          float b4[4];
          LoadBias4(zs == 0 ? p.bias : nullptr, n, N, b4);
#pragma unroll
          for (int i = 0; i < TM; i++) {
            const int m = m0 + wm * WM + i * 32 + frag_row;
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (m < M && n + r < N) C[(long long)m * p.ldc + n + r] = acc[i][j][blk * 4 + r] * p.scale + b4[r];
          }
        }
      return;
    }
  }
  const bool vec_ok = (p.ldc % 4 == 0);
  // Consumer side of a folded layer norm (GemmArgs::row_stats): mean and rstd of this lane's rows.
  float row_mean[TM], row_rstd[TM];
#pragma unroll
  for (int i = 0; i < TM; i++) {
    row_mean[i] = 0.0f;
    row_rstd[i] = 1.0f;
    if (p.row_stats != nullptr) {
      RowMeanRstd(p.row_stats, p.row_parts, min(m0 + wm * WM + i * 32 + frag_row, M - 1), p.norm_n, p.norm_eps,
                  row_mean[i], row_rstd[i]);
    }
  }
  DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int blk = 0; blk < 4; blk++) {
        const int n = n0 + wn * WN + j * 32 + blk * 8 + (lane >> 5) * 4;
        if (n >= N) continue;
        float b4[4], c4[4];
        LoadBias4(p.bias, n, N, b4);
        LoadBias4(p.row_stats != nullptr ? p.col_c : nullptr, n, N, c4);
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const int m = m0 + wm * WM + i * 32 + frag_row;
          if (m >= M) continue;
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; r++)
            v[r] = act_fn(row_rstd[i] * (acc[i][j][blk * 4 + r] * p.scale - row_mean[i] * c4[r]) + b4[r]);
          OutT* dst = C + (long long)m * p.ldc + n;
          if (vec_ok && n + 3 < N) {
            if constexpr (sizeof(OutT) == 2) {
              using ov4 = typename Vec16<OutT>::v4;
              ov4 h = {(OutT)v[0], (OutT)v[1], (OutT)v[2], (OutT)v[3]};
              *reinterpret_cast<ov4*>(dst) = h;
            } else {
              floatx4 f = {v[0], v[1], v[2], v[3]};
              *reinterpret_cast<floatx4*>(dst) = f;
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (n + r < N) dst[r] = (OutT)v[r];
          }
        }
      }
    }
  });
}

template <int BM, int BN, int BK, int WAVES_M, int WAVES_N>
void LaunchGemmTile(const GemmArgs& a, hipStream_t stream) {
  dim3 grid((a.M + BM - 1) / BM, (a.N + BN - 1) / BN, a.batch * a.split_k);
  if (a.bf16) {
    if (a.out_f32) {
      hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, WAVES_M, WAVES_N, float, bf16_t>), grid, dim3(256), 0, stream, a);
    } else {
      hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, WAVES_M, WAVES_N, bf16_t, bf16_t>), grid, dim3(256), 0, stream, a);
    }
  } else if (a.out_f32) {
    hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, WAVES_M, WAVES_N, float>), grid, dim3(256), 0, stream, a);
  } else {
    hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, WAVES_M, WAVES_N, half_t>), grid, dim3(256), 0, stream, a);
  }
}

}  // namespace

namespace {
int g_variant_override = -1;

GemmVariant PickGemmVariant(const GemmArgs& a);

// Cost model of the five direct-to-LDS tile shapes in halves, in microseconds per launch (see PickGemmVariant), outside the range of the
// one below.
struct FittedCosts {
  double t256, t192, t128, ts, t64;
  double Best() const { return std::min(std::min(std::min(t256, t192), std::min(t128, ts)), t64); }
};
inline bool InFittedDomain(const GemmArgs& a) { return a.batch == 1 && a.M >= 4096 && a.K >= 512 && a.N >= 512; }
inline FittedCosts FitCosts(int M, int N, int K) {
  const double kt = K / 64.0;
  auto tiles = [&](int bm, int bn) { return (double)((M + bm - 1) / bm) * (double)((N + bn - 1) / bn); };
  auto rounds_of = [](double x) {
    const double whole = std::floor(x + 1e-9), frac = x - whole;
    return whole + (frac > 1e-9 ? 0.55 + 0.45 * frac : 0.0);
  };
  FittedCosts c;
  c.t256 = 1.6 + rounds_of(tiles(256, 256) / 256.0) * (6.93 + 1.814 * kt);
  c.t192 = 1.6 + rounds_of(tiles(256, 192) / 256.0) * (5.37 + 1.444 * kt);
  c.t128 = 1.08 * (1.6 + rounds_of(tiles(256, 128) / 256.0) * (2.53 + 1.215 * kt));
  c.ts = 2.62 + std::max(0.5, tiles(128, 128) / 512.0) * (3.62 + 1.140 * kt);
  c.t64 = 1.19 + std::max(0.34, tiles(128, 64) / 768.0) * (2.75 + 1.119 * kt);
  return c;
}

// Cost model of the direct-to-LDS tiles in microseconds: fixed + rounds * (round + step * k-tiles), a k-tile being 128 bytes and
// a round a tile on each of the 256 CUs; a last round that fills a fraction f of the CUs counts partial + (1 - partial) f.
// (Shapes that share a CU follow it as well: a tile beside others takes proportionally longer.) Fitted to all shapes on 120
// problems in halves and 140 in e4m3, M 1536 to 57600 in steps of 64, N 512 to 3072, K 512 to 2048, in the order of tiles of
// PickTileOrder; rms error 2 to 7 %. Back to back the shape it picks is 0.4 % (halves) and 0.5 % (e4m3) behind the fastest one
// measured, the choice before it 2.5 and 1.9 %.
// Within a pass that holds only in part: from 80 positions the projection has the smolgen chain beside it, which finds no
// room on CUs that 256x256 tiles fill (us a pass, choice before -> by this model: fp16 100 positions 3131 -> 3438, e4m3 200 3749
// -> 4221), and from 16384 rows the other products leave through the cache only from 256-row tiles (e4m3 300 5080 -> 5185). So
// it decides on wide products up to 2559 rows in halves (32 positions 1621 -> 1573, 36 1888 -> 1782; from there to 64 they are level at
// best, 46 2010 -> 2026) and up to 5119 in e4m3 (32 1172 -> 1140, 36 1349 -> 1305, 50 1553 -> 1522; the other products of so few
// rows are level or 1 % slower) and on the others from 5120 to 16383 rows (fp16 90 3047 -> 2988, 150 4240 -> 4008; e4m3 100 2436 -> 2372,
// 117 2564 -> 2480, 200 3612 -> 3540, but 90 2248 -> 2267).
struct TileCost {
  GemmVariant variant;
  int bm, bn;
  double fixed, round, step, partial;
};
constexpr TileCost kHalfCosts[] = {{kDma256x256, 256, 256, 2.07, 5.95, 1.700, 0.655}, {kDma256x192, 256, 192, 1.92, 4.94, 1.368, 0.634},
                                   {kDma256x128, 256, 128, 3.59, 1.46, 1.156, 0.536}, {kDma128x128, 128, 128, 3.43, 1.27, 0.531, 0.566},
                                   {kDma128x64, 128, 64, 2.58, 0.38, 0.365, 0.453}};
constexpr TileCost kF8Costs[] = {{kDma256x256, 256, 256, 3.64, 5.31, 1.699, 0.647}, {kDma256x192, 256, 192, 2.85, 4.69, 1.369, 0.630},
                                 {kDma256x128, 256, 128, 2.85, 2.98, 1.021, 0.632}, {kDma128x128, 128, 128, 4.01, 1.37, 0.488, 0.501},
                                 {kDma128x64, 128, 64, 3.21, 0.61, 0.305, 0.432}, {kDma64x64, 64, 64, 2.56, 0.35, 0.186, 0.476}};

constexpr int kHalfWideEnd = 2560, kF8WideEnd = 5120;
inline bool InTileCostDomain(int M, int N, int K, int wide_end) {
  if (K < 512 || N < 512) return false;
  return N >= 2 * K ? M >= 1536 && M < wide_end : M >= 5120 && M < 16384;
}

double CostOf(const TileCost& c, int M, int N, int k_tiles) {
  const double x = (double)((M + c.bm - 1) / c.bm) * (double)((N + c.bn - 1) / c.bn) / 256.0, whole = std::floor(x + 1e-9);
  const double rounds = whole + (x - whole > 1e-9 ? c.partial + (1.0 - c.partial) * (x - whole) : 0.0);
  return c.fixed + rounds * (c.round + c.step * k_tiles);
}

template <size_t COUNT, typename Accept>
const TileCost* Cheapest(const TileCost (&costs)[COUNT], int M, int N, int k_tiles, Accept&& accept) {
  const TileCost* best = nullptr;
  double cost = 0.0;
  for (const TileCost& c : costs) {
    if (!accept(c.variant)) continue;
    const double v = CostOf(c, M, N, k_tiles);
    if (best == nullptr || v < cost) { best = &c; cost = v; }
  }
  return best;
}
template <size_t COUNT>
const TileCost* Cheapest(const TileCost (&costs)[COUNT], int M, int N, int k_tiles) {
  return Cheapest(costs, M, N, k_tiles, [](GemmVariant) { return true; });
}

// A large product whose tiles do not fill whole rounds of the 256 CUs, cut along its rows: the rows that make whole
// rounds of 256x256 (or 256x192) tiles go to one launch and the rest to a second launch on whatever shape suits it
// (20480x1024x1536 in halves: 87 us on 320 tiles of 256x256, one and a quarter rounds, or 78 us on 128x128 tiles, against
// 49 + 19 us for 16384 rows on one full round of large tiles and 4096 rows on small ones). Cut when the model above prices the
// pair at least 3 % below the best single shape.
bool g_row_split = true;   // (profiling and tests switch it off through SetGemmRowSplit)
struct RowSplit {
  int rows = 0;                                    // of the first launch (0: one launch)
  GemmVariant first = kDma256x256, rest = kNoVariant;   // (rest kNoVariant: as a product of its own)
};
// (Below 5120 rows a product of its own can get another shape than the cheapest of this table, by which the rest is priced. The rest runs
// on the cheapest where the other is priced more than the model's error above it: us of a product, rest as of its own -> this, 12608x2048x2048
// 130 -> 124, one launch 124, 12416x1984x1856 119 -> 112 and 113; where they are close its own shape is the faster one, 4096x1088x1728 26.9 on
// 128x128 tiles against 28.7 on 128x64.)
RowSplit PlanRowSplitByTileCost(const GemmArgs& a) {
  const auto& costs = kHalfCosts;
  const int M = a.M, N = a.N, k_tiles = a.K / 64;
  double best = CostOf(*Cheapest(costs, M, N, k_tiles), M, N, k_tiles) * 0.97;
  RowSplit plan;
  for (int v = 0; v < 2; v++) {
    const int col_tiles = (N + costs[v].bn - 1) / costs[v].bn;
    if (col_tiles > 256) continue;
    const int rows_per_round = (256 / col_tiles) * 256;
    for (int m1 = rows_per_round; m1 + 4096 <= M; m1 += rows_per_round) {   // (cut at 2048 rows, 96 positions lost 4 %)
      const TileCost& rest = *Cheapest(costs, M - m1, N, k_tiles);
      const double c = CostOf(costs[v], m1, N, k_tiles) + CostOf(rest, M - m1, N, k_tiles) + 1.0;
      if (c < best) { best = c; plan = {m1, costs[v].variant, rest.variant}; }
    }
  }
  if (plan.rows > 0) {
    GemmArgs rest = a;
    rest.M = M - plan.rows;
    const GemmVariant own = PickGemmVariant(rest);
    const TileCost* c = Cheapest(costs, rest.M, N, k_tiles, [&](GemmVariant v) { return v == own; });
    if (c != nullptr && CostOf(*c, rest.M, N, k_tiles) <= 1.05 * CostOf(*Cheapest(costs, rest.M, N, k_tiles), rest.M, N, k_tiles)) plan.rest = own;
  }
  return plan;
}

RowSplit PlanRowSplit(const GemmArgs& a) {
  if (!g_row_split || g_variant_override >= 0 || a.batch != 1 || a.out_f32 || a.split_k != 1 || a.K % 64 != 0 || a.skip != nullptr ||
      a.row_stats != nullptr) {
    return {};
  }
  if (InTileCostDomain(a.M, a.N, a.K, kHalfWideEnd)) return PlanRowSplitByTileCost(a);
  if (!InFittedDomain(a)) return {};
  double best = FitCosts(a.M, a.N, a.K).Best() * 0.97;
  RowSplit plan;
  for (int v = 0; v < 2; v++) {
    const int bn = v == 0 ? 256 : 192;
    const int col_tiles = (a.N + bn - 1) / bn;
    if (col_tiles > 256) continue;
    const int rows_per_round = (256 / col_tiles) * 256;
    // (the rest stays inside the range of sizes the model was fitted on: cut at 2048 rows, a 15x1024 pass at 96
    //  positions lost 4 %)
    for (int m1 = rows_per_round; m1 + 4096 <= a.M; m1 += rows_per_round) {
      const FittedCosts top = FitCosts(m1, a.N, a.K);
      const double c = (v == 0 ? top.t256 : top.t192) + FitCosts(a.M - m1, a.N, a.K).Best() + 1.0;
      if (c < best) { best = c; plan = {m1, v == 0 ? kDma256x256 : kDma256x192, kNoVariant}; }
    }
  }
  return plan;
}

// The smallest direct-to-LDS tile with which an output fits the CUs with one workgroup each (kNoVariant: none does). A
// workgroup's time hardly depends on how many others run (us at K = 1024 / 1536: 64x64 5.6 / 6.9, 128x64 7.1 / 8.8,
// 128x128 9.6 / 12.2), a second workgroup on some of the CUs costs most of that time again: 832x1536x1024 8.0 us on 168
// tiles of 128x64 against 9.4 on 312 of 64x64, 832x3072x1024 12.8 on 168 tiles of 128x128 against 13.5 on 336 of 128x64,
// 1024x1024x1536 7.7 on 256 tiles of 64x64 against 9.2 on 128 of 128x64.
inline GemmVariant OneRoundTile(int M, int N, int batch) {
  auto fits = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * batch <= 256; };
  return fits(64, 64) ? kDma64x64 : fits(128, 64) ? kDma128x64 : fits(128, 128) ? kDma128x128 : kNoVariant;
}

// Whether the workgroups of a second product of N2 columns are no more per CU than those of the first one alone: the
// launch then takes no longer than without them.
bool SecondFits(GemmVariant v, int M, int N, int N2) {
  if (v == kRowPanel) {
    for (const RowPanelShape& c : kRowPanelShapes) {   // (the panel that the first product gets)
      const long long first = RowPanelWorkgroups(M, N, 1, c);
      if (first <= kRowPanelWorkgroups) return first + RowPanelWorkgroups(M, N2, 1, c) <= kRowPanelWorkgroups;
    }
    return false;
  }
  const int bm = v == kDma64x64 ? 64 : 128, bn = v == kDma128x128 ? 128 : 64;
  if (v != kDma64x64 && v != kDma128x64 && v != kDma128x128) return false;
  const long long rows = (M + bm - 1) / bm, first = rows * ((N + bn - 1) / bn), both = first + rows * ((N2 + bn - 1) / bn);
  return (both + 255) / 256 == (first + 255) / 256;
}
// The cheapest shape by the cost model. With a second product the cheapest that takes it is allowed 1.5 us more: a launch of its own for
// the second one costs more, but the smaller tiles lose some of that again (with 4 us 50 positions in halves 2053 -> 2078 a pass).
template <size_t COUNT, typename Accept>
GemmVariant PickFitted(const TileCost (&costs)[COUNT], int M, int N, int k_tiles, int N2, Accept&& accept) {
  const TileCost* best = Cheapest(costs, M, N, k_tiles, accept);
  if (N2 > 0 && !SecondFits(best->variant, M, N, N2)) {
    const TileCost* both = Cheapest(costs, M, N, k_tiles, [&](GemmVariant v) { return accept(v) && SecondFits(v, M, N, N2); });
    if (both != nullptr && CostOf(*both, M, N, k_tiles) <= CostOf(*best, M, N, k_tiles) + 1.5) best = both;
  }
  return best->variant;
}

GemmVariant PickGemmVariant(const GemmArgs& a) {
  if (g_variant_override >= 0) {
    const bool dma_ok = !a.out_f32 && a.split_k == 1 && a.K % 64 == 0;
    const bool is_dma = g_variant_override <= kDma256x128 || g_variant_override == kDma128x128 ||
                        g_variant_override == kDma128x64 || g_variant_override == kDma128x32 ||
                        g_variant_override == kDma64x64;
    bool ok = is_dma ? dma_ok : (g_variant_override != kRowPanel || a.split_k == 1);
    if (g_variant_override == kNoVariant) ok = false;
    if (g_variant_override == kResident) ok = GemmResidentWorkgroups(a) > 0;
    if (ok) return static_cast<GemmVariant>(g_variant_override);
  }
  const long long tiles128 = (long long)((a.M + 127) / 128) * ((a.N + 127) / 128) * a.batch;
  if (!a.out_f32 && a.split_k == 1 && a.K % 64 == 0 && a.K <= 512 && a.batch > 1) {
    // Many products with short reductions (36 winograd-domain products of a convolution; the longer reductions of the
    // policy logits, one product per position, keep the register-staged tiles).
    // Resident weights from 512 rows up where the row blocks fill their rounds (us against the best of the tiles, 36 x M
    // x 256x256: M = 512 9.5 / 9.4, 640 10.0 / 11.6, 768 10.6 / 12.9, 2048 21.8 / 23.5, 4096 32.2 / 37.3; with 8 blocks on
    // 7 workgroups M = 1024 15.1 / 13.9).
    const int share = GemmResidentWorkgroups(a), blocks = (a.M + 127) / 128;
    if (share > 0 && a.M >= 512 && 10 * blocks >= 7 * share * ((blocks + share - 1) / share)) return kResident;
    // 64x64 tiles while about two workgroups share a CU (M = 32 3.5 us against 5.4 on the register-staged tiles, 128
    // 4.3 / 6.1, 256 5.3 against 5.9 on 128x64; M = 384 10.8), then 128x128 alone on a CU (384: 7.1) or 128x64 tiles; with
    // narrow products 64x64 throughout (1536 x 64x64 4.2 us against 6.2).
    // (What one workgroup per CU of the row panels below covers is left to them: 16 x 64x64x256 2.7 us against 3.3, 20 x
    // 4x256x256 2.8 against 3.3.)
    const bool panels = a.K >= 256 && RowPanelWorkgroups(a.M, a.N, a.batch, kRowPanelShapes[3]) <= kRowPanelWorkgroups;
    if (!panels && (long long)((a.M + 63) / 64) * ((a.N + 63) / 64) * a.batch <= 640) return kDma64x64;
    if (!panels && a.N >= 128 && tiles128 <= 256) return kDma128x128;
    if (!panels && (a.M < 1024 || a.N < 128 || a.K < 128)) return a.N <= 64 ? kDma64x64 : kDma128x64;
  }
  if (!a.out_f32 && a.split_k == 1 && a.K % 64 == 0 && a.K >= 128 && a.N >= 128 && a.M >= (a.latency_first ? 256 : 1024) && tiles128 >= 64) {
    // Direct-to-LDS kernels. Cost = rounds over the 256 CUs x tile area x a measured cost per
    // output element and round (ns per element at K = 1024): 0.60 for 256x256, 0.61 for 256x192;
    // the two small shapes run two workgroups per CU, 0.68 (256x128) and 0.75 (128x128) per element
    // while sharing a CU, 0.84 and 0.95 when a single round leaves every workgroup alone on its CU.
    if (a.batch == 1 && InTileCostDomain(a.M, a.N, a.K, kHalfWideEnd)) {
      auto known = [&](GemmVariant v) { return v != kDma256x192 || a.skip == nullptr; };
      return PickFitted(kHalfCosts, a.M, a.N, a.K / 64, a.N2, known);
    }
    if (InFittedDomain(a)) {
      const FittedCosts c = FitCosts(a.M, a.N, a.K);
      GemmVariant best = kDma256x256;
      double cost = c.t256;
      if (c.t192 < cost && a.skip == nullptr) { best = kDma256x192; cost = c.t192; }
      if (c.t128 < cost) { best = kDma256x128; cost = c.t128; }
      if (c.ts < cost) { best = kDma128x128; cost = c.ts; }
      if (c.t64 < cost) { best = kDma128x64; cost = c.t64; }
      return best;
    }
    if (a.K >= 512 && a.batch == 1) {
      const GemmVariant v = OneRoundTile(a.M, a.N, 1);
      if (v != kNoVariant) return v;
    }
    auto rounds = [&](int bm, int bn) {
      const long long tiles = (long long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn) * a.batch;
      return (double)((tiles + 255) / 256);
    };
    const double r256 = rounds(256, 256), r192 = rounds(256, 192), r128 = rounds(256, 128), rs = rounds(128, 128);
    const double c256 = r256 * 256 * 256 * 0.60;
    const double c192 = r192 * 256 * 192 * 0.61;
    const double c128 = r128 * 256 * 128 * (r128 > 1 ? 0.68 : 0.84);
    // (short reductions are dominated by the epilogue, where the smallest tile loses a little more)
    const double cs = rs * 128 * 128 * (rs > 1 ? 0.75 : 0.95) * (a.K <= 256 ? 1.12 : 1.0);
    GemmVariant best = kDma256x256;
    double cost = c256;
    // (a producer of a folded layer norm needs a power-of-two column count per wave: not the 192-wide tile)
    if (c192 < cost && a.skip == nullptr) { best = kDma256x192; cost = c192; }
    if (c128 < cost) { best = kDma256x128; cost = c128; }
    if (cs < cost) { best = kDma128x128; cost = cs; }
    // 128x64 tiles (three workgroups per CU, so partial rounds are counted as fractions) move more operand
    // bytes from L2 per flop, but they split small problems over all CUs and odd tile counts evenly
    // (4096x512x1024: 10.5 us against 14.6 for 128x128; 36 x 2048x256x256: 23.1 us against 26.0 for 256x128).
    {
      const double tiles = (double)((a.M + 127) / 128) * ((a.N + 63) / 64) * a.batch;
      const double c64 = std::max(1.0, tiles / 256.0) * 128 * 64 * 0.80;
      if (c64 < cost) { best = kDma128x64; cost = c64; }
    }
    return best;
  }
  // Very many rows, at most 32 columns (the smolgen compression at 512 positions and more): a memory-bound stream of
  // the activation rows. 128x32 direct-to-LDS tiles (four workgroups per CU) read them once at full line width
  // (65536x32x1024: 34 us against 96 for the row-panel kernel).
  if (!a.out_f32 && a.split_k == 1 && a.batch == 1 && a.N <= 32 && a.K % 64 == 0 && a.K >= 128 && a.M >= 32768) {
    return kDma128x32;
  }
  // Small problems: the row-panel kernel (K split over the waves of a workgroup, panels sized to give every CU one) as
  // long as panels of 32x32 cover the output with one workgroup per CU (64x3072x1024 5.6 us against 7.1 on 64x64
  // direct-to-LDS tiles, 256x1024x1536 7.4 against 9.2, 1x8192x256 3.6 against 5; beyond that the tiles win:
  // 128x3072x1024 7.2 against 7.7 to 9.6, 64x8192x256 4.3 against 5.1 to 6.4).
  if (a.split_k == 1 && a.K >= 256 && RowPanelWorkgroups(a.M, a.N, a.batch, kRowPanelShapes[3]) <= kRowPanelWorkgroups) {
    return kRowPanel;
  }
  // At most 128 rows and too many columns or products for that, up to 128 tiles of 64x64: direct-to-LDS tiles where they
  // serve (33x8192x256 3.5 us against 4.0 on 64x32 panels and 5.4 on the register-staged tiles, 33x8192x1024 5.8 against
  // 6.2 and 12.4, 64x8192x256 3.5 against 4.2 and 5.4, 77 products of 64x64x1024 5.4 against 7.9 and 10.5), else 64x32 panels
  // (float output: 33x8192x256 4.0 against 5.5, 128x3072x1024 6.2 against 10.0, 77 products of 64x64x1024 8.0 against 12.9).
  const long long tiles64 = (long long)((a.M + 63) / 64) * ((a.N + 63) / 64) * a.batch;
  if (a.split_k == 1 && a.K >= 256 && a.M <= 128 && tiles64 <= 128) {
    return !a.out_f32 && a.K % 64 == 0 && a.N >= 64 ? kDma64x64 : kRowPanel;
  }
  // A few hundred rows (3 to 12 positions), or few columns: too small for the cost model above, too large for row
  // panels. Small direct-to-LDS tiles with three or four stages in flight stream the weights, which come from
  // memory, better than the register-staged tiles below (512x1024x1024: 6.8 against 9.9 us; a pass of 8 positions
  // 1.94 -> 1.46 ms).
  // (With a short reduction only on request: beside a large GEMM on the other stream the register-staged tiles
  // disturb it less.)
  if (!a.out_f32 && a.split_k == 1 && a.K % 64 == 0 && a.K >= (a.latency_first ? 256 : 512) && a.N >= 64 && a.M >= (a.batch == 1 ? 64 : 192)) {
    const GemmVariant v = OneRoundTile(a.M, a.N, a.batch);
    return v != kNoVariant ? v : kDma128x64;
  }
  // A single 32-column panel (the smolgen compression): one workgroup per 64 rows, K split over its waves
  // (16384x32x1024: 6.8 us against 12.8 on the 64x64 tiles and 9.6 on the 128x32 ones, but with twice the threads on
  // every CU; 4096 rows 4.2 / 9.8 / 6.1).
  if (a.latency_first && a.split_k == 1 && a.N <= 32 && a.K >= 512) return kRowPanel;
  // Float output has no direct-to-LDS form. 64x32 panels, up to two for every CU, instead of register-staged 64x64 tiles (the
  // dense policy layer of a tower, 256x1858x2048 10.1 us against 19.6, 512 17.8 / 24.4, 700 25.1 / 26.5, 1024 36.4 / 28.8).
  if (a.out_f32 && a.split_k == 1 && a.batch == 1 && a.K >= 1024 && RowPanelWorkgroups(a.M, a.N, 1, kRowPanelShapes[4]) <= 2 * kRowPanelWorkgroups) {
    return kRowPanel;
  }
  // Many products that each fit a 64x64 tile (the policy head's Q.K^T per position) would leave three quarters of
  // every 128x128 tile empty (256 x 64x64x1024: 14.5 against 21.4 us).
  if (a.M <= 64 && a.N <= 64) return kTile64;
  const long long big_tiles = tiles128;
  return big_tiles >= 192 ? kTile128 : kTile64;
}
}  // namespace

void SetGemmVariantOverride(int variant) { g_variant_override = variant; }
void SetGemmRowSplit(bool on) { g_row_split = on; }

namespace {
// Column-tile width of the direct-to-LDS variants (0 for the others).
int DmaTileN(GemmVariant v) {
  switch (v) {
    case kDma256x256: return 256;
    case kDma256x192: return 192;
    case kDma256x128: case kDma128x128: return 128;
    case kDma128x64: case kDma64x64: return 64;
    case kDma128x32: return 32;
    default: return 0;
  }
}
}  // namespace

bool GemmSupportsNormFolding(const GemmArgs& a) {
  if (a.bf16 && (a.skip != nullptr || a.row_stats != nullptr)) return false;
  const GemmVariant v = PickGemmVariant(a);
  if (a.skip != nullptr) {
    return DmaTileN(v) != 0 && v != kDma256x192 && !a.out_f32 && a.act == 3 && a.batch == 1 && a.N % 8 == 0 &&
           a.ldc % 8 == 0 && a.ldskip % 8 == 0 && a.row_stats == nullptr;
  }
  if (a.row_stats != nullptr) {
    if (a.split_k != 1 || a.batch != 1 || a.col_c == nullptr) return false;
    return DmaTileN(v) != 0 || v == kTile128 || v == kTile64 || v == kRowPanel;
  }
  return true;
}

bool GemmTakesSecond(const GemmArgs& a) {
  return a.batch == 1 && a.split_k == 1 && !a.out_f32 && a.skip == nullptr && a.row_stats == nullptr && a.N2 % 8 == 0 &&
         a.ldw2 % 8 == 0 && a.ldc2 % 8 == 0 && PlanRowSplit(a).rows == 0 && SecondFits(PickGemmVariant(a), a.M, a.N, a.N2);
}

int GemmStatsParts(const GemmArgs& a) {
  const int bn = DmaTileN(PickGemmVariant(a));
  return bn == 0 ? 0 : (a.N + bn - 1) / bn;
}

int GemmRowSplit(const GemmArgs& a) {
  return PlanRowSplit(a).rows;
}

namespace {
const char* NameOf(GemmVariant v, const GemmArgs& a) {
  switch (v) {
    case kDma256x256: return "gemm_dma_256x256x64";
    case kDma256x192: return "gemm_dma_256x192x64";
    case kDma256x128: return "gemm_dma_256x128x32";
    case kDma128x128: return "gemm_dma_128x128x64";
    case kDma128x64: return "gemm_dma_128x64x64";
    case kDma128x32: return "gemm_dma_128x32x64";
    case kDma64x64: return "gemm_dma_64x64x64";
    case kResident: return "gemm_resident";
    case kRowPanel: return "gemm_rowpanel";
    case kTile128: return "gemm_128x128x64";
    default: return a.split_k > 1 ? "gemm_64x64x64_splitk" : "gemm_64x64x64";
  }
}

GemmArgs RestOf(const GemmArgs& a, int rows) {
  GemmArgs rest = a;
  rest.M = a.M - rows;
  rest.A = a.A + static_cast<long long>(rows) * a.lda;
  rest.C = static_cast<half_t*>(a.C) + static_cast<long long>(rows) * a.ldc;
  return rest;
}
GemmVariant RestVariant(const RowSplit& plan, const GemmArgs& rest) { return plan.rest != kNoVariant ? plan.rest : PickGemmVariant(rest); }
}  // namespace

const char* GemmVariantName(const GemmArgs& a) {
  const RowSplit plan = PlanRowSplit(a);
  if (plan.rows > 0) return plan.first == kDma256x256 ? "gemm_dma_256x256x64+rest" : "gemm_dma_256x192x64+rest";
  return NameOf(PickGemmVariant(a), a);
}

const char* GemmRestVariantName(const GemmArgs& a) {
  const RowSplit plan = PlanRowSplit(a);
  GemmArgs rest = a;
  rest.M = a.M - plan.rows;
  return plan.rows > 0 ? NameOf(RestVariant(plan, rest), rest) : "";
}

namespace {
void LaunchDma(GemmVariant v, const GemmArgs& a, hipStream_t stream) {
  if (a.bf16) LaunchGemmDmaBf16(v, a, stream);
  else LaunchGemmDmaHalf(v, a, stream);
}

void LaunchGemmOne(GemmVariant v, const GemmArgs& a, hipStream_t stream) {
  switch (v) {
    case kRowPanel: LaunchGemmRowPanel(a, stream); break;
    case kResident: LaunchGemmResident(a, stream); break;
    case kTile128: LaunchGemmTile<128, 128, 64, 2, 2>(a, stream); break;
    case kTile64: LaunchGemmTile<64, 64, 64, 2, 2>(a, stream); break;
    default: LaunchDma(v, a, stream); break;
  }
}
}  // namespace

void LaunchGemm(const GemmArgs& a, hipStream_t stream) {
  if (a.M <= 0 || a.N <= 0 || a.batch <= 0) return;
  if (a.N2 > 0 && !GemmTakesSecond(a)) throw std::runtime_error("LaunchGemm: no kernel with a second product for this shape");
  if ((a.skip != nullptr || a.row_stats != nullptr) && !GemmSupportsNormFolding(a)) {
    throw std::runtime_error("LaunchGemm: no kernel variant with the folded layer-norm epilogue for this shape");
  }
  const RowSplit plan = PlanRowSplit(a);
  if (plan.rows > 0) {
    GemmArgs top = a, rest = RestOf(a, plan.rows);
    top.out_stores = rest.out_stores = ResolvedOutStores(a);   // as for the whole product
    top.M = plan.rows;
    LaunchDma(plan.first, top, stream);
    LaunchGemmOne(RestVariant(plan, rest), rest, stream);   // (the rest is below one round of the large tiles: one launch)
    return;
  }
  LaunchGemmOne(PickGemmVariant(a), a, stream);
}

namespace {
// Few rows: row panels, as for fp16 operands.
bool GemmF8TakesRowPanels(const GemmF8Args& a) {
  return a.K >= 256 && RowPanelWorkgroups(a.M, a.N, 1, kRowPanelShapes[3]) <= kRowPanelWorkgroups;
}

// Outside the fitted range kDma256x256, kDma256x192, kDma256x128, kDma128x128 and kDma128x64 (two / three workgroups per CU) by
// the cost per element of the fp16 kernels (the k-tile structure is the same).
GemmVariant PickGemmF8Variant(const GemmF8Args& a) {
  if (g_variant_override >= 0 && (g_variant_override <= 2 || g_variant_override == kDma128x128 ||
                                  g_variant_override == kDma128x64 || g_variant_override == kRowPanel ||
                                  g_variant_override == kDma64x64)) {
    return static_cast<GemmVariant>(g_variant_override);
  }
  if (GemmF8TakesRowPanels(a)) return kRowPanel;
  if (InTileCostDomain(a.M, a.N, a.K, kF8WideEnd)) return PickFitted(kF8Costs, a.M, a.N, (a.K + 127) / 128, a.N2, [](GemmVariant) { return true; });
  // A few hundred to a few thousand rows: 64x64 tiles, up to three workgroups of which share a CU and fill each other's
  // gaps (us against 128x64 tiles: 1024x1024x1536 5.5 / 6.8, 2048x1024x1024 5.5 / 6.3, 2048x1536x1024 on 768 tiles
  // 7.4 / 7.9, 4096x1024x1024 on 1024 tiles 8.9 / 8.5). With several per CU, few rows and weights beyond the 4 MiB of an
  // XCD's L2 the 128x64 tiles, which read them half as often, stay ahead (512x3072x1536 8.8 / 6.8, 256x8192x2048 12.2 / 9.1,
  // 300x8192x1024 9.1 / 7.9; 256x8192x512 with 4 MiB 4.4 / 4.8, 1024x3072x1536 with twice the rows 10.6 / 11.2).
  const long long tiles64 = (long long)((a.M + 63) / 64) * ((a.N + 63) / 64);
  const bool few_rows_large_weights = tiles64 > 256 && a.M < 1024 && (long long)a.N * a.K > (4LL << 20);
  if (a.N >= 64 && tiles64 <= 768 && !few_rows_large_weights) {
    // (A second product whose tiles would make a fourth per CU: the next larger tiles, 1024x3072x1024 8.1 us against 7.9, and one launch less.)
    const bool larger = a.N2 > 0 && !SecondFits(kDma64x64, a.M, a.N, a.N2) && SecondFits(kDma128x64, a.M, a.N, a.N2);
    return larger ? kDma128x64 : kDma64x64;
  }
  if (a.M < 1024 && a.N >= 64) return kDma128x64;
  auto rounds = [&](int bm, int bn) {
    const long long tiles = (long long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    return (double)((tiles + 255) / 256);
  };
  const double r128 = rounds(256, 128), rs = rounds(128, 128);
  const double c256 = rounds(256, 256) * 256 * 256 * 0.60;
  const double c192 = rounds(256, 192) * 256 * 192 * 0.61;
  const double c128 = r128 * 256 * 128 * 0.84;   // 96 KiB of LDS: one workgroup per CU
  const double cs = rs * 128 * 128 * (rs > 1 ? 0.75 : 0.95);
  GemmVariant best = kDma256x256;
  double cost = c256;
  if (c192 < cost) { best = kDma256x192; cost = c192; }
  if (c128 < cost) { best = kDma256x128; cost = c128; }
  if (cs < cost) { best = kDma128x128; cost = cs; }
  const double tiles128x64 = (double)((a.M + 127) / 128) * ((a.N + 63) / 64);
  const double c64 = std::max(1.0, tiles128x64 / 256.0) * 128 * 64 * 0.80;
  if (c64 < cost) { best = kDma128x64; cost = c64; }
  return best;
}
}  // namespace

bool GemmF8TakesSecond(const GemmF8Args& a) {
  return !a.out_f8 && a.N2 % 4 == 0 && a.ldw2 % 16 == 0 && a.ldc2 % 4 == 0 && SecondFits(PickGemmF8Variant(a), a.M, a.N, a.N2);
}

const char* GemmF8VariantName(const GemmF8Args& a) {
  switch (PickGemmF8Variant(a)) {
    case kDma256x256: return "gemm_f8_256x256x128";
    case kDma256x192: return "gemm_f8_256x192x128";
    case kDma256x128: return "gemm_f8_256x128x128";
    case kDma128x64: return "gemm_f8_128x64x128";
    case kRowPanel: return "gemm_f8_rowpanel";
    case kDma64x64: return "gemm_f8_64x64x128";
    default: return "gemm_f8_128x128x128";
  }
}

void LaunchGemmF8(const GemmF8Args& a, hipStream_t stream) {
  if (a.M <= 0 || a.N <= 0) return;
  if (a.N2 > 0 && !GemmF8TakesSecond(a)) throw std::runtime_error("LaunchGemmF8: no kernel with a second product for this shape");
  const GemmVariant v = PickGemmF8Variant(a);
  if (v == kRowPanel) LaunchGemmF8RowPanel(a, stream);
  else LaunchGemmDmaF8(v, a, stream);
}

}  // namespace lc0mi
