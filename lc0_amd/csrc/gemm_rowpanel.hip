// Matrix products with few rows or few columns: row panels with the reduction split over the waves of a workgroup.
#include "gemm_variants.h"
#include "kernel_common.h"
#include "row_panel.h"

#include <type_traits>

namespace lc0mi {

namespace {

// The smallest panel (in operand rows a workgroup reads) with which the problem still fits into one workgroup per
// CU; the largest one otherwise (64x1024x1024: 4.4 us in 256 panels of 16x16, 4.9 in 64 of 32x32; 64x3072x1024: 5.6 in
// 192 panels of 32x32, 7.7 in 768 of 16x16).
inline RowPanelShape PickRowPanelShape(int M, int N, int batch) {
  for (const RowPanelShape& c : kRowPanelShapes) {
    if (RowPanelWorkgroups(M, N, batch, c) <= kRowPanelWorkgroups) return c;
  }
  return kRowPanelShapes[4];
}

// ---------------------------------------------------------------------------
// Row-panel GEMM for small problems (few rows, or few columns): a workgroup owns a
// 16 RT x 16 CT output panel and its KS waves split the reduction dimension, so even a 16 x 16 x K problem keeps KS waves busy. Such problems are bound
// by memory latency and by the rate at which a CU's address path takes operand loads,
// not by arithmetic: fragments go from global memory straight into registers, 64 bytes
// of a row per four lanes (row_panel.h), a whole share of K in flight at once when it is
// one or two steps; the partial sums are added in wave order through LDS, so results do
// not depend on timing.
// ---------------------------------------------------------------------------
template <typename ET, int RT, int CT, int KS, typename OutT, typename Args, bool TWO>
__global__ __launch_bounds__(64 * KS) void gemm_rowpanel_kernel(Args p) {
  constexpr bool F8 = std::is_same<ET, uint8_t>::value;
  constexpr int ES = F8 ? 1 : 2;
  constexpr int ROWS = 16 * RT, COLS = 16 * CT, NT = 64 * KS, LD = COLS + 4;
  __shared__ __attribute__((aligned(16))) float part[KS][ROWS * LD];
  const int tid = threadIdx.x, lane = tid & 63;
  const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // With TWO panels past the columns of the first product belong to a second one.
  const int panels = TWO ? (p.N + COLS - 1) / COLS : 0;
  const int2 tile = TileOfWorkgroup(p.tile_order);
  const bool second = TWO && tile.y >= panels;
  const int m0 = tile.x * ROWS, n0 = (second ? tile.y - panels : tile.y) * COLS;
  const int M = p.M, N = second ? p.N2 : p.N, ldw = second ? p.ldw2 : p.ldw;
  const char* A = reinterpret_cast<const char*>(p.A) + (long long)m0 * p.lda * ES;
  const char* W = (second ? reinterpret_cast<const char*>(p.W2) : reinterpret_cast<const char*>(p.W)) + (long long)n0 * ldw * ES;
  if constexpr (!F8) {
    A += (long long)blockIdx.z * p.strideA * ES;
    W += (long long)blockIdx.z * p.strideW * ES;
  }
  TileOffsets ta[RT], tw[CT];
#pragma unroll
  for (int t = 0; t < RT; t++) ta[t].Set(16 * t, M - m0, ES * p.lda);
#pragma unroll
  for (int c = 0; c < CT; c++) tw[c].Set(16 * c, N - n0, ES * ldw);
  floatx4 acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // A contiguous share of the steps per wave.
  const int row_bytes = ES * p.K, steps = (row_bytes + kStepBytes - 1) / kStepBytes, per_wave = (steps + KS - 1) / KS;
  const int s_begin = min(steps, ks * per_wave), s_end = min(steps, s_begin + per_wave);
  PanelProducts<RT, CT>(A, ta, W, tw, row_bytes, s_begin, s_end, acc, PanelOp<ET>{});
  // Accumulator lane (r, g) of tile (t, c): row 16 t + r, columns 16 c + 4 g + e.
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++)
      *reinterpret_cast<floatx4*>(&part[ks][(16 * t + r) * LD + 16 * c + 4 * g]) = acc[t][c];
  __syncthreads();
  if (second) {   // (an epilogue of its own: neither bias nor activation, and e4m3 output with e4m3 operands)
#pragma unroll
    for (int i = 0; i < (ROWS * COLS + NT - 1) / NT; i++) {
      const int idx = tid + NT * i, row = idx / COLS, col = idx % COLS;
      const int m = m0 + row, n = n0 + col;
      if (row >= ROWS || m >= M || n >= N) continue;
      float sum = part[0][row * LD + col];
#pragma unroll
      for (int w = 1; w < KS; w++) sum += part[w][row * LD + col];
      if constexpr (F8) {
        reinterpret_cast<uint8_t*>(p.C2)[(long long)m * p.ldc2 + n] =
            (uint8_t)(PackFp8x4(sum * p.col_scale2[n] * p.out_mul2, 0.0f, 0.0f, 0.0f) & 0xFFu);
      } else if constexpr (sizeof(OutT) == 2) {
        reinterpret_cast<OutT*>(p.C2)[(long long)m * p.ldc2 + n] = (OutT)sum;
      }
    }
    return;
  }
  OutT* C = reinterpret_cast<OutT*>(p.C);
  if constexpr (!F8) C += (long long)blockIdx.z * p.strideC;
  DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
    for (int i = 0; i < (ROWS * COLS + NT - 1) / NT; i++) {
      const int idx = tid + NT * i;        // consecutive threads along n
      const int row = idx / COLS, col = idx % COLS;
      const int m = m0 + row, n = n0 + col;
      if (row < ROWS && m < M && n < N) {
        float sum = part[0][row * LD + col];
#pragma unroll
        for (int w = 1; w < KS; w++) sum += part[w][row * LD + col];
        const float bias = p.bias ? p.bias[n] : 0.0f;
        if constexpr (F8) {
          const float v = act_fn(sum * p.col_scale[n] + bias);
          if constexpr (sizeof(OutT) == 1) {
            C[(long long)m * p.ldc + n] = (uint8_t)(PackFp8x4(v * p.out_mul, 0.0f, 0.0f, 0.0f) & 0xFFu);
          } else {
            C[(long long)m * p.ldc + n] = (OutT)v;
          }
        } else {
          sum *= p.scale;
          if (p.row_stats != nullptr) {   // consumer side of a folded layer norm
            float mean, rstd;
            RowMeanRstd(p.row_stats, p.row_parts, m, p.norm_n, p.norm_eps, mean, rstd);
            sum = rstd * (sum - mean * p.col_c[n]);
          }
          C[(long long)m * p.ldc + n] = (OutT)act_fn(sum + bias);
        }
      }
    }
  });
}

// Waves that share the reduction: eight steps of 128 values (K = 1024) for the 16-bit types; e4m3 steps hold twice as
// many. (Four waves are as fast at 64x1024x1024 and 64x256x2048, two at K = 256; one count serves all.)
template <typename ET> constexpr int kPanelWaves = std::is_same<ET, uint8_t>::value ? 4 : 8;

template <typename ET, typename OutT, typename Args>
void LaunchPanel(const Args& args, int batch, hipStream_t stream) {
  Args a = args;
  const RowPanelShape s = PickRowPanelShape(a.M, a.N, batch);
  auto launch = [&](auto rt_tag, auto ct_tag) {
    constexpr int RT = decltype(rt_tag)::value, CT = decltype(ct_tag)::value, KS = kPanelWaves<ET>;
    dim3 grid((a.M + 16 * RT - 1) / (16 * RT), (a.N + 16 * CT - 1) / (16 * CT) + (a.N2 + 16 * CT - 1) / (16 * CT), batch);
    a.tile_order = PickTileOrder(a.M, 1024, grid);
    if constexpr (sizeof(OutT) == 2) {
      if (a.N2 > 0) {
        hipLaunchKernelGGL((gemm_rowpanel_kernel<ET, RT, CT, KS, OutT, Args, true>), grid, dim3(64 * KS), 0, stream, a);
        return;
      }
    }
    hipLaunchKernelGGL((gemm_rowpanel_kernel<ET, RT, CT, KS, OutT, Args, false>), grid, dim3(64 * KS), 0, stream, a);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (s.rt == 1 && s.ct == 1) launch(One{}, One{});
  else if (s.rt == 2 && s.ct == 1) launch(Two{}, One{});
  else if (s.rt == 1 && s.ct == 2) launch(One{}, Two{});
  else if (std::is_same<ET, uint8_t>::value || s.rt == 2) launch(Two{}, Two{});
  else launch(std::integral_constant<int, std::is_same<ET, uint8_t>::value ? 2 : 4>{}, Two{});
}
}  // namespace

void LaunchGemmRowPanel(const GemmArgs& a, hipStream_t stream) {
  if (a.bf16) {
    if (a.out_f32) LaunchPanel<bf16_t, float>(a, a.batch, stream);
    else LaunchPanel<bf16_t, bf16_t>(a, a.batch, stream);
  } else if (a.out_f32) {
    LaunchPanel<half_t, float>(a, a.batch, stream);
  } else {
    LaunchPanel<half_t, half_t>(a, a.batch, stream);
  }
}

void LaunchGemmF8RowPanel(const GemmF8Args& a, hipStream_t stream) {
  if (a.out_f8) LaunchPanel<uint8_t, uint8_t>(a, 1, stream);
  else LaunchPanel<uint8_t, half_t>(a, 1, stream);
}

}  // namespace lc0mi
