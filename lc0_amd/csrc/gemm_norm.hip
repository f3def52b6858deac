// Dense layers of the smolgen chain that normalise their input rows themselves (few positions).
//
// Replaces LayerNorm2DWithSkipConnection without skip followed by FullyConnectedLayer::Forward1D:
// blas/network_blas.cc:310-347 (blas/encoder.h:29-66, blas/fully_connected_layer.cc:49-106).
#include "kernel_common.h"
#include "row_panel.h"

#include <cmath>
#include <stdexcept>
#include <type_traits>

namespace lc0mi {

namespace {

constexpr int kNormK = 256;        // columns of the input rows

// ---------------------------------------------------------------------------
// C[m][n] = act(sum_k norm(A)[m][k] W[n][k] + bias[n]) with rows of 256 values, `group` consecutive rows normalised
// together (1: smolgen's second dense layer, one row per position; the number of heads: the shared generator layer, whose
// input is one normalised row of heads x 256 values per position).
//
// Bound by latency. Alone, the norm of so few rows is a launch in a chain of dependent ones, 2.5 to 3 us inside a replayed
// graph, of which its 16 KiB per position take a tenth. A workgroup of the product reads whole rows anyway; so it normalises
// them on their way into LDS (the same formula and the same rounding to the element type as the kernel of its own), while
// its first weights, which do not depend on them, are in flight. us back to back, product alone -> with the norm:
// 1x8192x256 2.9 -> 3.4, 64 rows 3.5 -> 4.7; the generator layer, whose gamma and beta are 64 KiB per workgroup, 1 position
// 3.0 -> 5.2, 13 6.4 -> 7.3, 64 12.1 -> 15.8. NW waves, 16 CT columns each at a time, all of K per wave: fragments of W straight from
// memory in the order of row_panel.h, fragments of A from LDS in the same order. Column 4 CT q + 4 c + i of a wave's 16 CT
// is row 4 q + i of its weight tile c, so that a lane ends up with 4 CT neighbouring outputs.
// ---------------------------------------------------------------------------
template <typename ET, int NW, int RT, int CT, bool GROUPED>
__global__ __launch_bounds__(64 * NW) void norm_gemm_kernel(NormGemmArgs p, int groups, int blocks) {
  constexpr bool F8 = std::is_same<ET, uint8_t>::value;
  constexpr int ES = F8 ? 1 : 2, ROW = kNormK * ES, STEPS = ROW / kStepBytes, LD = ROW + 16;
  constexpr int STRIDE = 2 * NW, V = 16 * RT / STRIDE;     // 8-element vectors of A per thread: rows tid / 32 + STRIDE v
  static_assert(V >= 1, "a row for every 32 threads");
  using IT = std::conditional_t<F8, half_t, ET>;           // type of A and of C
  using iv8 = typename Vec16<IT>::v8;
  __shared__ __attribute__((aligned(16))) char rows_lds[16 * RT * LD];
  __shared__ float2 moments[16 * RT];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.x * groups * p.group;
  const int rows = min(p.M - m0, groups * p.group);        // of this workgroup: whole groups
  const int N = p.N, n_end = min(N, (int)(blockIdx.y + 1) * blocks * 16 * NW * CT);
  const char* W = reinterpret_cast<const char*>(p.W);

  // This lane's weights of the 16 CT columns at n: rows 16 CT / 16 ... in the order explained above, clamped.
  const int in_row = 64 * g + 16 * (lane & 3), q = (lane >> 2) & 3;
  auto load_w = [&](int n, intx4 (&w)[CT][STEPS][4]) {
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const char* src = W + (long long)min(n + 4 * CT * q + 4 * c + i, N - 1) * p.ldw * ES + in_row;
#pragma unroll
        for (int s = 0; s < STEPS; s++) w[c][s][i] = *reinterpret_cast<const intx4*>(src + s * kStepBytes);
      }
  };
  int n = blockIdx.y * blocks * 16 * NW * CT + wave * 16 * CT;

  // The rows, gamma and beta first (the norm waits for them), then the first weights.
  const int row0 = tid >> 5, kv = (tid & 31) * 8;
  iv8 x[V];
  floatx4 gm[GROUPED ? V : 1][2], bt[GROUPED ? V : 1][2];
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int row = min(row0 + STRIDE * v, rows - 1);
    x[v] = *reinterpret_cast<const iv8*>(p.A + (long long)(m0 + row) * kNormK + kv);
    if (GROUPED || v == 0) {
      const int at = (GROUPED ? row % p.group * kNormK : 0) + kv;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        gm[v][h] = *reinterpret_cast<const floatx4*>(p.gamma + at + 4 * h);
        bt[v][h] = *reinterpret_cast<const floatx4*>(p.beta + at + 4 * h);
      }
    }
  }
  intx4 w[CT][STEPS][4];
  load_w(n, w);

  float mean[V], m2[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) s += (float)x[v][e];
    mean[v] = s * 0.125f;
    m2[v] = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float d = (float)x[v][e] - mean[v];
      m2[v] = fmaf(d, d, m2[v]);
    }
    // Over the 32 lanes of the row: lane ^ 1, lane ^ 2, the other quad of 8, the other 8 of 16, the other 16 of 32.
    MergeMoments(mean[v], m2[v], DppMove<0xB1>(mean[v]), DppMove<0xB1>(m2[v]), 8.0f);
    MergeMoments(mean[v], m2[v], DppMove<0x4E>(mean[v]), DppMove<0x4E>(m2[v]), 16.0f);
    MergeMoments(mean[v], m2[v], DppMove<0x141>(mean[v]), DppMove<0x141>(m2[v]), 32.0f);
    MergeMoments(mean[v], m2[v], DppMove<0x140>(mean[v]), DppMove<0x140>(m2[v]), 64.0f);
    MergeMoments(mean[v], m2[v], __shfl_xor(mean[v], 16, 64), __shfl_xor(m2[v], 16, 64), 128.0f);
  }
  float rstd[V];
  if constexpr (GROUPED) {
#pragma unroll
    for (int v = 0; v < V; v++)
      if ((tid & 31) == 0) moments[row0 + STRIDE * v] = make_float2(mean[v], m2[v]);
    __syncthreads();
    // Every wave adds up every group: lane l takes row l of it (group <= 64), as differences from the mean of its row 0.
    const float inv = 1.0f / (float)p.group;
    for (int gr = 0; gr < groups && gr * p.group < rows; gr++) {
      const bool in = lane < p.group;
      const float2 m = moments[gr * p.group + (in ? lane : 0)];
      const float ref = moments[gr * p.group].x;
      float s1 = in ? m.x - ref : 0.0f, s2 = in ? fmaf((m.x - ref) * (float)kNormK, m.x - ref, m.y) : 0.0f;
      s1 += DppMove<0xB1>(s1); s2 += DppMove<0xB1>(s2);
      s1 += DppMove<0x4E>(s1); s2 += DppMove<0x4E>(s2);
      s1 += DppMove<0x141>(s1); s2 += DppMove<0x141>(s2);
      s1 += DppMove<0x140>(s1); s2 += DppMove<0x140>(s2);
      s1 += __shfl_xor(s1, 16, 64); s2 += __shfl_xor(s2, 16, 64);
      s1 += __shfl_xor(s1, 32, 64); s2 += __shfl_xor(s2, 32, 64);
      const float d = s1 * inv, mean_g = ref + d;
      const float var = fmaxf(s2 * inv * (1.0f / kNormK) - d * d, 0.0f);
      const float rs = 1.0f / sqrtf(var + p.eps);
#pragma unroll
      for (int v = 0; v < V; v++) {
        const int at = row0 + STRIDE * v - gr * p.group;
        if (at >= 0 && at < p.group) {
          mean[v] = mean_g;
          rstd[v] = rs;
        } else if (gr == 0) {
          rstd[v] = 0.0f;
        }
      }
    }
  } else {
#pragma unroll
    for (int v = 0; v < V; v++) rstd[v] = 1.0f / sqrtf(m2[v] * (1.0f / kNormK) + p.eps);
  }
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int gv = GROUPED ? v : 0;
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] = bt[gv][e / 4][e % 4] + gm[gv][e / 4][e % 4] * ((float)x[v][e] - mean[v]) * rstd[v];
    char* dst = rows_lds + (row0 + STRIDE * v) * LD + kv * ES;
    if constexpr (F8) {
      uint2 o;
      o.x = PackFp8x4(f[0] * p.in_mul, f[1] * p.in_mul, f[2] * p.in_mul, f[3] * p.in_mul);
      o.y = PackFp8x4(f[4] * p.in_mul, f[5] * p.in_mul, f[6] * p.in_mul, f[7] * p.in_mul);
      *reinterpret_cast<uint2*>(dst) = o;
    } else {
      iv8 o;
#pragma unroll
      for (int e = 0; e < 8; e++) o[e] = (IT)f[e];
      *reinterpret_cast<iv8*>(dst) = o;
    }
  }
  __syncthreads();

  IT* C = reinterpret_cast<IT*>(p.C);
  const PanelOp<ET> op;
  DispatchAct(p.act, [&](auto act_fn) {
    for (; n < n_end; n += 16 * NW * CT) {
      floatx4 acc[RT][CT];
      intx4 wt[CT][STEPS][4];
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
#pragma unroll
          for (int i = 0; i < 4; i++) wt[c][s][i] = w[c][s][i];
          QuadTranspose(wt[c][s]);
        }
      if (n + 16 * NW * CT < n_end) load_w(n + 16 * NW * CT, w);   // (while this block's products run)
#pragma unroll
      for (int t = 0; t < RT; t++) {
#pragma unroll
        for (int c = 0; c < CT; c++) acc[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
          intx4 a[4];
#pragma unroll
          for (int j = 0; j < 4; j++)
            a[j] = *reinterpret_cast<const intx4*>(rows_lds + (16 * t + r) * LD + s * kStepBytes + 64 * g + 16 * j);
#pragma unroll
          for (int c = 0; c < CT; c++) op(wt[c][s], a, acc[t][c]);
        }
      }
      const int at = n + 4 * CT * g;   // this lane's 4 CT columns
      float scale[4 * CT], bias[4 * CT];
#pragma unroll
      for (int c = 0; c < CT; c++) {
        LoadBias4(p.bias, at + 4 * c, N, bias + 4 * c);
        if constexpr (F8) LoadBias4(p.col_scale, at + 4 * c, N, scale + 4 * c);
      }
#pragma unroll
      for (int t = 0; t < RT; t++) {
        const int row = 16 * t + r;
        IT* dst = C + (long long)(m0 + row) * p.ldc + at;
        IT o[4 * CT];
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
          for (int e = 0; e < 4; e++)
            o[4 * c + e] = (IT)act_fn(F8 ? acc[t][c][e] * scale[4 * c + e] + bias[4 * c + e] : acc[t][c][e] + bias[4 * c + e]);
        if (row < rows) {   // (ldc and N are multiples of 16: whole vectors)
          if (at < N) {
            if constexpr (CT == 2) {
              *reinterpret_cast<iv8*>(dst) = iv8{o[0], o[1], o[2], o[3], o[4], o[5], o[6], o[7]};
            } else {
              using iv4 = typename Vec16<IT>::v4;
              *reinterpret_cast<iv4*>(dst) = iv4{o[0], o[1], o[2], o[3]};
            }
          }
        }
      }
    }
  });
}

// The instances: one row per position (smolgen's second dense layer), then grouped ones (the generator layer).
struct NormGemmShape { int nw, rt, ct; bool grouped; };
constexpr NormGemmShape kNormGemmShapes[] = {{4, 1, 1, false}, {4, 2, 1, false}, {4, 4, 1, false},
                                             {4, 2, 1, true}, {8, 2, 2, true}, {8, 4, 2, true}};

// The instance and the blocks of columns per workgroup with the least bytes through one CU; a workgroup's start is priced
// as 40 KiB.
int PickNormGemmShape(const NormGemmArgs& a, int* blocks_out) {
  const int es = a.f8 ? 1 : 2, all_groups = a.M / a.group;
  int best = -1;
  double cost = 0.0;
  for (int i = 0; i < 6; i++) {
    const NormGemmShape& s = kNormGemmShapes[i];
    const int groups = 16 * s.rt / a.group, cols = 16 * s.nw * s.ct;
    if (s.grouped != (a.group > 1) || groups < 1) continue;
    for (int blocks = 1; blocks <= (s.ct > 1 ? 8 : 1); blocks *= 2) {
      const double wgs = (double)((all_groups + groups - 1) / groups) * ((a.N + cols * blocks - 1) / (cols * blocks));
      const double bytes = 8.0 * a.group * kNormK + 2.0 * groups * a.group * kNormK + (double)cols * blocks * kNormK * es + 40960.0;
      const double c = bytes * std::ceil(wgs / 256.0);
      if (best < 0 || c < cost) {
        best = i;
        *blocks_out = blocks;
        cost = c;
      }
    }
  }
  return best;
}

template <typename ET>
void LaunchNormGemmT(const NormGemmArgs& a, hipStream_t stream) {
  int blocks = 1;
  const int pick = PickNormGemmShape(a, &blocks);
  auto launch = [&](auto tag) {
    constexpr NormGemmShape s = kNormGemmShapes[decltype(tag)::value];
    const int groups = 16 * s.rt / a.group, cols = 16 * s.nw * s.ct * blocks;
    const dim3 grid((a.M / a.group + groups - 1) / groups, (a.N + cols - 1) / cols);
    hipLaunchKernelGGL((norm_gemm_kernel<ET, s.nw, s.rt, s.ct, s.grouped>), grid, dim3(64 * s.nw), 0, stream, a, groups, blocks);
  };
  switch (pick) {
    case 0: return launch(std::integral_constant<int, 0>{});
    case 1: return launch(std::integral_constant<int, 1>{});
    case 2: return launch(std::integral_constant<int, 2>{});
    case 3: return launch(std::integral_constant<int, 3>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    default: return launch(std::integral_constant<int, 5>{});
  }
}
}  // namespace

bool NormGemmSupported(int K, int group, int N) { return K == kNormK && group >= 1 && group <= 64 && N % 16 == 0; }

void LaunchNormGemm(const NormGemmArgs& a, hipStream_t stream) {
  if (a.M <= 0 || a.N <= 0) return;
  if (!NormGemmSupported(a.K, a.group, a.N) || a.M % a.group != 0 || a.ldc % 16 != 0) {
    throw std::runtime_error("LaunchNormGemm: unsupported shape");
  }
  if (a.f8) LaunchNormGemmT<uint8_t>(a, stream);
  else if (a.bf16) LaunchNormGemmT<bf16_t>(a, stream);
  else LaunchNormGemmT<half_t>(a, stream);
}

}  // namespace lc0mi
