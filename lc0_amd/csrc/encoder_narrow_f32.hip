// Encoder layers of narrow attention bodies (embedding of 128 or 256) in floats, in two kernels instead of seven, on the bfloat16
// matrix instructions (split_bf16.h). The 16-bit kernels for the same layers are in encoder_narrow.hip.
//
//   qkv_attention_f32_kernel   Q/K/V projection and attention       blas/network_blas.cc:352-439
//   encoder_tail_f32_kernel    output projection, layer norm with skip, FFN, layer norm with skip
//                                                                   blas/network_blas.cc:441-486, blas/encoder.h:29-66
#include "split_bf16.h"

#include <algorithm>
#include <stdexcept>

namespace lc0mi {

namespace {

// Weights come as 1 KiB fragments of 32 outputs x 16 inputs of one part (lane l: output l % 32, inputs 8 (l / 32) .. + 7), in the order
// in which a wave multiplies them. Rows lie in LDS as [part][column], padded so that the 16-byte reads of 16 rows meet different
// banks.

// ---------------------------------------------------------------------------
// Attention with its projection: a workgroup computes Q, K and V of one position and one or two heads of depth 32 (64 x 96 outputs
// each) and their attention, which stay in LDS. Projection: wave (share of the inputs, head, row tile) multiplies 32 rows by the 96
// columns of its head; the shares are exchanged through LDS. Attention as attention_f32_kernel, 16 queries of a head per wave.
// Bound by latency (16 KiB of rows and 74 KiB of weights per position and head: 6.7 k of a wave's 21.6 k cycles are products) up to one
// round, then by the products: 20 positions of 8 heads 11 us, where projection and attention on their own took 15.6.
// ---------------------------------------------------------------------------
template <int C, int HEADS>
__global__ __launch_bounds__(512, 1) void qkv_attention_f32_kernel(const float* __restrict__ x, const intx4* __restrict__ packed,
                                                                   const float* __restrict__ bias, float* __restrict__ out,
                                                                   int d_model, float scale) {
  constexpr int KW = 4 / HEADS, S = C / 16, SH = S / KW, LD = kParts * C + 8, V4 = 64 * (C / 4) / 512, kRing = 2, LQ = 36;
  __shared__ __attribute__((aligned(16))) bf16_t rows[64 * LD];
  __shared__ __attribute__((aligned(16))) float heads[HEADS][3][64 * LQ];
  // Sums go to the wave that ends them, 12 / KW vectors to each: in the place of the rows where they fit.
  constexpr int N = 4 / KW, kExchange = 8 * (KW - 1) * 3 * N * 64;
  constexpr bool kOwn = kExchange * sizeof(floatx4) > sizeof(rows);
  __shared__ floatx4 own[kOwn ? kExchange : 1];
  floatx4* exchange = kOwn ? own : reinterpret_cast<floatx4*>(rows);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rt = wave & 1, hd = (wave >> 1) % HEADS, kh = wave / (2 * HEADS);
  const long long row0 = (long long)blockIdx.y * 64;
  const int head0 = blockIdx.x * HEADS;

  floatx4 xv[V4];
  const floatx4* xs = reinterpret_cast<const floatx4*>(x + row0 * C);
#pragma unroll
  for (int i = 0; i < V4; i++) xv[i] = xs[i * 512 + tid];
  const intx4* ws = packed + ((long long)(head0 + hd) * S + kh * SH) * (3 * kParts * 64) + lane;
  intx4 w[kRing][3][kParts];
  auto load_weights = [&](int slot, int s) {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int f = 0; f < kParts; f++) w[slot][c][f] = ws[((s * 3 + c) * kParts + f) * 64];
  };
#pragma unroll
  for (int s = 0; s < kRing; s++) load_weights(s, s);
  const int r = lane & 31, g = lane >> 5;
  // This wave ends elements 8 (N kh + i) + 4 g .. + 3, i < N, of its head's Q, K and V.
  floatx4 b[3][N] = {};
  if (bias != nullptr) {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int i = 0; i < N; i++)
        b[c][i] = *reinterpret_cast<const floatx4*>(bias + c * d_model + (head0 + hd) * 32 + 8 * (N * kh + i) + 4 * g);
  }
#pragma unroll
  for (int i = 0; i < V4; i++) {
    const int at = i * 512 + tid, row = at / (C / 4), v = at % (C / 4);
    bf16x4 part[kParts];
    Split3(xv[i], part);
#pragma unroll
    for (int f = 0; f < kParts; f++) *reinterpret_cast<bf16x4*>(rows + row * LD + f * C + 4 * v) = part[f];
  }
  __syncthreads();

  floatx16 hi[3] = {}, lo[3] = {};
  {
    intx4 a[2][kParts];
    auto read = [&](int s) {
#pragma unroll
      for (int f = 0; f < kParts; f++)
        a[s & 1][f] = *reinterpret_cast<const intx4*>(rows + (32 * rt + r) * LD + f * C + 16 * (kh * SH + s) + 8 * g);
    };
    read(0);
#pragma unroll
    for (int s = 0; s < SH; s++) {
      if (s + 1 < SH) read(s + 1);
#pragma unroll
      for (int i = 0; i < kProducts; i++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
          floatx16& acc = i + 1 < kProducts ? lo[c] : hi[c];
          acc = Mfma32(__builtin_bit_cast(bf16x8, w[s % kRing][c][kFirst[i]]), __builtin_bit_cast(bf16x8, a[s & 1][kSecond[i]]), acc);
        }
      if (s + kRing < SH) load_weights(s % kRing, s + kRing);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();   // (the rows are not read again)
  auto sums = [&](int c, int n) {
    floatx4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = SumOfProducts(hi[c][4 * n + e], lo[c][4 * n + e]);
    return v;
  };
  floatx4 mine[3][N];
#pragma unroll
  for (int to = 0; to < KW; to++) {   // (of the waves of this head and row tile)
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int i = 0; i < N; i++) {
        const floatx4 v = sums(c, N * to + i);
        if (to == kh) mine[c][i] = v;
        else exchange[(((to * 2 * HEADS + hd * 2 + rt) * (KW - 1) + (kh < to ? kh : kh - 1)) * 3 * N + N * c + i) * 64 + lane] = v;
      }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int i = 0; i < N; i++) {
      floatx4 v = mine[c][i];
#pragma unroll
      for (int from = 0; from < KW - 1; from++) v += exchange[(((kh * 2 * HEADS + hd * 2 + rt) * (KW - 1) + from) * 3 * N + N * c + i) * 64 + lane];
      *reinterpret_cast<floatx4*>(&heads[hd][c][(32 * rt + r) * LQ + 8 * (N * kh + i) + 4 * g]) = v + b[c][i];
    }
  __syncthreads();

  if (wave < 4 * HEADS) {
    const int head = wave >> 2, r = lane & 15, g = lane >> 4, q = 16 * (wave & 3) + r;
    const float *Q = heads[head][0], *K = heads[head][1], *Vs = heads[head][2];
    floatx4 st[4];   // keys 16 t + 4 g + e of query q
#pragma unroll
    for (int t = 0; t < 4; t++) st[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const floatx4 qf = *reinterpret_cast<const floatx4*>(&Q[q * LQ + 16 * c + 4 * g]);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const floatx4 kf = *reinterpret_cast<const floatx4*>(&K[(16 * t + r) * LQ + 16 * c + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; e++) st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[e], st[t], 0, 0, 0);
      }
    }
    float mx = -3.0e38f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        st[t][e] *= scale;
        mx = fmaxf(mx, st[t][e]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        st[t][e] = expf(st[t][e] - mx);
        sum += st[t][e];
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    floatx4 o[2] = {};
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int d = 0; d < 2; d++)
          o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(Vs[(16 * t + 4 * g + e) * LQ + 16 * d + r], st[t][e], o[d], 0, 0, 0);
    float* dst = out + (row0 + q) * d_model + (head0 + head) * 32 + 4 * g;
#pragma unroll
    for (int d = 0; d < 2; d++) {
      floatx4 v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = o[d][e] / sum;
      *reinterpret_cast<floatx4*>(dst + 16 * d) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// The rest of the layer: u = LN1(alpha (att . dense + b) + x), x <- LN2(alpha (act(u . ffn1 + b1) . ffn2 + b2) + u). A workgroup owns
// 32 rows; its waves share the columns of every product (32 each of the C that are in work at a time) and stream the layer's
// weights once, from L2, kRing steps of 16 inputs ahead. Activations stay in LDS as their three parts, that is, exactly.
// With few rows several workgroups share the FFN's hidden columns; each leaves its sums to encoder_tail_sum_kernel.
// Bound by the products (55 k cycles at width 256 and 1024 hidden columns, as many as the 3.5 MB of weights take at 64 bytes a cycle, for one
// workgroup per row; with four that share the FFN 18.4 k of a wave's 40.7 k, counted) and by what lies between them, norms, activations
// and splits. us for 20 positions of a 10x256 body: five
// launches on the float instructions 40, this with one workgroup per row 42, with four that share its FFN and the launch after it 23.
// ---------------------------------------------------------------------------
template <int C>
__global__ __launch_bounds__(2 * C, 1) void encoder_tail_f32_kernel(EncoderTailArgs p) {
  constexpr int NW = C / 32, NT = 64 * NW, S = C / 16, R = 32, LD = kParts * C + 8, kRing = 4, V = R * (C / 4) / NT;
  __shared__ __attribute__((aligned(16))) bf16_t u_lds[R * LD];        // rows after the first norm
  __shared__ __attribute__((aligned(16))) bf16_t h_lds[2][R * LD];     // C columns of the attention output, then of the FFN
  __shared__ float2 moments[2][NW][R];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  const long long row0 = (long long)blockIdx.x * R;
  const int col = wave * 32 + 4 * g;                                   // of this lane's four, + 8 n
  const int att_parts = p.d_model / C, ffn_parts = p.dff / C;
  const int slice = blockIdx.y, slices = gridDim.y;                    // this workgroup's part of the FFN: of [f0, f1)
  const int f0 = slice * ffn_parts / slices, f1 = (slice + 1) * ffn_parts / slices;

  // C columns of the attention output into LDS.
  floatx4 av[V];
  auto load_att = [&](int part) {
    const float* att = reinterpret_cast<const float*>(p.att) + part * C;
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int at = i * NT + tid;
      av[i] = *reinterpret_cast<const floatx4*>(att + (row0 + at / (C / 4)) * p.d_model + at % (C / 4) * 4);
    }
  };
  auto store4 = [&](bf16_t* dst, const floatx4& v) {
    bf16x4 part[kParts];
    Split3(v, part);
#pragma unroll
    for (int f = 0; f < kParts; f++) *reinterpret_cast<bf16x4*>(dst + f * C) = part[f];
  };
  auto store_att = [&](bf16_t* dst) {
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int at = i * NT + tid;
      store4(dst + at / (C / 4) * LD + at % (C / 4) * 4, av[i]);
    }
  };
  load_att(0);
  // The weights of a part (C x C): kRing steps, replaced by those kRing further as they are used.
  constexpr int kStep = kParts * 64, kPart = NW * S * kStep;
  intx4 w[kRing][kParts];
  const intx4* ws = reinterpret_cast<const intx4*>(p.packed) + wave * S * kStep + lane;
#pragma unroll
  for (int s = 0; s < kRing; s++)
#pragma unroll
    for (int f = 0; f < kParts; f++) w[s][f] = ws[s * kStep + f * 64];
  // `step` parts on the next one begins (0 after the last: its own weights once more).
  auto multiply = [&](const bf16_t* rows, floatx16& hi, floatx16& lo, int step) {
    const intx4* next = ws + (long long)step * kPart;
    intx4 a[2][kParts];
    auto read = [&](int s) {
#pragma unroll
      for (int f = 0; f < kParts; f++) a[s & 1][f] = *reinterpret_cast<const intx4*>(rows + r * LD + f * C + 16 * s + 8 * g);
    };
    read(0);
#pragma unroll
    for (int s = 0; s < S; s++) {
      if (s + 1 < S) read(s + 1);
#pragma unroll
      for (int i = 0; i < kProducts; i++) {
        floatx16& acc = i + 1 < kProducts ? lo : hi;
        acc = Mfma32(__builtin_bit_cast(bf16x8, w[s % kRing][kFirst[i]]), __builtin_bit_cast(bf16x8, a[s & 1][kSecond[i]]), acc);
      }
#pragma unroll
      for (int f = 0; f < kParts; f++)
        w[s % kRing][f] = s + kRing < S ? ws[(s + kRing) * kStep + f * 64] : next[(s + kRing - S) * kStep + f * 64];
      __builtin_amdgcn_sched_barrier(0);
    }
    ws = next;
  };
  auto load4 = [&](const float* v, int at, floatx4 (&o)[4]) {
#pragma unroll
    for (int n = 0; n < 4; n++) o[n] = *reinterpret_cast<const floatx4*>(v + at + 8 * n);
  };
  // (Without a branch around loads, or behind one whether they are on their way is not known and everything is waited for. A bias that
  // is not there reads another vector and is left out where it is added.)
  auto load_bias = [&](const float* v, int at, floatx4 (&o)[4]) { load4(v != nullptr ? v : p.ln1_g, v != nullptr ? at : col, o); };
  auto add_bias = [&](const float* v, const floatx4& b, const floatx4& x) { return v != nullptr ? x + b : x; };
  auto sums = [&](const floatx16& hi, const floatx16& lo, int n) {
    floatx4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = SumOfProducts(hi[4 * n + e], lo[4 * n + e]);
    return v;
  };
  // t <- layer norm of the rows whose values t holds, over the waves.
  auto norm = [&](floatx4 (&t)[4], const floatx4 (&gamma)[4], const floatx4 (&beta)[4], float2 (&part_of)[NW][R]) {
    float mean = 0.0f, m2 = 0.0f;
#pragma unroll
    for (int n = 0; n < 4; n++) mean += (t[n][0] + t[n][1]) + (t[n][2] + t[n][3]);
    mean *= 1.0f / 16.0f;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) m2 = fmaf(t[n][e] - mean, t[n][e] - mean, m2);
    MergeMoments(mean, m2, __shfl_xor(mean, 32, 64), __shfl_xor(m2, 32, 64), 16.0f);
    if (g == 0) part_of[wave][r] = make_float2(mean, m2);
    __syncthreads();
    float means[NW], m2s[NW];
#pragma unroll
    for (int v = 0; v < NW; v++) {
      const float2 m = part_of[v][r];
      means[v] = m.x;
      m2s[v] = m.y;
    }
#pragma unroll
    for (int n = 1; n < NW; n *= 2)
#pragma unroll
      for (int v = 0; v < NW; v += 2 * n) MergeMoments(means[v], m2s[v], means[v + n], m2s[v + n], 32.0f * n);
    const float rstd = 1.0f / sqrtf(m2s[0] * (1.0f / C) + p.eps);
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) t[n][e] = beta[n][e] + gamma[n][e] * (t[n][e] - means[0]) * rstd;
  };

  // Output projection, skip and first norm.
  floatx4 bias[4], gamma[4], beta[4], t[4];
  load_bias(p.dense_b, col, bias);
  load4(p.ln1_g, col, gamma);
  load4(p.ln1_b, col, beta);
  float* x = reinterpret_cast<float*>(p.x) + (row0 + r) * C + col;
#pragma unroll
  for (int n = 0; n < 4; n++) t[n] = *reinterpret_cast<const floatx4*>(x + 8 * n);
  store_att(h_lds[0]);
  floatx16 sum_hi = {}, sum_lo = {};
  __syncthreads();
  multiply(h_lds[0], sum_hi, sum_lo, att_parts > 1 ? 1 : 1 + 2 * f0);
  for (int a = 1; a < att_parts; a++) {
    load_att(a);
    store_att(h_lds[a & 1]);
    __syncthreads();
    multiply(h_lds[a & 1], sum_hi, sum_lo, a + 1 < att_parts ? 1 : 1 + 2 * f0);
  }
#pragma unroll
  for (int n = 0; n < 4; n++) t[n] += add_bias(p.dense_b, bias[n], sums(sum_hi, sum_lo, n)) * p.alpha;
  norm(t, gamma, beta, moments[0]);
#pragma unroll
  for (int n = 0; n < 4; n++) store4(u_lds + r * LD + col + 8 * n, t[n]);
  if (slices > 1 && slice == 0) {
#pragma unroll
    for (int n = 0; n < 4; n++) *reinterpret_cast<floatx4*>(p.u + (row0 + r) * C + col + 8 * n) = t[n];
  }
  __syncthreads();

  // FFN, C of its columns at a time. (The barrier of one part also says that every wave has read the part two before.)
  sum_hi = sum_lo = floatx16{};
  load4(p.ln2_g, col, gamma);
  load4(p.ln2_b, col, beta);
  for (int f = f0; f < f1; f++) {
    load_bias(p.ffn1_b, f * C + col, bias);
    floatx16 hi = {}, lo = {};
    multiply(u_lds, hi, lo, 1);
    bf16_t* h = h_lds[f & 1];
    DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
      for (int n = 0; n < 4; n++) {
        const floatx4 v = add_bias(p.ffn1_b, bias[n], sums(hi, lo, n));
        store4(h + r * LD + col + 8 * n, floatx4{act_fn(v[0]), act_fn(v[1]), act_fn(v[2]), act_fn(v[3])});
      }
    });
    __syncthreads();
    multiply(h, sum_hi, sum_lo, f + 1 < f1 ? 1 : 0);
  }
  if (slices > 1) {
    float* sum = p.partial + ((long long)slice * p.M + row0 + r) * C + col;
#pragma unroll
    for (int n = 0; n < 4; n++) *reinterpret_cast<floatx4*>(sum + 8 * n) = sums(sum_hi, sum_lo, n);
    return;
  }
  load_bias(p.ffn2_b, col, bias);
#pragma unroll
  for (int n = 0; n < 4; n++) t[n] = add_bias(p.ffn2_b, bias[n], sums(sum_hi, sum_lo, n)) * p.alpha + Join3(u_lds + r * LD + col + 8 * n, C);
  norm(t, gamma, beta, moments[1]);
#pragma unroll
  for (int n = 0; n < 4; n++) *reinterpret_cast<floatx4*>(x + 8 * n) = t[n];
}

// x <- LN2(alpha (the slices' sums + b2) + u), one row per wave.
template <int C>
__global__ __launch_bounds__(256) void encoder_tail_sum_kernel(EncoderTailArgs p, int slices) {
  constexpr int E = C / 64;
  using Row = float __attribute__((ext_vector_type(E)));
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  auto load = [&](const float* v, long long r) { return *reinterpret_cast<const Row*>(v + r * C + E * lane); };
  Row v = load(p.partial, row);
  for (int i = 1; i < slices; i++) v += load(p.partial, (long long)i * p.M + row);
  const Row u = load(p.u, row), gamma = load(p.ln2_g, 0), beta = load(p.ln2_b, 0);
  if (p.ffn2_b != nullptr) v += load(p.ffn2_b, 0);
  v = v * p.alpha + u;
  float sum = 0.0f, m2 = 0.0f;
#pragma unroll
  for (int e = 0; e < E; e++) sum += v[e];
  const float mean = WaveSum(sum) * (1.0f / C);
#pragma unroll
  for (int e = 0; e < E; e++) m2 = fmaf(v[e] - mean, v[e] - mean, m2);
  const float rstd = 1.0f / sqrtf(WaveSum(m2) * (1.0f / C) + p.eps);
#pragma unroll
  for (int e = 0; e < E; e++) v[e] = beta[e] + gamma[e] * (v[e] - mean) * rstd;
  *reinterpret_cast<Row*>(reinterpret_cast<float*>(p.x) + row * C + E * lane) = v;
}
}  // namespace

long long QkvF32FragmentIndex(int row, int col, int emb, int d_model) {
  const int which = row / d_model, at = row % d_model;   // Q, K or V
  return (((((long long)(at / 32) * (emb / 16) + col / 16) * 3 + which) * kParts) * 64 + at % 32 + 32 * (col % 16 / 8)) * 8 + col % 8;
}

void LaunchQkvAttentionF32(const QkvAttentionArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  if (!QkvAttentionSupported(a.emb, a.heads, 32)) throw std::runtime_error("LaunchQkvAttentionF32: unsupported shape");
  auto launch = [&](auto kernel, int heads) {
    hipLaunchKernelGGL(kernel, dim3(a.heads / heads, a.batch), dim3(512), 0, stream, reinterpret_cast<const float*>(a.x),
                       reinterpret_cast<const intx4*>(a.packed), a.bias, reinterpret_cast<float*>(a.out), 32 * a.heads, a.scale);
  };
  // One head per workgroup while that is one round of the CUs, then two, which split the position's rows once. us of a 10x256 pass, one /
  // two: 1 position 407 / 444, 20 443 / 472, 32 505 / 528, 33 627 / 574, 64 762 / 704, 256 2307 / 2109.
  const bool one = a.batch * a.heads <= 256;
  if (a.emb == 256) one ? launch(qkv_attention_f32_kernel<256, 1>, 1) : launch(qkv_attention_f32_kernel<256, 2>, 2);
  else one ? launch(qkv_attention_f32_kernel<128, 1>, 1) : launch(qkv_attention_f32_kernel<128, 2>, 2);
}

long long EncoderTailF32FragmentIndex(int layer, int row, int col, int emb, int d_model) {
  // Parts of emb x emb: those of the output projection, then of the FFN's two layers in turn.
  int p = col / emb, r = row, c = col % emb;
  if (layer == 1) {
    p = d_model / emb + 2 * (row / emb);
    r = row % emb;
  } else if (layer == 2) {
    p = d_model / emb + 2 * (col / emb) + 1;
  }
  const long long step = ((long long)p * (emb / 32) + r / 32) * (emb / 16) + c / 16;
  return (step * kParts * 64 + r % 32 + 32 * (c % 16 / 8)) * 8 + c % 8;
}

// The two kernels take as long for one position as for many; us of a ten-layer pass, layers one by one -> this. Width 256, 512 hidden
// columns 6 positions 398 -> 410, 8 416 -> 414, 16 531 -> 439, 100 1643 -> 780, 1000 13027 -> 6294; 1024 4 385 -> 413, 8 462 -> 419, 20 664 ->
// 443, 64 1428 -> 704, 256 4565 -> 2103, with smolgen (this kernel only) 4 676 -> 692, 6 740 -> 721, 1000 20836 -> 13398; 2048 2 402 -> 421, 4
// 432 -> 425, 1000 26879 -> 11370. Width 128, 512 hidden columns 1 320 -> 273, 100 969 -> 444; 2048 1 367 -> 315, 1000 14003 -> 5634.
int NarrowF32MinBatch(int emb, int dff) { return emb <= 128 ? 1 : dff <= 512 ? 8 : dff <= 1024 ? 6 : 4; }

// As many as one round of the CUs has room for: they repeat the output projection and the norm, and a launch adds their sums. us of a
// 10x256 pass with up to 128, 256 and 384 workgroups: 20 positions 512, 443, 443; 33 735, 575, 753; 64 787, 704, 933; 96 937, 939, 1149.
int EncoderTailF32Slices(int M, int emb, int dff) { return std::max(1, std::min(dff / emb, 256 / (M / 32))); }

void LaunchEncoderTailF32(const EncoderTailArgs& a, hipStream_t stream) {
  if (a.M <= 0) return;
  if (!EncoderTailSupported(a.emb, a.d_model, a.dff) || a.M % 64 != 0) throw std::runtime_error("LaunchEncoderTailF32: unsupported shape");
  const int slices = EncoderTailF32Slices(a.M, a.emb, a.dff);
  const dim3 grid(a.M / 32, slices);
  if (a.emb == 256) hipLaunchKernelGGL(encoder_tail_f32_kernel<256>, grid, dim3(512), 0, stream, a);
  else hipLaunchKernelGGL(encoder_tail_f32_kernel<128>, grid, dim3(256), 0, stream, a);
  if (slices == 1) return;
  if (a.emb == 256) hipLaunchKernelGGL(encoder_tail_sum_kernel<256>, dim3(a.M / 4), dim3(256), 0, stream, a, slices);
  else hipLaunchKernelGGL(encoder_tail_sum_kernel<128>, dim3(a.M / 4), dim3(256), 0, stream, a, slices);
}

}  // namespace lc0mi
