// Encoder layers of narrow attention bodies (embedding of 128 or 256) in two kernels instead of seven.
//
//   qkv_attention_kernel   Q/K/V projection and attention          blas/network_blas.cc:352-439
//   encoder_tail_kernel    output projection, layer norm with skip, FFN, layer norm with skip
//                                                                   blas/network_blas.cc:441-486, blas/encoder.h:29-66
#include "kernel_common.h"

#include <algorithm>
#include <stdexcept>
#include <type_traits>

namespace lc0mi {

namespace {

// Both kernels take their weights as 1 KiB fragments of 16 outputs x 32 inputs in the order in which a wave multiplies them
// (lane l: output l % 16, inputs 8 (l / 16) ... + 7), so that every load is one contiguous KiB and a wave's stream is
// contiguous too. That is the layout of v_mfma_f32_16x16x32's operands.

constexpr int kPad = 8;   // 16-bit values between the rows of an LDS tile: 16-byte reads of 16 rows meet different banks

// ---------------------------------------------------------------------------
// Attention with its projection: a workgroup computes Q, K and V of one position and two heads of depth 32 (64 x 192 outputs)
// and their attention, which stay in LDS. Wave w: 16 columns of each of Q, K and V (head w / 2, half w % 2 of its depth), then
// the 16 queries from 16 w of both heads. V is multiplied with its operands exchanged, so that it comes out transposed, as the
// second product wants it.
// Bound by latency and by the 130 KiB of rows and weights a workgroup reads. us back to back at width 256 (8 heads): 1 position 5.7,
// 64 6.6, 256 16.2, 1024 48 (30 GFLOP: 626 TFLOP/s).
// ---------------------------------------------------------------------------
template <typename ET, int C>
__global__ __launch_bounds__(256, 2) void qkv_attention_kernel(const half_t* __restrict__ x, const half_t* __restrict__ packed,
                                                               const float* __restrict__ bias, half_t* __restrict__ out,
                                                               int d_model, float scale) {
  using ev8 = typename Vec16<ET>::v8;
  using ev4 = typename Vec16<ET>::v4;
  constexpr int S = C / 32, LD = C + kPad, LQ = 32 + kPad, LV = 64 + kPad;
  constexpr int V8 = C / 32;   // 16-byte loads of the position's rows per thread
  constexpr int kHeads = 2 * (2 * 64 * LQ + 32 * LV);
  __shared__ __attribute__((aligned(16))) ET lds[64 * LD > kHeads ? 64 * LD : kHeads];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const long long row0 = (long long)blockIdx.y * 64;
  const int pair = blockIdx.x;

  intx4 xv[V8];
  const intx4* xs = reinterpret_cast<const intx4*>(x + row0 * C);
#pragma unroll
  for (int i = 0; i < V8; i++) xv[i] = xs[i * 256 + tid];
  intx4 w[S][3];
  const intx4* ws = reinterpret_cast<const intx4*>(packed) + ((long long)(pair * 4 + wave) * S * 3) * 64 + lane;
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int j = 0; j < 3; j++) w[s][j] = ws[(s * 3 + j) * 64];
  const int col = pair * 64 + wave * 16;   // of this wave's 16, in each of Q, K and V
  floatx4 bq = {0.0f, 0.0f, 0.0f, 0.0f}, bk = bq;
  float bv = 0.0f;
  if (bias != nullptr) {
    bq = *reinterpret_cast<const floatx4*>(bias + col + 4 * g);
    bk = *reinterpret_cast<const floatx4*>(bias + d_model + col + 4 * g);
    bv = bias[2 * d_model + col + r];
  }
#pragma unroll
  for (int i = 0; i < V8; i++) {
    const int at = i * 256 + tid;   // C / 8 vectors a row
    *reinterpret_cast<intx4*>(lds + at / (C / 8) * LD + at % (C / 8) * 8) = xv[i];
  }
  __syncthreads();

  floatx4 acc[3][4];
#pragma unroll
  for (int j = 0; j < 3; j++)
#pragma unroll
    for (int t = 0; t < 4; t++) acc[j][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < S; s++) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const ev8 a = *reinterpret_cast<const ev8*>(lds + (16 * t + r) * LD + 32 * s + 8 * g);
      acc[0][t] = Mfma16(__builtin_bit_cast(ev8, w[s][0]), a, acc[0][t]);
      acc[1][t] = Mfma16(__builtin_bit_cast(ev8, w[s][1]), a, acc[1][t]);
      acc[2][t] = Mfma16(a, __builtin_bit_cast(ev8, w[s][2]), acc[2][t]);
    }
  }
  __syncthreads();   // (the rows are not read again: their place takes the heads)
  ET* Q = lds;
  ET* K = Q + 2 * 64 * LQ;
  ET* Vt = K + 2 * 64 * LQ;
  {
    const int head = wave >> 1, d0 = (wave & 1) * 16;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      ev4 q, k, v;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        q[e] = (ET)(acc[0][t][e] + bq[e]);
        k[e] = (ET)(acc[1][t][e] + bk[e]);
        v[e] = (ET)(acc[2][t][e] + bv);
      }
      *reinterpret_cast<ev4*>(Q + (head * 64 + 16 * t + r) * LQ + d0 + 4 * g) = q;
      *reinterpret_cast<ev4*>(K + (head * 64 + 16 * t + r) * LQ + d0 + 4 * g) = k;
      *reinterpret_cast<ev4*>(Vt + (head * 32 + d0 + r) * LV + 16 * t + 4 * g) = v;
    }
  }
  __syncthreads();

#pragma unroll
  for (int head = 0; head < 2; head++) {
    const ev8 qf = *reinterpret_cast<const ev8*>(Q + (head * 64 + 16 * wave + r) * LQ + 8 * g);
    floatx4 st[4];   // keys 16 t + 4 g + e of query r
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const ev8 kf = *reinterpret_cast<const ev8*>(K + (head * 64 + 16 * t + r) * LQ + 8 * g);
      st[t] = Mfma16(kf, qf, floatx4{0.0f, 0.0f, 0.0f, 0.0f});
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
    const float kLog2e = 1.44269504f, neg_mx = -mx * kLog2e;
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        st[t][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[t][e], kLog2e, neg_mx));
        sum += st[t][e];
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / sum;
    floatx4 o[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int s = 0; s < 2; s++) {   // 32 keys: 32 s + 4 g + e and 32 s + 16 + 4 g + e
      ev8 pf;
#pragma unroll
      for (int e = 0; e < 8; e++) pf[e] = (ET)(st[2 * s + e / 4][e % 4] * inv);
#pragma unroll
      for (int dt = 0; dt < 2; dt++) {
        const ET* src = Vt + (head * 32 + 16 * dt + r) * LV + 32 * s + 4 * g;
        const ev4 lo = *reinterpret_cast<const ev4*>(src), hi = *reinterpret_cast<const ev4*>(src + 16);
        o[dt] = Mfma16(ev8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, pf, o[dt]);
      }
    }
    ET* dst = reinterpret_cast<ET*>(out) + (row0 + 16 * wave + r) * d_model + pair * 64 + head * 32 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
      *reinterpret_cast<ev4*>(dst + 16 * dt) = ev4{(ET)o[dt][0], (ET)o[dt][1], (ET)o[dt][2], (ET)o[dt][3]};
  }
}

// ---------------------------------------------------------------------------
// The rest of the layer: u = LN1(alpha (att . dense + b) + x), x <- LN2(alpha (act(u . ffn1 + b1) . ffn2 + b2) + u). A
// workgroup owns 16 RT rows; its eight waves share the columns of every product (16 CT each of the C = 128 CT that are in
// work at a time) and stream the layer's weights once, from L2, a whole product of C x C ahead in registers. Activations
// stay in LDS in 16 bits, sums and norms in float.
// Bound by the weight stream (1.18 MB at width 256, d_model 256 and 1024 hidden columns; a CU takes 64 bytes per cycle from L2,
// here 88 GB/s per CU) up to 32 rows per workgroup, with 64 rows by that, the matrix cores and the LDS reads alike. us back to back at
// that width: 16 rows on 4 CUs 13.3, on 256 CUs 16.3; 32 rows on 256 CUs 19.8; 64 rows on 256 CUs 27.9 = 690 TFLOP/s. A pass
// of the 10x256 net, seven kernels per layer -> these two: 16 positions 389 -> 305, 64 477 -> 330, 256 926 -> 526, 1024 2687 -> 1690
// (below five positions: EncoderTailMinBatch); of ten layers of width 128 (4 heads, 512 hidden columns) 1 361 -> 209, 64 452 -> 250, 256
// 740 -> 471, 1000 1946 -> 1270, with smolgen, where only this kernel is used, 64 654 -> 497, 1000 3721 -> 3166; width 256 with smolgen
// 64 712 -> 606, 1000 4986 -> 4216. One launch at a width of 512 or more would stream more bytes through every CU than the separate products take.
// ---------------------------------------------------------------------------
template <typename ET, int CT, int RT, int SPLIT>
__global__ __launch_bounds__(512) void encoder_tail_kernel(EncoderTailArgs p) {
  using ev8 = typename Vec16<ET>::v8;
  using ev4 = typename Vec16<ET>::v4;
  constexpr int C = 128 * CT, S = C / 32, R = 16 * RT, LD = C + kPad;
  constexpr int VECS = R * C / 8, V = (VECS + 511) / 512;
  __shared__ __attribute__((aligned(16))) ET u_lds[R * LD];        // rows after the first norm
  __shared__ __attribute__((aligned(16))) ET h_lds[2][R * LD];     // C columns of the attention output, then of the FFN
  __shared__ float2 moments[2][8][R];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int block = blockIdx.x / SPLIT, slice = blockIdx.x % SPLIT;
  const long long row0 = (long long)block * R;
  const int col = wave * 16 * CT + 4 * g;                          // of this lane's four, + 16 c
  const int att_parts = p.d_model / C, ffn_begin = slice * (p.dff / C) / SPLIT, ffn_end = (slice + 1) * (p.dff / C) / SPLIT;
  const int parts = att_parts + 2 * (ffn_end - ffn_begin);

  // C columns of the attention output into LDS.
  intx4 av[V];
  auto load_att = [&](int part) {
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int at = min(i * 512 + tid, VECS - 1);
      av[i] = *reinterpret_cast<const intx4*>(p.att + (row0 + at / (C / 8)) * p.d_model + part * C + at % (C / 8) * 8);
    }
  };
  auto store_att = [&](ET* dst) {
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int at = i * 512 + tid;
      if (VECS % 512 == 0 || at < VECS) *reinterpret_cast<intx4*>(dst + at / (C / 8) * LD + at % (C / 8) * 8) = av[i];
    }
  };
  load_att(0);
  // The weights of one part (C x C), replaced by those of the next one as they are used.
  intx4 w[S][CT];
  const intx4* next = reinterpret_cast<const intx4*>(p.packed) + wave * S * CT * 64 + lane;
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int c = 0; c < CT; c++) w[s][c] = next[(s * CT + c) * 64];
  int part = 0;
  floatx4 acc[RT][CT], sum[RT][CT];
  auto clear = [&](floatx4 (&a)[RT][CT]) {
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int c = 0; c < CT; c++) a[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  auto multiply = [&](const ET* rows, floatx4 (&a)[RT][CT]) {
    if (++part < parts) next += 8 * S * CT * 64 * (part == att_parts ? 1 + 2 * ffn_begin : 1);   // (after the last part its own weights once more)
    // Rows DEPTH steps ahead; the order is fixed, or the compiler gathers the loads at the end of a part, where the next part
    // waits for them.
    constexpr int DEPTH = RT == 1 ? S : RT == 2 ? S / 2 : 2;
    ev8 b[DEPTH][RT];
    auto read = [&](int s) {
#pragma unroll
      for (int t = 0; t < RT; t++) b[s % DEPTH][t] = *reinterpret_cast<const ev8*>(rows + (16 * t + r) * LD + 32 * s + 8 * g);
    };
#pragma unroll
    for (int s = 0; s < DEPTH; s++) read(s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S; s++) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CT; c++) a[t][c] = Mfma16(__builtin_bit_cast(ev8, w[s][c]), b[s % DEPTH][t], a[t][c]);
#pragma unroll
      for (int c = 0; c < CT; c++) w[s][c] = next[(s * CT + c) * 64];
      if (s + DEPTH < S) read(s + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto load4 = [&](const float* v, int at, floatx4 (&o)[CT]) {
#pragma unroll
    for (int c = 0; c < CT; c++)
      o[c] = v != nullptr ? *reinterpret_cast<const floatx4*>(v + at + 16 * c) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  // t[..] <- layer norm of the rows whose values t holds, over the eight waves.
  auto norm = [&](floatx4 (&t)[RT][CT], const floatx4 (&gamma)[CT], const floatx4 (&beta)[CT], float2 (&part_of)[8][R]) {
#pragma unroll
    for (int i = 0; i < RT; i++) {
      float mean = 0.0f, m2 = 0.0f;
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) mean += t[i][c][e];
      mean *= 1.0f / (4 * CT);
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) m2 = fmaf(t[i][c][e] - mean, t[i][c][e] - mean, m2);
      MergeMoments(mean, m2, __shfl_xor(mean, 16, 64), __shfl_xor(m2, 16, 64), 4.0f * CT);
      MergeMoments(mean, m2, __shfl_xor(mean, 32, 64), __shfl_xor(m2, 32, 64), 8.0f * CT);
      if (g == 0) part_of[wave][16 * i + r] = make_float2(mean, m2);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RT; i++) {
      float mean[8], m2[8];
#pragma unroll
      for (int v = 0; v < 8; v++) {
        const float2 m = part_of[v][16 * i + r];
        mean[v] = m.x;
        m2[v] = m.y;
      }
#pragma unroll
      for (int n = 1; n < 8; n *= 2)
#pragma unroll
        for (int v = 0; v < 8; v += 2 * n) MergeMoments(mean[v], m2[v], mean[v + n], m2[v + n], 16.0f * CT * n);
      const float rstd = 1.0f / sqrtf(m2[0] * (1.0f / C) + p.eps);
#pragma unroll
      for (int c = 0; c < CT; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) t[i][c][e] = beta[c][e] + gamma[c][e] * (t[i][c][e] - mean[0]) * rstd;
    }
  };
  auto to16 = [](const floatx4& v) { return ev4{(ET)v[0], (ET)v[1], (ET)v[2], (ET)v[3]}; };

  // Output projection, skip and first norm.
  floatx4 bias[CT], gamma[CT], beta[CT];
  ev4 skip[RT][CT];
  load4(p.dense_b, col, bias);
  load4(p.ln1_g, col, gamma);
  load4(p.ln1_b, col, beta);
  const ET* x = reinterpret_cast<const ET*>(p.x) + row0 * C;
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) skip[t][c] = *reinterpret_cast<const ev4*>(x + (16 * t + r) * C + col + 16 * c);
  store_att(h_lds[0]);
  clear(sum);
  for (int a = 0; a < att_parts; a++) {
    if (a + 1 < att_parts) load_att(a + 1);
    __syncthreads();
    multiply(h_lds[a & 1], sum);
    if (a + 1 < att_parts) store_att(h_lds[(a + 1) & 1]);
  }
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
      for (int e = 0; e < 4; e++) sum[t][c][e] = (sum[t][c][e] + bias[c][e]) * p.alpha + (float)skip[t][c][e];
  norm(sum, gamma, beta, moments[0]);
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) {
      *reinterpret_cast<ev4*>(u_lds + (16 * t + r) * LD + col + 16 * c) = to16(sum[t][c]);
    }
  __syncthreads();

  // FFN, C of its columns at a time. (The barrier of one part also says that every wave has read the part two before.)
  clear(sum);
  load4(p.ln2_g, col, gamma);
  load4(p.ln2_b, col, beta);
  for (int f = ffn_begin; f < ffn_end; f++) {
    load4(p.ffn1_b, f * C + col, bias);
    clear(acc);
    multiply(u_lds, acc);
    ET* h = h_lds[f & 1];
    DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CT; c++) {
          floatx4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = act_fn(acc[t][c][e] + bias[c][e]);
          *reinterpret_cast<ev4*>(h + (16 * t + r) * LD + col + 16 * c) = to16(v);
        }
    });
    __syncthreads();
    multiply(h, sum);
  }
  if constexpr (SPLIT > 1) {
    // Every slice leaves its sums, written through to memory; the last one of the block to arrive adds all of them, in the order of
    // the slices whoever that is, and goes on. Nobody waits for another workgroup. (The counter is relaxed and no release fence precedes it:
    // stores at device scope, which pass by the L2 of their XCD, and the wait for them before the barrier and the count take its place.
    // Ordinary or streaming stores would not do here.)
    __shared__ int last;
    floatx4* place = reinterpret_cast<floatx4*>(p.partial) + (long long)block * SPLIT * RT * CT * 512 + tid;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int c = 0; c < CT; c++) StoreThrough16(place + ((slice * RT + t) * CT + c) * 512, __builtin_bit_cast(intx4, sum[t][c]));
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __syncthreads();
    if (tid == 0) {
      last = __hip_atomic_fetch_add(p.arrived + block, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == SPLIT - 1;
      if (last) __hip_atomic_store(p.arrived + block, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (for the next launch)
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    if (!last) return;
    floatx4 other[SPLIT][RT][CT];
#pragma unroll
    for (int j = 0; j < SPLIT; j++)
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CT; c++)
          other[j][t][c] = place[((j * RT + t) * CT + c) * 512];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int c = 0; c < CT; c++) {
        sum[t][c] = other[0][t][c];
#pragma unroll
        for (int j = 1; j < SPLIT; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) sum[t][c][e] += other[j][t][c][e];
      }
  }
  load4(p.ffn2_b, col, bias);
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) {
      const ev4 u = *reinterpret_cast<const ev4*>(u_lds + (16 * t + r) * LD + col + 16 * c);
#pragma unroll
      for (int e = 0; e < 4; e++) sum[t][c][e] = (sum[t][c][e] + bias[c][e]) * p.alpha + (float)u[e];
    }
  norm(sum, gamma, beta, moments[1]);
  ET* y = reinterpret_cast<ET*>(p.x) + row0 * C;
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) *reinterpret_cast<ev4*>(y + (16 * t + r) * C + col + 16 * c) = to16(sum[t][c]);
}

template <typename ET, int CT>
void LaunchTailT(const EncoderTailArgs& a, hipStream_t stream) {
  const EncoderTailShape shape = PickEncoderTailShape(a.M, a.emb, a.dff);
  auto launch = [&](auto rt_tag, auto split_tag) {
    constexpr int RT = decltype(rt_tag)::value, SPLIT = decltype(split_tag)::value;
    hipLaunchKernelGGL((encoder_tail_kernel<ET, CT, RT, SPLIT>), dim3(a.M / (16 * RT) * SPLIT), dim3(512), 0, stream, a);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  using Four = std::integral_constant<int, 4>;
  if constexpr (CT == 2) {   // (slices at width 256 only, with 16 rows each)
    if (shape.slices == 4) return launch(One{}, Four{});
    if (shape.slices == 2) return launch(One{}, Two{});
  }
  if (shape.rows == 16) launch(One{}, One{});
  else if (shape.rows == 32) launch(Two{}, One{});
  else launch(Four{}, One{});
}

template <typename ET>
void LaunchQkvAttentionT(const QkvAttentionArgs& a, hipStream_t stream) {
  const dim3 grid(a.heads / 2, a.batch);
  if (a.emb == 256) {
    hipLaunchKernelGGL((qkv_attention_kernel<ET, 256>), grid, dim3(256), 0, stream, a.x, a.packed, a.bias, a.out, 32 * a.heads, a.scale);
  } else {
    hipLaunchKernelGGL((qkv_attention_kernel<ET, 128>), grid, dim3(256), 0, stream, a.x, a.packed, a.bias, a.out, 32 * a.heads, a.scale);
  }
}
}  // namespace

bool QkvAttentionSupported(int emb, int heads, int depth) {
  return (emb == 128 || emb == 256) && depth == 32 && heads > 0 && heads % 2 == 0;
}

long long QkvFragmentIndex(int row, int col, int emb, int d_model) {
  const int which = row / d_model, at = row % d_model;   // Q, K or V
  const int tile = at / 16;                              // four per pair of heads, one per wave
  return ((((long long)tile * (emb / 32) + col / 32) * 3 + which) * 64 + at % 16 + 16 * (col % 32 / 8)) * 8 + col % 8;
}

void LaunchQkvAttention(const QkvAttentionArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  if (!QkvAttentionSupported(a.emb, a.heads, 32)) throw std::runtime_error("LaunchQkvAttention: unsupported shape");
  if (a.bf16) LaunchQkvAttentionT<bf16_t>(a, stream);
  else LaunchQkvAttentionT<half_t>(a, stream);
}

bool EncoderTailSupported(int emb, int d_model, int dff) {
  return (emb == 128 || emb == 256) && d_model > 0 && d_model % emb == 0 && dff > 0 && dff % emb == 0;
}

// 16 rows per workgroup while they all fit the CUs, else 32, else 64: a workgroup takes the weights through its CU once
// whatever its rows, so more of them per workgroup cost nothing until their products take longer than the stream. Where that leaves
// half of the CUs without work, four or two workgroups (SPLIT) share the FFN of their rows: each takes that much less of the weights, and
// leaving and adding the sums costs about 3 us, the time of 0.3 MB. us of a ten-layer pass of width 256 with 1024 hidden columns, alone ->
// shared: by four 5 positions 312 -> 263, 8 312 -> 268, by two 16 318 -> 297. By four up to 16 positions (293) and by two up to 28 (330 -> 321) a
// pass alone is faster still, but four threads together lose 10 % (16 positions 127k -> 112k evals/s; as it is 123k -> 125k). With 32 rows per
// workgroup and two slices 64 positions 360 -> 377. Parts of width 128 are a quarter as large: not there.
EncoderTailShape PickEncoderTailShape(int M, int emb, int dff) {
  if (emb == 256) {
    if (M <= 8 * 64 && dff >= 4 * emb) return {16, 4};
    if (M <= 16 * 64 && dff >= 2 * emb) return {16, 2};
  }
  return {M <= 16 * 256 ? 16 : M <= 32 * 256 ? 32 : 64, 1};
}

// A few workgroups stream all weights through one CU each, whatever the batch, where five launches spread them over the chip;
// how many positions that costs follows from their bytes. us of a ten-layer pass, layers one by one -> the kernel with one workgroup per
// row. Width 256, 0.66 MB (512 hidden columns) 1 position 275 -> 255; 1.2 MB (1024) 1 287 -> 304, 4 302 -> 311, 8 341 -> 310, with
// smolgen 1 440 -> 453, 4 463 -> 469, 8 559 -> 522; 2.2 MB (2048) 1 305 -> 406, 12 392 -> 411, 16 386 -> 410, 24 460 -> 418. Width 128, whose
// own products have short reductions, 0.3 MB 1 292 -> 200, 1.1 MB (2048) 1 330 -> 319, 16 378 -> 329.
// Where workgroups share the FFN the kernel is ahead below this line too for one thread and for two, and from 3 positions for four threads,
// unless there is smolgen: 1024 1 252 -> 232, 3 278 -> 239, 4 281 -> 240, with smolgen 1 447 -> 415, 4 484 -> 436; 2048 1 281 -> 262, 4 332 -> 268, 8
// 362 -> 272, 16 393 -> 323; thousands of evals/s of four threads 1024 1 9.4 -> 8.7, 3 25.1 -> 25.3, 4 31.5 -> 32.2, with smolgen 1 5.4 -> 4.7, 4
// 17.9 -> 18.0; 2048 1 8.5 -> 7.9, 4 28.5 -> 28.7, 16 80 -> 90, with smolgen 4 17.8 -> 17.0, 12 38.7 -> 34.0. The line is that of one workgroup
// per row all the same.
int EncoderTailMinBatch(int emb, int d_model, int dff) {
  const int kib = 2 * emb * (d_model + 2 * dff) / 1024;
  return emb <= 128 ? 1 : std::max(1, (kib - 768 + 79) / 80);
}

long long EncoderTailFragmentIndex(int layer, int row, int col, int emb, int d_model) {
  // Parts of emb x emb: those of the output projection, then of the FFN's two layers in turn.
  const int ct = emb / 128, steps = emb / 32;
  int p = col / emb, r = row, c = col % emb;
  if (layer == 1) {
    p = d_model / emb + 2 * (row / emb);
    r = row % emb;
  } else if (layer == 2) {
    p = d_model / emb + 2 * (col / emb) + 1;
  }
  const int wave = r / (16 * ct), tile = r / 16 % ct;
  const long long frag = ((long long)(p * 8 + wave) * steps + c / 32) * ct + tile;
  return (frag * 64 + r % 16 + 16 * (c % 32 / 8)) * 8 + c % 8;
}

void LaunchEncoderTail(const EncoderTailArgs& a, hipStream_t stream) {
  if (a.M <= 0) return;
  if (!EncoderTailSupported(a.emb, a.d_model, a.dff) || a.M % 64 != 0) throw std::runtime_error("LaunchEncoderTail: unsupported shape");
  if (PickEncoderTailShape(a.M, a.emb, a.dff).slices > 1 && (a.partial == nullptr || a.arrived == nullptr)) {
    throw std::runtime_error("LaunchEncoderTail: no place for the slices' sums");
  }
  if (a.emb == 256) {
    if (a.bf16) LaunchTailT<bf16_t, 2>(a, stream);
    else LaunchTailT<half_t, 2>(a, stream);
  } else {
    if (a.bf16) LaunchTailT<bf16_t, 1>(a, stream);
    else LaunchTailT<half_t, 1>(a, stream);
  }
}

}  // namespace lc0mi
