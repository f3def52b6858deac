// gfx950 kernels of the SE-ResNet tower (bandwidth-bound parts; the 36 batched
// GEMMs of each convolution run on the GEMM kernels of kernels.hip).
//
// What each kernel replaces in the reference CPU backend (file:line):
//   winograd_input_transform    WinogradConvolution3::TransformIn   blas/winograd_convolution3.cc:59-166
//   winograd_output_transform   TransformOut + BiasActivate / BiasResidual / ApplySEUnit
//                               blas/winograd_convolution3.cc:256-324, shared/activation.cc:166-267,
//                               blas/se_unit.cc:31-91
//   WinogradFilterTransform4x4  WinogradFilterTransformF            shared/winograd_filter.cc:54-90
//   conv_policy_gather          kConvPolicyMap gather               blas/network_blas.cc:931-942
// The reference uses F(2x2,3x3); this backend uses F(4x4,3x3) (4 tiles per board
// instead of 16): the same convolution with 2.25x fewer multiplications.
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace lc0mi {
namespace {

__device__ __forceinline__ float RActivate(float v, int act) {
  switch (act) {
    case 1: {  // mish = v * n / (n + 2), n = e^v (e^v + 2); exponent clamped where the ratio rounds to 1
      const float e = __expf(__builtin_fminf(v, 20.0f));
      const float n = e * (e + 2.0f);
      return v * n * __builtin_amdgcn_rcpf(n + 2.0f);
    }
    case 2: return v > 0.0f ? v : 0.0f;
    case 4: return tanhf(v);
    case 5: return __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    case 6: return v > 0.0f ? 1.05070098f * v : 1.05070098f * 1.67326324f * (__expf(v) - 1.0f);
    case 7: return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    case 8: return v > 0.0f ? v * v : 0.0f;
    default: return v;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void expand_planes_nhwc_kernel(const uint64_t* __restrict__ masks,
                                                                 const float* __restrict__ values,
                                                                 T* __restrict__ out) {
  const int b = blockIdx.x;
  __shared__ uint64_t smask[112];
  __shared__ float sval[112];
  if (threadIdx.x < 112) {
    smask[threadIdx.x] = masks[(long long)b * 112 + threadIdx.x];
    sval[threadIdx.x] = values[(long long)b * 112 + threadIdx.x];
  }
  __syncthreads();
  T* o = out + (long long)b * 64 * 112;
  for (int i = threadIdx.x; i < 64 * 112; i += 256) {
    int sq = i / 112, c = i - sq * 112;
    o[i] = ((smask[c] >> sq) & 1ull) ? (T)sval[c] : (T)0.0f;
  }
}

// One thread per (sample, tile, channel); channels are the fastest index so that
// loads and stores of neighbouring threads are contiguous.
template <typename T>
__global__ __launch_bounds__(256) void winograd_input_transform_kernel(const T* __restrict__ x, T* __restrict__ v,
                                                                       int batch, int C, int ldv) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int bt = blockIdx.y;  // b * 4 + tile
  if (c >= ldv) return;
  if (c >= C) {   // padding columns of a row longer than C: zeros, so that the GEMM may reduce over ldv
#pragma unroll
    for (int k = 0; k < 36; k++) v[((long long)k * batch * 4 + bt) * ldv + c] = (T)0.0f;
    return;
  }
  const int b = bt >> 2, tile = bt & 3;
  const int y0 = (tile >> 1) * 4 - 1, x0 = (tile & 1) * 4 - 1;
  const T* xb = x + (long long)b * 64 * C + c;
  float d[6][6];
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j < 6; j++) {
      const int yy = y0 + i, xx = x0 + j;
      d[i][j] = (yy >= 0 && yy < 8 && xx >= 0 && xx < 8) ? (float)xb[(long long)(yy * 8 + xx) * C] : 0.0f;
    }
  // t = B^T d (rows), then v = t B (columns); B^T rows scaled by 1/(4,6,6,24,24,1).
  float t[6][6];
#pragma unroll
  for (int j = 0; j < 6; j++) {
    const float d0 = d[0][j], d1 = d[1][j], d2 = d[2][j], d3 = d[3][j], d4 = d[4][j], d5 = d[5][j];
    t[0][j] = d0 - 1.25f * d2 + 0.25f * d4;
    t[1][j] = (-4.0f * (d1 + d2) + d3 + d4) * (1.0f / 6.0f);
    t[2][j] = (4.0f * (d1 - d2) - d3 + d4) * (1.0f / 6.0f);
    t[3][j] = (-2.0f * d1 - d2 + 2.0f * d3 + d4) * (1.0f / 24.0f);
    t[4][j] = (2.0f * d1 - d2 - 2.0f * d3 + d4) * (1.0f / 24.0f);
    t[5][j] = 4.0f * d1 - 5.0f * d3 + d5;
  }
  T* vo = v + (long long)bt * ldv + c;
  const long long kstride = (long long)batch * 4 * ldv;
#pragma unroll
  for (int i = 0; i < 6; i++) {
    const float t0 = t[i][0], t1 = t[i][1], t2 = t[i][2], t3 = t[i][3], t4 = t[i][4], t5 = t[i][5];
    float r[6];
    r[0] = t0 - 1.25f * t2 + 0.25f * t4;
    r[1] = (-4.0f * (t1 + t2) + t3 + t4) * (1.0f / 6.0f);
    r[2] = (4.0f * (t1 - t2) - t3 + t4) * (1.0f / 6.0f);
    r[3] = (-2.0f * t1 - t2 + 2.0f * t3 + t4) * (1.0f / 24.0f);
    r[4] = (2.0f * t1 - t2 - 2.0f * t3 + t4) * (1.0f / 24.0f);
    r[5] = 4.0f * t1 - 5.0f * t3 + t5;
#pragma unroll
    for (int j = 0; j < 6; j++) vo[(long long)(i * 6 + j) * kstride] = (T)r[j];
  }
}

// One workgroup per sample, one thread per channel (channels beyond blockDim loop).
// Shared memory: pool[C] | hidden[K] floats.
template <typename T, typename MT>
__global__ void winograd_output_transform_kernel(const MT* __restrict__ m, const float* __restrict__ bias,
                                                 const T* skip, const float* __restrict__ se_w1,
                                                 const float* __restrict__ se_b1,
                                                 const float* __restrict__ se_w2,
                                                 const float* __restrict__ se_b2, int se_k, T* out, int batch,
                                                 int C, int act) {
  extern __shared__ float shm[];
  float* pool = shm;
  float* hidden = shm + C;
  const int b = blockIdx.x;
  const int c = threadIdx.x;  // blockDim.x == C (C <= 1024)
  const long long kstride = (long long)batch * 4 * C;
  float y[64];
  float sum = 0.0f;
#pragma unroll
  for (int tile = 0; tile < 4; tile++) {
    const MT* mp = m + (long long)(b * 4 + tile) * C + c;
    // s = A^T mm (4x6), then o = s A (4x4); A^T = [1 1 1 1 1 0; 0 1 -1 2 -2 0; 0 1 1 4 4 0; 0 1 -1 8 -8 1].
    float s[4][6];
#pragma unroll
    for (int j = 0; j < 6; j++) {
      const float m0 = (float)mp[(long long)(0 * 6 + j) * kstride], m1 = (float)mp[(long long)(1 * 6 + j) * kstride];
      const float m2 = (float)mp[(long long)(2 * 6 + j) * kstride], m3 = (float)mp[(long long)(3 * 6 + j) * kstride];
      const float m4 = (float)mp[(long long)(4 * 6 + j) * kstride], m5 = (float)mp[(long long)(5 * 6 + j) * kstride];
      s[0][j] = m0 + m1 + m2 + m3 + m4;
      s[1][j] = m1 - m2 + 2.0f * (m3 - m4);
      s[2][j] = m1 + m2 + 4.0f * (m3 + m4);
      s[3][j] = m1 - m2 + 8.0f * (m3 - m4) + m5;
    }
    const int ty = (tile >> 1) * 4, tx = (tile & 1) * 4;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float s0 = s[i][0], s1 = s[i][1], s2 = s[i][2], s3 = s[i][3], s4 = s[i][4], s5 = s[i][5];
      const float o0 = s0 + s1 + s2 + s3 + s4;
      const float o1 = s1 - s2 + 2.0f * (s3 - s4);
      const float o2 = s1 + s2 + 4.0f * (s3 + s4);
      const float o3 = s1 - s2 + 8.0f * (s3 - s4) + s5;
      y[(ty + i) * 8 + tx + 0] = o0;
      y[(ty + i) * 8 + tx + 1] = o1;
      y[(ty + i) * 8 + tx + 2] = o2;
      y[(ty + i) * 8 + tx + 3] = o3;
      sum += o0 + o1 + o2 + o3;
    }
  }
  const float bc = bias[c];
  float gamma = 1.0f, beta = bc;
  if (se_k > 0) {
    pool[c] = sum * (1.0f / 64.0f) + bc;
    __syncthreads();
    for (int k = c; k < se_k; k += blockDim.x) {
      float h = se_b1[k];
      const float* w = se_w1 + (long long)k * C;
      for (int i = 0; i < C; i++) h += w[i] * pool[i];
      hidden[k] = RActivate(h, act);
    }
    __syncthreads();
    float sg = se_b2[c], sb = se_b2[C + c];
    for (int k = 0; k < se_k; k++) {   // se_w2 is stored [K][2C]: neighbouring channels, neighbouring addresses
      sg += se_w2[(long long)k * 2 * C + c] * hidden[k];
      sb += se_w2[(long long)k * 2 * C + C + c] * hidden[k];
    }
    gamma = 1.0f / (1.0f + __expf(-sg));
    beta = sb + gamma * bc;
  }
  const T* sk = skip ? skip + (long long)b * 64 * C + c : nullptr;
  T* o = out + (long long)b * 64 * C + c;
#pragma unroll
  for (int sq = 0; sq < 64; sq++) {
    float v = gamma * y[sq] + beta;
    if (sk) v += (float)sk[(long long)sq * C];
    o[(long long)sq * C] = (T)RActivate(v, act);
  }
}

// V neighbouring channels (a vector type: a struct of halves would be kept in a register each).
template <typename T, int V> using Channels = T __attribute__((ext_vector_type(V)));

// A winograd-domain tile m (6x6) back to its 4x4 outputs: A^T m A.
__device__ __forceinline__ void OutputTile(const float (&mm)[36], float (&y)[4][4]) {
  float s[4][6];
#pragma unroll
  for (int j = 0; j < 6; j++) {
    const float m0 = mm[j], m1 = mm[6 + j], m2 = mm[12 + j], m3 = mm[18 + j], m4 = mm[24 + j], m5 = mm[30 + j];
    s[0][j] = m0 + m1 + m2 + m3 + m4;
    s[1][j] = m1 - m2 + 2.0f * (m3 - m4);
    s[2][j] = m1 + m2 + 4.0f * (m3 + m4);
    s[3][j] = m1 - m2 + 8.0f * (m3 - m4) + m5;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float s0 = s[i][0], s1 = s[i][1], s2 = s[i][2], s3 = s[i][3], s4 = s[i][4], s5 = s[i][5];
    y[i][0] = s0 + s1 + s2 + s3 + s4;
    y[i][1] = s1 - s2 + 2.0f * (s3 - s4);
    y[i][2] = s1 + s2 + 4.0f * (s3 + s4);
    y[i][3] = s1 - s2 + 8.0f * (s3 - s4) + s5;
  }
}

// A 6x6 patch d to the winograd domain: B^T d B.
__device__ __forceinline__ void InputTile(const float (&d)[6][6], float (&r)[6][6]) {
  float t[6][6];
#pragma unroll
  for (int j = 0; j < 6; j++) {
    const float d0 = d[0][j], d1 = d[1][j], d2 = d[2][j], d3 = d[3][j], d4 = d[4][j], d5 = d[5][j];
    t[0][j] = d0 - 1.25f * d2 + 0.25f * d4;
    t[1][j] = (-4.0f * (d1 + d2) + d3 + d4) * (1.0f / 6.0f);
    t[2][j] = (4.0f * (d1 - d2) - d3 + d4) * (1.0f / 6.0f);
    t[3][j] = (-2.0f * d1 - d2 + 2.0f * d3 + d4) * (1.0f / 24.0f);
    t[4][j] = (2.0f * d1 - d2 - 2.0f * d3 + d4) * (1.0f / 24.0f);
    t[5][j] = 4.0f * d1 - 5.0f * d3 + d5;
  }
#pragma unroll
  for (int i = 0; i < 6; i++) {
    const float t0 = t[i][0], t1 = t[i][1], t2 = t[i][2], t3 = t[i][3], t4 = t[i][4], t5 = t[i][5];
    r[i][0] = t0 - 1.25f * t2 + 0.25f * t4;
    r[i][1] = (-4.0f * (t1 + t2) + t3 + t4) * (1.0f / 6.0f);
    r[i][2] = (4.0f * (t1 - t2) - t3 + t4) * (1.0f / 6.0f);
    r[i][3] = (-2.0f * t1 - t2 + 2.0f * t3 + t4) * (1.0f / 24.0f);
    r[i][4] = (2.0f * t1 - t2 - 2.0f * t3 + t4) * (1.0f / 24.0f);
    r[i][5] = 4.0f * t1 - 5.0f * t3 + t5;
  }
}

// Same for C <= 256 with one thread per (tile, V neighbouring channels), blockDim.x == 4 * C / V.
// Shared memory: part[4][C] | hidden[K] | fc2[4][2][C] floats | xs[64][C]; with WIDTH xs[64][WIDTH].
//
// With few positions the chain of memory latencies bounds it (m, first squeeze-and-excitation layer, second one, skip):
// the skip and the first four weights of either layer are asked for together with m (per launch, 32 positions x 64
// float channels: 8.8 -> 7.2 us; a 20x256 pass of 32 positions in halves 1035 -> 988 us, of one position 819 -> 804).
// In bulk it moves its bytes at about 4 TB/s (512 positions x 256 half channels, 92 MB: 24 us), every CU reading, then
// computing, then writing at the same time as the others; V = 2 keeps two workgroups on a CU there (128 registers) and
// halves the instructions (1000 positions 4082 -> 4007 us a pass; at 512 and below 300 the two forms are level, with
// few positions V = 1 has twice the waves). One channel per thread in bulk (floats, and halves of 16 times an odd
// number of channels) wants the waves more than the early requests: without them (EARLY = false) it takes 61 registers
// instead of 114 and eight waves per SIMD instead of four (a pass of a ten-block tower in halves, 1000 positions: 176 channels
// 1854 -> 1630 us, 240 2590 -> 2310).
// WIDTH > 0: no squeeze-and-excitation, and a workgroup takes WIDTH channels from blockIdx.y * WIDTH instead of all C.
// The squeeze-and-excitation layers are spread over all threads: every wave pools the channels it needs itself, the
// second layer is split four ways over k, and every thread adds the four partial sums of its own channels.
template <typename T, typename MT, int V, bool EARLY, int WIDTH>
__global__ __launch_bounds__((WIDTH > 0 ? 4 * WIDTH : 1024) / V, EARLY ? 4 : WIDTH > 0 ? 6 : 8) void winograd_output_transform_tiles_kernel(
    const MT* __restrict__ m, const float* __restrict__ bias, const T* skip, const float* __restrict__ se_w1,
    const float* __restrict__ se_b1, const float* __restrict__ se_w2, const float* __restrict__ se_b2, int se_k,
    T* out, T* __restrict__ v_next, int ldv, int batch, int C, int act) {
  using Ch = Channels<T, V>;
  using ChM = Channels<MT, V>;
  using ChF = Channels<float, V>;
  extern __shared__ __attribute__((aligned(16))) float shm[];
  float* part = shm;               // [4][C]
  float* hidden = shm + 4 * C;     // [K]
  float* fc2 = hidden + se_k + (se_k & 1);   // [4][gamma | beta][C] partial sums of the second layer
  // activations [64][width] for the fused input transform
  T* xs = reinterpret_cast<T*>(WIDTH > 0 ? shm : fc2 + 8 * C);
  const int b = blockIdx.x;
  const int width = WIDTH > 0 ? WIDTH : C;
  const int per_tile = width / V;
  const int tile = threadIdx.x / per_tile, c_in = V * (threadIdx.x - tile * per_tile);
  const int c = WIDTH > 0 ? (int)blockIdx.y * WIDTH + c_in : c_in;
  const int ty = (tile >> 1) * 4, tx = (tile & 1) * 4;
  const long long kstride = (long long)batch * 4 * C;
  // (a base that all lanes share and a 32-bit lane offset: one address register for the 36 loads)
  const MT* mp = m + (long long)b * 4 * C;
  const unsigned m_off = tile * C + c;
  ChM mm[36];
#pragma unroll
  for (int k = 0; k < 36; k++) mm[k] = *reinterpret_cast<const ChM*>(mp + (long long)k * kstride + m_off);
  const ChF bc = *reinterpret_cast<const ChF*>(bias + c);
  const unsigned sq_off = (ty * 8 + tx) * C + c, xs_off = WIDTH > 0 ? (ty * 8 + tx) * width + c_in : sq_off;
  using Raw = std::conditional_t<sizeof(Ch) == 4, uint32_t, uint16_t>;   // (as halves the pairs would be split into registers)
  static_assert(sizeof(Ch) == sizeof(Raw), "2 or 4 bytes per lane");
  Raw sk[16];
  auto load_skip = [&]() {
    const T* sp = skip + (long long)b * 64 * C;
#pragma unroll
    for (int i = 0; i < 16; i++) sk[i] = *reinterpret_cast<const Raw*>(sp + (i / 4 * 8 + i % 4) * C + sq_off);
  };
  // Squeeze-and-excitation weights. First layer: one wave per k = wave, wave + nwaves, ..., lanes stride over the
  // channels, four k at a time. Second layer: k = tile, tile + 4, ..., four at a time.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  constexpr int kMaxPerLane = 4;   // C <= 256
  constexpr int U = EARLY ? 4 : 2;
  float w1[U][kMaxPerLane], b1[U];
  ChF wg[4], wb[4], sg, sb;
  auto load_w1 = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = min(k0 + u * nwaves, se_k - 1);
      b1[u] = se_b1[k];
#pragma unroll
      for (int q = 0; q < kMaxPerLane; q++) w1[u][q] = se_w1[(long long)k * C + min(lane + 64 * q, C - 1)];
    }
  };
  auto load_w2 = [&](int k0) {   // se_w2 is stored [K][2C]: neighbouring channels, neighbouring addresses
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float* w = se_w2 + (long long)min(k0 + 4 * u, se_k - 1) * 2 * C + c;
      wg[u] = *reinterpret_cast<const ChF*>(w);
      wb[u] = *reinterpret_cast<const ChF*>(w + C);
    }
  };
  auto ask = [&]() {
    if (WIDTH == 0 && se_k > 0) {
      load_w1(wave);
      load_w2(tile);
      sg = *reinterpret_cast<const ChF*>(se_b2 + c);
      sb = *reinterpret_cast<const ChF*>(se_b2 + C + c);
    }
  };
  if constexpr (V == 1 && EARLY) {
    if (skip != nullptr) load_skip();
    ask();
  }
  float y[V][4][4];
#pragma unroll
  for (int v = 0; v < V; v++) {
    float f[36];
#pragma unroll
    for (int k = 0; k < 36; k++) f[k] = (float)mm[k][v];
    OutputTile(f, y[v]);
  }
  if constexpr (V > 1 && EARLY) ask();   // (the registers of m are free now; the skip has to wait for those of the weights)
  float gamma[V], beta[V];
#pragma unroll
  for (int v = 0; v < V; v++) gamma[v] = 1.0f, beta[v] = bc[v];
  if (WIDTH == 0 && se_k > 0) {
    ChF sum;
#pragma unroll
    for (int v = 0; v < V; v++) {
      sum[v] = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; i++) sum[v] += y[v][i][0] + y[v][i][1] + y[v][i][2] + y[v][i][3];
    }
    *reinterpret_cast<ChF*>(&part[tile * C + c]) = sum;
    __syncthreads();
    // hidden[k] = act(w1[k] . pool + b1[k])
    float pool[kMaxPerLane];
#pragma unroll
    for (int q = 0; q < kMaxPerLane; q++) {
      const int i = lane + 64 * q;
      pool[q] = i < C ? (part[i] + part[C + i] + part[2 * C + i] + part[3 * C + i]) * (1.0f / 64.0f) + bias[i] : 0.0f;
    }
    for (int k0 = wave; k0 < se_k; k0 += U * nwaves) {
      if (!EARLY || k0 != wave) load_w1(k0);
      float h[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        h[u] = 0.0f;
#pragma unroll
        for (int q = 0; q < kMaxPerLane; q++) h[u] += w1[u][q] * pool[q];
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int u = 0; u < U; u++) h[u] += __shfl_xor(h[u], off, 64);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int k = k0 + u * nwaves;
        if (lane == 0 && k < se_k) hidden[k] = RActivate(h[u] + b1[u], act);
      }
    }
    __syncthreads();
    // Second layer: this thread's share of k.
    ChF pg, pb;
#pragma unroll
    for (int v = 0; v < V; v++) pg[v] = 0.0f, pb[v] = 0.0f;
    for (int k0 = tile; k0 < se_k; k0 += 16) {
      if (!EARLY || k0 != tile) load_w2(k0);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int k = k0 + 4 * u;
        const float h = k < se_k ? hidden[k] : 0.0f;
#pragma unroll
        for (int v = 0; v < V; v++) {
          pg[v] += wg[u][v] * h;
          pb[v] += wb[u][v] * h;
        }
      }
    }
    *reinterpret_cast<ChF*>(&fc2[(tile * 2) * C + c]) = pg;
    *reinterpret_cast<ChF*>(&fc2[(tile * 2 + 1) * C + c]) = pb;
    __syncthreads();
    if constexpr (!EARLY) {
      sg = *reinterpret_cast<const ChF*>(se_b2 + c);
      sb = *reinterpret_cast<const ChF*>(se_b2 + C + c);
    }
    ChF fg[4], fb[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      fg[t] = *reinterpret_cast<const ChF*>(&fc2[(t * 2) * C + c]);
      fb[t] = *reinterpret_cast<const ChF*>(&fc2[(t * 2 + 1) * C + c]);
    }
#pragma unroll
    for (int v = 0; v < V; v++) {
      const float g = sg[v] + ((fg[0][v] + fg[1][v]) + (fg[2][v] + fg[3][v]));
      const float a = sb[v] + ((fb[0][v] + fb[1][v]) + (fb[2][v] + fb[3][v]));
      gamma[v] = 1.0f / (1.0f + __expf(-g));
      beta[v] = a + gamma[v] * bc[v];
    }
  }
  if constexpr (V > 1 || !EARLY) {
    if (skip != nullptr) load_skip();
  }
  T* o = out ? out + (long long)b * 64 * C : nullptr;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int sq = i * 8 + j;
      Ch r;
#pragma unroll
      for (int v = 0; v < V; v++) {
        float x = gamma[v] * y[v][i][j] + beta[v];
        if (skip != nullptr) x += (float)__builtin_bit_cast(Ch, sk[4 * i + j])[v];
        r[v] = (T)RActivate(x, act);
      }
      if (o) *reinterpret_cast<Ch*>(o + sq * C + sq_off) = r;
      if (v_next) *reinterpret_cast<Ch*>(&xs[sq * width + xs_off]) = r;
    }
  if (!v_next) return;
  // Fused input transform of the next convolution: this thread's tile reads its 6x6
  // patch (with the halo owned by the other three tiles) from LDS.
  __syncthreads();
  const int y0 = ty - 1, x0 = tx - 1;
  Ch patch[6][6];
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j < 6; j++) {
      const int yy = y0 + i, xx = x0 + j;
      if (yy >= 0 && yy < 8 && xx >= 0 && xx < 8) {
        patch[i][j] = *reinterpret_cast<const Ch*>(&xs[(yy * 8 + xx) * width + c_in]);
      } else {
#pragma unroll
        for (int v = 0; v < V; v++) patch[i][j][v] = (T)0.0f;
      }
    }
#pragma unroll
  for (int v = 0; v < V; v++) {
    float d[6][6], r[6][6];
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
      for (int j = 0; j < 6; j++) d[i][j] = (float)patch[i][j][v];
    InputTile(d, r);
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
      for (int j = 0; j < 6; j++) patch[i][j][v] = (T)r[i][j];
  }
  T* vo = v_next + (long long)b * 4 * ldv;
  const unsigned v_off = tile * ldv + c;
  const long long vstride = (long long)batch * 4 * ldv;
#pragma unroll
  for (int i = 0; i < 36; i++) *reinterpret_cast<Ch*>(vo + (long long)i * vstride + v_off) = patch[i / 6][i % 6];
}

template <typename T>
__global__ __launch_bounds__(256) void conv_policy_gather_kernel(const T* __restrict__ t, int ld,
                                                                 const int16_t* __restrict__ inv_map,
                                                                 float* __restrict__ out) {
  const int b = blockIdx.x;
  for (int o = threadIdx.x; o < 1858; o += 256) {
    const int src = inv_map[o];
    const int plane = src >> 6, sq = src & 63;
    out[(long long)b * 1858 + o] = (float)t[((long long)b * 64 + sq) * ld + plane];
  }
}

}  // namespace

template <typename T>
void LaunchExpandPlanesNhwc(const uint64_t* masks, const float* values, T* out, int batch, hipStream_t stream) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(expand_planes_nhwc_kernel<T>, dim3(batch), dim3(256), 0, stream, masks, values, out);
}
template void LaunchExpandPlanesNhwc<half_t>(const uint64_t*, const float*, half_t*, int, hipStream_t);
template void LaunchExpandPlanesNhwc<float>(const uint64_t*, const float*, float*, int, hipStream_t);

void WinogradFilterTransform4x4(const float* filter, int cout, int cin, int ld_cin, float* u) {
  static const float G[6][3] = {{1, 0, 0}, {-1, -1, -1}, {-1, 1, -1}, {1, 2, 4}, {1, -2, 4}, {0, 0, 1}};
  const size_t plane = (size_t)cout * ld_cin;
  for (size_t i = 0; i < 36 * plane; i++) u[i] = 0.0f;
  for (int o = 0; o < cout; o++)
    for (int c = 0; c < cin; c++) {
      const float* g = filter + ((size_t)o * cin + c) * 9;
      float tmp[6][3];
      for (int i = 0; i < 6; i++)
        for (int j = 0; j < 3; j++) tmp[i][j] = G[i][0] * g[0 * 3 + j] + G[i][1] * g[1 * 3 + j] + G[i][2] * g[2 * 3 + j];
      for (int i = 0; i < 6; i++)
        for (int j = 0; j < 6; j++)
          u[(size_t)(i * 6 + j) * plane + (size_t)o * ld_cin + c] =
              tmp[i][0] * G[j][0] + tmp[i][1] * G[j][1] + tmp[i][2] * G[j][2];
    }
}

template <typename T>
void LaunchWinogradInputTransform(const T* x, T* v, int batch, int C, int ldv, hipStream_t stream) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(winograd_input_transform_kernel<T>, dim3((ldv + 255) / 256, batch * 4), dim3(256), 0, stream, x, v,
                     batch, C, ldv);
}
template void LaunchWinogradInputTransform<half_t>(const half_t*, half_t*, int, int, int, hipStream_t);
template void LaunchWinogradInputTransform<float>(const float*, float*, int, int, int, hipStream_t);

template <typename T, typename MT>
void LaunchWinogradOutputTransform(const MT* m, const float* bias, const T* skip, const float* se_w1,
                                   const float* se_b1, const float* se_w2, const float* se_b2, int se_k, T* out,
                                   int batch, int C, int act, hipStream_t stream, T* v_next, int ldv_next) {
  if (batch <= 0) return;
  const int k = se_k > 0 ? se_k : 0;
  if (C <= 256 && C % 16 == 0) {   // 4 * C threads in whole waves (the SE reduction shuffles across a wave)
    // Without squeeze-and-excitation the channels of a position need nothing of each other: while the positions do not fill the
    // CUs, 64 of them to a workgroup (at six waves per SIMD: eight spill), so that few positions lie on more CUs (a 20x256 pass in
    // halves, half of its transforms, us, whole positions -> 64 channels: 1 position 686 -> 622, 13 736 -> 671, 64 977 -> 917, 200 1331
    // -> 1296; 512 1910 -> 1943; in floats 1 742 -> 728, 13 963 -> 943, 64 1523 -> 1520, 200
    // 3291 -> 3318. 16 and 32 channels are level with 64).
    const bool split = k == 0 && C > 64 && C % 64 == 0 && batch <= (sizeof(T) == 2 ? 256 : 64);
    size_t shm = split ? 0 : sizeof(float) * (size_t)(12 * C + k + (k & 1));
    if (v_next) shm += sizeof(T) * 64 * (size_t)(split ? 64 : C);
    auto launch = [&](auto v_tag, auto early_tag, auto width_tag) {
      constexpr int V = decltype(v_tag)::value, W = decltype(width_tag)::value;
      hipLaunchKernelGGL((winograd_output_transform_tiles_kernel<T, MT, V, decltype(early_tag)::value, W>), dim3(batch, W > 0 ? C / std::max(W, 1) : 1),
                         dim3(4 * (W > 0 ? W : C) / V), shm, stream, m, bias, skip, se_w1, se_b1, se_w2, se_b2, se_k, out, v_next,
                         ldv_next, batch, C, act);
    };
    using Whole = std::integral_constant<int, 0>;
    if (split) return launch(std::integral_constant<int, 1>{}, std::false_type{}, std::integral_constant<int, 64>{});
    // Two channels per thread (see the kernel) where a CU has more than one position; that needs 2 * C threads in whole
    // waves and whole pairs of channels in every row.
    const bool pairs = C % 32 == 0 && (v_next == nullptr || ldv_next % 2 == 0);
    if constexpr (sizeof(T) == 2) {
      if (pairs && batch > 256) return launch(std::integral_constant<int, 2>{}, std::true_type{}, Whole{});
    }
    // The early requests while all positions are on the CUs at once (at four waves per SIMD a CU holds 256 / C workgroups),
    // the form of 61 registers beyond (us of the kernel, early / late: halves of 176 channels at 300 positions 20.8 / 16.7,
    // at 1000 41.0 / 30.2, floats of 192 22.5 / 18.0 and 54.1 / 46.2; the other way round floats of 64 at 300 13.1 / 13.5, halves
    // of 112 8.5 / 8.7).
    if (batch > 256 * (256 / C)) return launch(std::integral_constant<int, 1>{}, std::false_type{}, Whole{});
    launch(std::integral_constant<int, 1>{}, std::true_type{}, Whole{});
    return;
  }
  // Wide towers: separate kernels (the caller checks WinogradFusedInputTransform before asking for v_next).
  const size_t shm = sizeof(float) * (size_t)(C + k);
  hipLaunchKernelGGL((winograd_output_transform_kernel<T, MT>), dim3(batch), dim3(C), shm, stream, m, bias, skip,
                     se_w1, se_b1, se_w2, se_b2, se_k, out, batch, C, act);
}
// The fused kernel needs 4 * C threads and its staging area in the 64 KiB of dynamic LDS.
bool WinogradFusedInputTransform(int C, int elem_size, int se_k) {
  return C <= 256 && C % 16 == 0 && sizeof(float) * (12 * C + se_k + 1) + (size_t)elem_size * 64 * C <= 64 * 1024;
}

template void LaunchWinogradOutputTransform<half_t, half_t>(const half_t*, const float*, const half_t*, const float*,
                                                            const float*, const float*, const float*, int, half_t*,
                                                            int, int, int, hipStream_t, half_t*, int);
template void LaunchWinogradOutputTransform<half_t, float>(const float*, const float*, const half_t*, const float*,
                                                           const float*, const float*, const float*, int, half_t*, int,
                                                           int, int, hipStream_t, half_t*, int);
template void LaunchWinogradOutputTransform<float, float>(const float*, const float*, const float*, const float*,
                                                          const float*, const float*, const float*, int, float*, int,
                                                          int, int, hipStream_t, float*, int);

template <typename T>
void LaunchConvPolicyGather(const T* t, int ld, const int16_t* inv_map, float* out, int batch, hipStream_t stream) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(conv_policy_gather_kernel<T>, dim3(batch), dim3(256), 0, stream, t, ld, inv_map, out);
}
template void LaunchConvPolicyGather<half_t>(const half_t*, int, const int16_t*, float*, int, hipStream_t);
template void LaunchConvPolicyGather<float>(const float*, int, const int16_t*, float*, int, hipStream_t);

}  // namespace lc0mi
