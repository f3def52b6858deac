// A whole residual tower of 64 float filters in one kernel, on the bfloat16 matrix instructions.
//
//   resident_tower_f32_kernel   EncodePlanes, the 3x3 convolutions, BiasActivate / BiasResidual / ApplySEUnit
//                               blas/network_blas.cc:640-713, blas/winograd_convolution3.cc:326-382,
//                               shared/activation.cc:166-267, blas/se_unit.cc:31-91
#include "split_bf16.h"
#include "tower_common.h"

#include <stdexcept>

namespace lc0mi {

namespace {

constexpr int C = 64;
constexpr int kLd = kParts * C + 8;           // of a row of activations: [part][channel], 16-byte reads of 16 rows meet different banks
constexpr int kLdPlanes = kParts * kPlanes + 8;
constexpr int kTaps = 9;
constexpr int kRing = 3;                      // steps (tap and 16 inputs) of weights in flight
constexpr int kThreads = 512;

// ---------------------------------------------------------------------------
// A workgroup owns one position from the bit planes to the last block, as resident_tower_kernel does: activations stay in LDS,
// weights stream from L2 three steps ahead, convolutions are nine shifted products whose rows past the board's edge read a
// row of zeros.
//
// Products: floats are sums of three bfloat16 (split_bf16.h), weights split at load and activations where they are stored, six
// products for one. v_mfma_f32_32x32x16_bf16 does 16 times the work of v_mfma_f32_16x16x4_f32 in the same time, so six
// of it are 2.7 times faster, and an accumulator takes 9 roundings per convolution where the float instructions took 16 per tap.
//
// Split: wave (kq, cg) multiplies all 64 rows by 32 output channels over a quarter of the inputs, so that a fragment of weights is
// used twice and read by one wave (per step of a tap and 16 inputs 768 cycles of products on a SIMD's two waves, 384 of LDS
// reads, 384 of weights at 64 bytes a cycle). The quarters are exchanged through LDS; each wave then ends 32 rows of 16
// channels.
// What bounds it: the products on the one CU of a position (97 k of the 174 k cycles of a 6x64 tower, counted), the ends of a convolution, and
// what runs between convolutions: squeeze-and-excitation 11 % of the cycles, biases, skip and activations 11 %.
// us a pass through the interface, float instructions (up to 24 positions winograd) -> this: 6x64 with squeeze-and-excitation 1 position
// 172 -> 124, 32 222 -> 139, 200 331 -> 251, 512 (winograd) 708 -> 486. Relative error of the raw logits against 64 bits at 32 and
// 200 positions 2.28e-7 and 2.33e-7 -> 1.95e-7 and 1.98e-7 (most of it from the heads' products), of the values 1.4e-7 -> 8.6e-8.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads, 1) void resident_tower_f32_kernel(TowerArgs p) {
  constexpr int kOther = 64 * kLd, kPlanesAt = 2 * 64 * kLd, kZero = kPlanesAt + 64 * kLdPlanes;
  __shared__ __attribute__((aligned(16))) bf16_t lds[kZero + kLdPlanes];   // two activation buffers, planes, a row of zeros
  __shared__ floatx4 exchange[2][4][3][2][64];                             // [cg][to quarter][from][half of the sums][lane]
  __shared__ __attribute__((aligned(16))) float pool[2][C];
  __shared__ float hidden[kTowerMaxSe];
  __shared__ __attribute__((aligned(16))) float biases[2][C];              // of this convolution and the next
  __shared__ __attribute__((aligned(16))) float scale_shift[2][C];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cg = wave & 1, kq = wave >> 1;
  const int r = lane & 31, g = lane >> 5;
  const long long steps = 2 * kTaps + 2LL * kTaps * p.blocks;
  const intx4* ws = reinterpret_cast<const intx4*>(p.packed) + wave * steps * kParts * 64 + lane;
  intx4 w[kRing][kParts];
#pragma unroll
  for (int j = 0; j < kRing; j++)
#pragma unroll
    for (int f = 0; f < kParts; f++) w[j][f] = ws[(j * kParts + f) * 64];

  // Planes.
  {
    const int v = tid % (kPlanes / 4);
    const long long at = (long long)blockIdx.x * 112;
    uint64_t mask[4];
    floatx4 value;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int plane = v * 4 + e;
      mask[e] = plane < 112 ? p.masks[at + plane] : 0;
      value[e] = plane < 112 ? p.values[at + plane] : 0.0f;
    }
    bf16x4 part[kParts];
    Split3(value, part);
    const bf16_t zero = (bf16_t)0.0f;
    for (int sq = tid / (kPlanes / 4); sq < 64; sq += kThreads / (kPlanes / 4)) {
#pragma unroll
      for (int f = 0; f < kParts; f++) {
        bf16x4 x;
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = ((mask[e] >> sq) & 1) ? part[f][e] : zero;
        *reinterpret_cast<bf16x4*>(lds + kPlanesAt + sq * kLdPlanes + f * kPlanes + v * 4) = x;
      }
    }
    if (tid < kLdPlanes / 8) *reinterpret_cast<intx4*>(lds + kZero + tid * 8) = intx4{0, 0, 0, 0};
    if (tid < C) biases[0][tid] = p.biases[tid];
  }
  __syncthreads();

  // Sums of this wave's 32 rows (from 32 (kq / 2)) and 16 channels: element 4 i + e is channel ch0 + 8 i + e of row `row`.
  floatx4 sum[2];
  const int row = 32 * (kq >> 1) + r, ch0 = 32 * cg + 16 * (kq & 1) + 4 * g;
  // sum = the convolution of the rows at src (element offset) of ld values, `part` apart, over `inputs` of this wave.
  auto convolve = [&](int src, int ld, int part, int inputs) {
    floatx16 hi[2] = {}, lo[2] = {};
    for (int k = 0; k < inputs; k += 16) {
      intx4 a[2][2][kParts];
      auto load_rows = [&](intx4 (&x)[2][kParts], int tap) {
        const int dy = tap / 3 - 1, dx = tap % 3 - 1, col = (r & 7) + dx;
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const int y = 4 * t + (r >> 3) + dy;
          const bool on = (unsigned)col < 8u && (unsigned)y < 8u;
          const bf16_t* at = lds + (on ? src + (y * 8 + col) * ld : kZero) + kq * inputs + k + 8 * g;
#pragma unroll
          for (int f = 0; f < kParts; f++) x[t][f] = *reinterpret_cast<const intx4*>(at + f * part);
        }
      };
      load_rows(a[0], 0);
#pragma unroll
      for (int j = 0; j < kTaps; j++) {
        if (j + 1 < kTaps) load_rows(a[(j + 1) & 1], j + 1);
#pragma unroll
        for (int i = 0; i < kProducts; i++)
#pragma unroll
          for (int t = 0; t < 2; t++) {
            floatx16& acc = i + 1 < kProducts ? lo[t] : hi[t];
            acc = Mfma32(__builtin_bit_cast(bf16x8, w[j % kRing][kFirst[i]]), __builtin_bit_cast(bf16x8, a[j & 1][t][kSecond[i]]), acc);
          }
#pragma unroll
        for (int f = 0; f < kParts; f++) w[j % kRing][f] = ws[((kRing + j) * kParts + f) * 64];
        // The next rows go out one by one between these products, and nothing moves past them.
#pragma unroll
        for (int i = 0; i < 2 * kParts; i++) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      ws += kTaps * kParts * 64;
    }
    // Quarter q of the sums: rows 32 (q / 2) .. + 31, elements 8 (q % 2) .. + 7.
    auto quarter = [&](int q, int i) {
      floatx4 v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = SumOfProducts(hi[q >> 1][8 * (q & 1) + 4 * i + e], lo[q >> 1][8 * (q & 1) + 4 * i + e]);
      return v;
    };
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (q == kq) {
        sum[0] = quarter(q, 0);
        sum[1] = quarter(q, 1);
      } else {
        const int from = kq < q ? kq : kq - 1;
        exchange[cg][q][from][0][lane] = quarter(q, 0);
        exchange[cg][q][from][1][lane] = quarter(q, 1);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) sum[i] = (sum[i] + exchange[cg][kq][0][i][lane]) + (exchange[cg][kq][1][i][lane] + exchange[cg][kq][2][i][lane]);
  };
  float next_bias = 0.0f;
  auto ask_bias = [&](int conv) { next_bias = p.biases[(long long)min(conv, 2 * p.blocks) * C + tid % C]; };
  auto keep_bias = [&](int conv) {
    if (tid < C) biases[conv & 1][tid] = next_bias;
  };
  auto bias4 = [&](int conv, int i) { return *reinterpret_cast<const floatx4*>(&biases[conv & 1][ch0 + 8 * i]); };
  auto store = [&](int dst, int i, const floatx4& v) {
    bf16x4 part[kParts];
    Split3(v, part);
#pragma unroll
    for (int f = 0; f < kParts; f++) *reinterpret_cast<bf16x4*>(lds + dst + row * kLd + f * C + ch0 + 8 * i) = part[f];
  };
  auto plain_tail = [&](int conv, int dst) {
    TowerAct(p.act, [&](auto act) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const floatx4 v = sum[i] + bias4(conv, i);
        store(dst, i, floatx4{act(v[0]), act(v[1]), act(v[2]), act(v[3])});
      }
    });
    keep_bias(conv + 1);
    __syncthreads();
  };
  ask_bias(1);
  convolve(kPlanesAt, kLdPlanes, kPlanes, kPlanes / 4);
  plain_tail(0, 0);

  for (int conv = 1; conv <= 2 * p.blocks; conv += 2) {
    ask_bias(conv + 1);
    convolve(0, kLd, C, C / 4);
    plain_tail(conv, kOther);
    ask_bias(conv + 2);
    const TowerSe se = p.se[conv / 2];
    convolve(kOther, kLd, C, C / 4);
    if (se.k > 0) {
      // First layer: a wave does 16 hidden values, lane l value l % 16 and every fourth vector of the channels. Second layer: a
      // thread does four outputs and every sixteenth hidden value.
      constexpr int S1 = C / 16, O4 = 2 * C / 4, KP = kThreads / O4;
      const int k_lane = lane & 15, v_lane = lane >> 4, o4 = tid % O4, kp = tid / O4;
      floatx4 w1[S1], w2;
      auto load_w1 = [&](int k0) {
        const float* at = se.w1 + (long long)min(k0 + k_lane, se.k - 1) * C + 4 * v_lane;
#pragma unroll
        for (int i = 0; i < S1; i++) w1[i] = *reinterpret_cast<const floatx4*>(at + 16 * i);
      };
      auto load_w2 = [&](int k0) { w2 = *reinterpret_cast<const floatx4*>(se.w2 + (long long)min(k0, se.k - 1) * 2 * C + 4 * o4); };
      load_w1(16 * wave);
      load_w2(kp);
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const floatx4 bias = bias4(conv + 1, i);
        floatx4 s;
#pragma unroll
        for (int e = 0; e < 4; e++) s[e] = Sum32(sum[i][e]) * (1.0f / 64.0f) + (kq < 2 ? bias[e] : 0.0f);
        if (r == 16) *reinterpret_cast<floatx4*>(&pool[kq >> 1][ch0 + 8 * i]) = s;
      }
      __syncthreads();
      for (int k0 = 16 * wave; k0 < se.k; k0 += 16 * (kThreads / 64)) {
        if (k0 > 16 * wave) load_w1(k0);
        floatx4 h4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < S1; i++)
          h4 += w1[i] * (*reinterpret_cast<const floatx4*>(&pool[0][16 * i + 4 * v_lane]) + *reinterpret_cast<const floatx4*>(&pool[1][16 * i + 4 * v_lane]));
        float h = (h4[0] + h4[1]) + (h4[2] + h4[3]);
        h += __shfl_xor(h, 16, 64);
        h += __shfl_xor(h, 32, 64);
        const int k = k0 + k_lane;
        if (v_lane == 0 && k < se.k) TowerAct(p.act, [&](auto act) { hidden[k] = act(h + se.b1[k]); });
      }
      __syncthreads();
      floatx4 out = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int k = kp; k < se.k; k += KP) {
        if (k > kp) load_w2(k);
        out += w2 * hidden[k];
      }
      // (the sums that were exchanged have been read)
      float* part = reinterpret_cast<float*>(&exchange[0][0][0][0][0]);
      *reinterpret_cast<floatx4*>(part + kp * 2 * C + 4 * o4) = out;
      __syncthreads();
      if (tid < 2 * C) {
        float v = se.b2[tid];
#pragma unroll
        for (int j = 0; j < KP; j++) v += part[j * 2 * C + tid];
        scale_shift[tid / C][tid % C] = tid < C ? 1.0f / (1.0f + __expf(-v)) : v;
      }
      __syncthreads();
    }
    TowerAct(p.act, [&](auto act) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int ch = ch0 + 8 * i;
        floatx4 gamma = {1.0f, 1.0f, 1.0f, 1.0f}, beta = bias4(conv + 1, i);
        if (se.k > 0) {
          gamma = *reinterpret_cast<const floatx4*>(&scale_shift[0][ch]);
          beta = *reinterpret_cast<const floatx4*>(&scale_shift[1][ch]) + gamma * beta;
        }
        const floatx4 skip = Join3(lds + row * kLd + ch, C);
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = act(gamma[e] * sum[i][e] + beta[e] + skip[e]);
        if (conv + 1 < 2 * p.blocks) store(0, i, v);
        else *reinterpret_cast<floatx4*>(static_cast<float*>(p.out) + ((long long)blockIdx.x * 64 + row) * C + ch) = v;
      }
    });
    keep_bias(conv + 2);
    __syncthreads();
  }
}

}  // namespace

// Elements of the packed weights (a few steps' worth is asked for past the end), and the index of the first part of one of them;
// the others are kSplitPart further each.
long long TowerF32Fragments(int blocks) { return (8 * (2LL * kTaps + 2LL * kTaps * blocks) + kRing) * kParts * 512; }

long long TowerF32FragmentIndex(int blocks, int conv, int tap, int out, int in) {
  const long long steps = 2LL * kTaps + 2LL * kTaps * blocks;
  const int kq = conv == 0 ? in / 32 : in / 16, wave = 2 * kq + out / 32;
  const long long step = conv == 0 ? in / 16 % 2 * kTaps + tap : 2LL * kTaps + (conv - 1LL) * kTaps + tap;
  return ((wave * steps + step) * kParts * 64 + out % 32 + 32 * (in % 16 / 8)) * 8 + in % 8;
}

void LaunchTowerF32(const TowerArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  if (a.blocks < 1 || (a.act != kActMish && a.act != kActRelu) || a.filters != C) throw std::runtime_error("LaunchTowerF32: no kernel");
  hipLaunchKernelGGL(resident_tower_f32_kernel, dim3(a.batch), dim3(kThreads), 0, stream, a);
}

}  // namespace lc0mi
