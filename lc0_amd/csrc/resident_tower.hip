// A whole residual tower in one kernel: plane expansion, input convolution, every block with its squeeze-and-excitation.
//
//   resident_tower_kernel   EncodePlanes, the 3x3 convolutions, BiasActivate / BiasResidual / ApplySEUnit
//                           blas/network_blas.cc:640-713, blas/winograd_convolution3.cc:326-382,
//                           shared/activation.cc:166-267, blas/se_unit.cc:31-91
#include "tower_common.h"

#include <algorithm>
#include <stdexcept>
#include <type_traits>

namespace lc0mi {

namespace {

// A step of a convolution is 32 of one tap's inputs. Products are tiles of TILE rows (squares) and TILE output channels
// (v_mfma_f32_32x32x16, whose rate per operation is twice that of the 16x16x32 form: 32.5 and 30.2 cycles an instruction,
// measured). Weights are 1 KiB fragments of TILE channels (lane l: channel l % TILE, 16 bytes of inputs from l / TILE), a wave's in
// the order in which it multiplies them, over all convolutions of the tower.
constexpr int kWaves = 4;                 // that share the channels of a product
constexpr int kChunk = 8;                 // steps of a turn of the main loop, the most that are in flight per wave

template <int C> struct TowerShape {
  static constexpr int V = 8;                                      // values of a 16-byte vector
  static constexpr int KS = 4 * V;                                 // inputs of a step
  static constexpr int TILE = 32, G = 64 / TILE;
  static constexpr int SUB = KS / (G * V);                         // fragments of a tile in a step
  static constexpr int CT = C / (TILE * kWaves);                   // channel tiles of a wave
  static constexpr int F = CT * SUB;                               // weight fragments of a step
  static constexpr int NS = C / KS, NS_IN = kPlanes / KS;          // steps of a tap
  static constexpr int STEPS = (9 * NS + kChunk - 1) / kChunk * kChunk, STEPS_IN = (9 * NS_IN + kChunk - 1) / kChunk * kChunk;
  static constexpr int LD = (C > kPlanes ? C : kPlanes) + V;       // an odd number of vectors: 16 rows meet different banks
  static_assert(kChunk % NS == 0 && kChunk % NS_IN == 0, "a turn does whole taps");
};

// ---------------------------------------------------------------------------
// A workgroup owns POS positions from the bit planes to the last block: their activations never leave LDS (a block's input
// and its inner activations, 64 POS rows each), and the weights stream from L2 once per workgroup, four to eight steps ahead, across
// the ends of the convolutions too. Convolutions are direct: nine shifted products whose rows past the board's edge read a row
// of zeros. Four times the multiplications of winograd F(4x4,3x3), but no transforms, no winograd domain in memory (2 x 38 MB
// per convolution at 512 positions) and no launches; and sums in float over all of a convolution, where the winograd products
// of a half tower are rounded to halves twice.
//
// Split: with one wave per SIMD each takes 64 channels of all rows, so that a weight fragment and a row fragment are both used
// twice or more (two positions, a 64-byte step: 512 cycles of products, 256 of LDS reads, 256 of weights at 64 bytes a cycle); half
// the channels per wave would read the rows twice as often. One position per workgroup has half the products for the same
// weights and serves up to one round of the CUs.
// What bounds it: with two positions the matrix cores are busy 64 % of a wave's 2.34 M cycles (20x256 tower, 512 positions). By phases the
// convolutions take 75 % (their waits included), squeeze-and-excitation 16 % (192 KiB of float weights per block and workgroup, four
// barriers: 19 k cycles a block where the weights alone take 3 k), biases, skip and activations 9 %; with all CUs busy the clock falls to
// 1.9 GHz on top. One position: 71, 20 and 8 %. A round of 512 positions takes 1.21 ms (1.3 PFLOP/s of direct products), where 41
// transforms of 24 us and 40 launches of 36 x 2048x256x256 of 22 us took 1.86.
// Tried and not kept: the next squeeze-and-excitation weights touched during a convolution, so that they wait in the L2 (the stream
// waits for them in order: 512 positions 1558 -> 1727 us a pass); zeros in the banks of the rows they stand for (level).
// ---------------------------------------------------------------------------
template <int C, int POS>
__global__ __launch_bounds__(64 * kWaves, 1) void resident_tower_kernel(TowerArgs p) {
  using S = TowerShape<C>;
  constexpr int V = S::V, KS = S::KS, CT = S::CT, LD = S::LD, R = 64 * POS;
  constexpr int THREADS = 64 * kWaves;
  constexpr int TILE = S::TILE, SUB = S::SUB, F = S::F, RT = R / TILE, PT = RT / POS;   // a wave's row tiles, of a position
  constexpr int Q = TILE * TILE / 256;                   // a lane's output channels of a tile: Q times four, 8 apart
  constexpr int kRing = POS == 1 ? 8 : 4;                // steps of weights in flight
  constexpr int H = POS == 1 ? SUB : 1, ST = SUB / H;    // fragments of a tile that are read ahead together, and such reads in a step
  constexpr int kOther = R * LD, kZero = 2 * R * LD;     // the two activation buffers, then a row of zeros
  __shared__ __attribute__((aligned(16))) half_t lds[2 * R * LD + LD];
  __shared__ __attribute__((aligned(16))) float pool[POS][C];
  __shared__ float hidden[POS][kTowerMaxSe];
  __shared__ __attribute__((aligned(16))) float biases[2][C];   // of this convolution and the next
  __shared__ __attribute__((aligned(16))) float scale_shift[POS][2][C];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane % TILE, g = lane / TILE;
  const int pos0 = blockIdx.x * POS;
  const int ch0 = wave * TILE * CT + 4 * g;              // this lane's first output channel

  const long long steps = S::STEPS_IN + 2LL * p.blocks * S::STEPS;
  const intx4* ws = reinterpret_cast<const intx4*>(p.packed) + wave * steps * F * 64 + lane;
  intx4 w[kRing][F];
#pragma unroll
  for (int j = 0; j < kRing; j++)
#pragma unroll
    for (int f = 0; f < F; f++) w[j][f] = ws[(j * F + f) * 64];

  // Planes of the positions into the second buffer.
  {
    constexpr int PER_ROW = kPlanes / V, STRIDE = THREADS / PER_ROW;
    const int v = tid % PER_ROW;
#pragma unroll
    for (int q = 0; q < POS; q++) {
      const long long at = (long long)min(pos0 + q, p.batch - 1) * 112;
      uint64_t mask[V];
      half_t value[V];
#pragma unroll
      for (int e = 0; e < V; e++) {
        const int plane = v * V + e;
        mask[e] = plane < 112 ? p.masks[at + plane] : 0;
        value[e] = (half_t)(plane < 112 ? p.values[at + plane] : 0.0f);
      }
      for (int sq = tid / PER_ROW; sq < 64; sq += STRIDE) {
        half_t x[V];
#pragma unroll
        for (int e = 0; e < V; e++) x[e] = ((mask[e] >> sq) & 1) ? value[e] : (half_t)0.0f;
        *reinterpret_cast<intx4*>(lds + kOther + (q * 64 + sq) * LD + v * V) = *reinterpret_cast<const intx4*>(x);
      }
    }
    if (tid < LD / V) *reinterpret_cast<intx4*>(lds + kZero + tid * V) = intx4{0, 0, 0, 0};
    if (tid < C) biases[0][tid] = p.biases[tid];
  }
  __syncthreads();

  floatx16 acc[RT][CT];
  // acc = the convolution of the rows at src (element offset), NS_ steps per tap, STEPS_ in all.
  auto convolve = [&](int src, auto ns, auto total) {
    constexpr int NS_ = decltype(ns)::value, STEPS_ = decltype(total)::value;
    int at[RT];
    auto aim = [&](int tap) {
      const int dy = tap / 3 - 1, dx = tap - tap / 3 * 3 - 1, x = (r & 7) + dx;
#pragma unroll
      for (int t = 0; t < RT; t++) {
        const int y = ((TILE * t + r) >> 3 & 7) + dy;
        const bool on = (unsigned)x < 8u && (unsigned)y < 8u && tap < 9;
        at[t] = (on ? src + (t / PT * 64 + y * 8 + x) * LD : kZero) + V * g;
      }
    };
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int c = 0; c < CT; c++) acc[t][c] = floatx16{};
    intx4 a[2][RT][H];
    auto load_rows = [&](intx4 (&x)[RT][H], int s, int u0) {
#pragma unroll
      for (int h = 0; h < H; h++)
#pragma unroll
        for (int t = 0; t < RT; t++) x[t][h] = *reinterpret_cast<const intx4*>(lds + at[t] + s * KS + (u0 + h) * (KS / SUB));
    };
    aim(0);
    load_rows(a[0], 0, 0);
    for (int base = 0; base < STEPS_; base += kChunk) {
#pragma unroll
      for (int j = 0; j < kChunk; j++) {
#pragma unroll
        for (int st = 0; st < ST; st++) {
          const int now = (j * ST + st) & 1;
          if (st == ST - 1 && (j + 1) % NS_ == 0) aim((base + j + 1) / NS_);   // (past the last tap: the zeros, not used)
          load_rows(a[now ^ 1], (j + (st + 1) / ST) % NS_, (st + 1) % ST * H);
#pragma unroll
          for (int h = 0; h < H; h++)
#pragma unroll
            for (int t = 0; t < RT; t++)
#pragma unroll
              for (int c = 0; c < CT; c++)
                acc[t][c] = Mfma32(__builtin_bit_cast(half8, w[j % kRing][c * SUB + st * H + h]), __builtin_bit_cast(half8, a[now][t][h]),
                                   acc[t][c]);
          if (st == ST - 1) {
#pragma unroll
            for (int f = 0; f < F; f++) w[j % kRing][f] = ws[((j + kRing) * F + f) * 64];
          }
          // The next rows go out one by one between these products, and nothing moves past them (the compiler's own order reads a
          // fragment right before its products and waits for it).
#pragma unroll
          for (int i = 0; i < RT * H; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      ws += kChunk * F * 64;
    }
  };
  // Output channels ch0 + TILE c + 8 q .. + 3: element 4 q .. + 3 of acc[.][c].
  auto bias4 = [&](int conv, int c, int q) { return *reinterpret_cast<const floatx4*>(&biases[conv & 1][ch0 + TILE * c + 8 * q]); };
  float next_bias = 0.0f;
  auto ask_bias = [&](int conv) { next_bias = p.biases[(long long)min(conv, 2 * p.blocks) * C + tid % C]; };
  auto keep_bias = [&](int conv) {
    if (tid < C) biases[conv & 1][tid] = next_bias;
  };
  auto four = [&](int t, int c, int q) {
    return floatx4{acc[t][c][4 * q], acc[t][c][4 * q + 1], acc[t][c][4 * q + 2], acc[t][c][4 * q + 3]};
  };
  auto store = [&](int dst, int t, int c, int q, const floatx4& v) {
    *reinterpret_cast<half4*>(lds + dst + (TILE * t + r) * LD + ch0 + TILE * c + 8 * q) = half4{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
  };

  auto plain_tail = [&](int conv, int dst) {
    TowerAct(p.act, [&](auto act) {
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
          for (int q = 0; q < Q; q++) {
            const floatx4 v = four(t, c, q) + bias4(conv, c, q);
            store(dst, t, c, q, floatx4{act(v[0]), act(v[1]), act(v[2]), act(v[3])});
          }
    });
    keep_bias(conv + 1);
    __syncthreads();
  };
  ask_bias(1);
  convolve(kOther, std::integral_constant<int, S::NS_IN>(), std::integral_constant<int, S::STEPS_IN>());
  plain_tail(0, 0);

  for (int conv = 1; conv <= 2 * p.blocks; conv++) {
    const bool second = (conv & 1) == 0;
    ask_bias(conv + 1);
    convolve(second ? kOther : 0, std::integral_constant<int, S::NS>(), std::integral_constant<int, S::STEPS>());
    if (!second) {
      plain_tail(conv, kOther);
      continue;
    }
    const TowerSe se = p.se[conv / 2 - 1];
    if (se.k > 0) {
      // First layer: a wave does 16 hidden values, lane l value l % 16 and every fourth vector of the channels. Second layer: a
      // thread does four outputs and every KP-th hidden value. What comes from memory is asked for ahead: biases and first-layer weights
      // before the pooling, the second layer's first weights before the first layer with one position (kEarly) and, for want of
      // registers, after it with two. (Scheduling barriers keep the compiler from reading all of a layer's operands at once with two
      // positions: 37 spilled registers -> 13. us of a 20x256 pass, biases read where they are added and the weights after the first layer -> this: 17
      // positions 712 -> 657, 64 712 -> 656, 256 938 -> 890, 400 1384 -> 1306, 512 1533 -> 1498, 1000 2975 -> 2891.)
      constexpr bool kEarly = POS == 1;
      constexpr int B2 = 2 * C / THREADS;
      static_assert(2 * C % THREADS == 0, "whole rounds of threads over the outputs");
      constexpr int S1 = C / 16, O4 = 2 * C / 4, KP = THREADS / O4, U = 16;
      const int k_lane = lane & 15, v_lane = lane >> 4, o4 = tid % O4, kp = tid / O4;
      floatx4 w1[S1], w2[U];
      float b1, b2[B2];
#pragma unroll
      for (int j = 0; j < B2; j++) b2[j] = se.b2[tid + j * THREADS];
      auto load_w1 = [&](int k0) {
        b1 = se.b1[min(k0 + k_lane, se.k - 1)];
        const float* w = se.w1 + (long long)min(k0 + k_lane, se.k - 1) * C + 4 * v_lane;
#pragma unroll
        for (int i = 0; i < S1; i++) w1[i] = *reinterpret_cast<const floatx4*>(w + 16 * i);
      };
      auto load_w2 = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; u++)
          w2[u] = *reinterpret_cast<const floatx4*>(se.w2 + (long long)min(k0 + u * KP, se.k - 1) * 2 * C + 4 * o4);
      };
      load_w1(16 * wave);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < POS; b++)
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
          for (int q = 0; q < Q; q++) {
            const floatx4 bias = bias4(conv, c, q);
            floatx4 s = four(b * PT, c, q);
#pragma unroll
            for (int t = 1; t < PT; t++) s += four(b * PT + t, c, q);
#pragma unroll
            for (int e = 0; e < 4; e++) {
              s[e] = Sum32(s[e]) * (1.0f / 64.0f) + bias[e];
            }
            if (r == TILE - 16) *reinterpret_cast<floatx4*>(&pool[b][ch0 + TILE * c + 8 * q]) = s;
          }
      if constexpr (kEarly) {
        __builtin_amdgcn_sched_barrier(0);
        load_w2(kp);
      }
      __syncthreads();
      for (int k0 = 16 * wave; k0 < se.k; k0 += 16 * kWaves) {
        if (k0 > 16 * wave) load_w1(k0);
#pragma unroll
        for (int b = 0; b < POS; b++) {
          floatx4 h4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int i = 0; i < S1; i++) {
            h4 += w1[i] * *reinterpret_cast<const floatx4*>(&pool[b][16 * i + 4 * v_lane]);
            if (POS > 1 && i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
          }
          float h = (h4[0] + h4[1]) + (h4[2] + h4[3]);
          h += __shfl_xor(h, 16, 64);
          h += __shfl_xor(h, 32, 64);
          const int k = k0 + k_lane;
          if (v_lane == 0 && k < se.k) TowerAct(p.act, [&](auto act) { hidden[b][k] = act(h + b1); });
        }
      }
      if (!kEarly) load_w2(kp);
      __syncthreads();
      floatx4 out[POS];
#pragma unroll
      for (int b = 0; b < POS; b++) out[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int k0 = kp; k0 < se.k; k0 += U * KP) {
        if (k0 > kp) load_w2(k0);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int b = 0; b < POS; b++) {
            const int k = k0 + u * KP;
            const float h = hidden[b][min(k, se.k - 1)];
            out[b] += w2[u] * (k < se.k ? h : 0.0f);
            if (POS > 1 && b + 1 == POS && u % 4 == 3) __builtin_amdgcn_sched_barrier(0);
          }
      }
      // The partial sums take the place of the block's inner activations: no wave reads those any more.
      float* part = reinterpret_cast<float*>(lds + kOther);
#pragma unroll
      for (int b = 0; b < POS; b++) *reinterpret_cast<floatx4*>(part + (kp * POS + b) * 2 * C + 4 * o4) = out[b];
      __syncthreads();
#pragma unroll
      for (int n = 0; n < POS * B2; n++) {
        const int i = tid + n * THREADS, b = i / (2 * C), o = i % (2 * C);
        float v = b2[n % B2];
#pragma unroll
        for (int j = 0; j < KP; j++) v += part[j * POS * 2 * C + i];
        scale_shift[b][o / C][o % C] = o < C ? 1.0f / (1.0f + __expf(-v)) : v;
      }
      __syncthreads();
    }
    TowerAct(p.act, [&](auto act) {
#pragma unroll
      for (int b = 0; b < POS; b++)
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
          for (int q = 0; q < Q; q++) {
            const int ch = ch0 + TILE * c + 8 * q;
            floatx4 gamma = {1.0f, 1.0f, 1.0f, 1.0f}, beta = bias4(conv, c, q);
            if (se.k > 0) {
              gamma = *reinterpret_cast<const floatx4*>(&scale_shift[b][0][ch]);
              beta = *reinterpret_cast<const floatx4*>(&scale_shift[b][1][ch]) + gamma * beta;
            }
#pragma unroll
            for (int t = b * PT; t < (b + 1) * PT; t++) {
              const half4 skip = *reinterpret_cast<const half4*>(lds + (TILE * t + r) * LD + ch);
              const floatx4 y = four(t, c, q);
              floatx4 v;
#pragma unroll
              for (int e = 0; e < 4; e++) v[e] = act(gamma[e] * y[e] + beta[e] + (float)skip[e]);
              store(0, t, c, q, v);
            }
          }
    });
    keep_bias(conv + 1);
    __syncthreads();
  }

  half_t* out = static_cast<half_t*>(p.out) + (long long)pos0 * 64 * C;
  for (int i = tid; i < R * (C / V); i += THREADS) {
    const int row = i / (C / V), v = i % (C / V);
    if (pos0 + row / 64 < p.batch)
      *reinterpret_cast<intx4*>(out + (long long)row * C + v * V) = *reinterpret_cast<const intx4*>(lds + row * LD + v * V);
  }
}

template <int C>
long long FragmentIndex(int blocks, int conv, int tap, int out, int in) {
  using S = TowerShape<C>;
  const long long steps = S::STEPS_IN + 2LL * blocks * S::STEPS;
  const int wave = out / (S::TILE * S::CT), c = out / S::TILE % S::CT, sub = in % S::KS / (S::G * S::V);
  const long long first = conv == 0 ? 0 : S::STEPS_IN + (conv - 1LL) * S::STEPS;
  const long long step = wave * steps + first + tap * (conv == 0 ? S::NS_IN : S::NS) + in / S::KS;
  return ((step * S::F + c * S::SUB + sub) * 64 + in / S::V % S::G * S::TILE + out % S::TILE) * S::V + in % S::V;
}
template <int C>
long long Fragments(int blocks) {   // (and a turn's worth that is asked for past the end)
  using S = TowerShape<C>;
  return ((S::STEPS_IN + 2LL * blocks * S::STEPS) * kWaves + kChunk) * S::F * 64 * S::V;
}

}  // namespace

// 64 float (resident_tower_f32.hip), 128 and 256 half filters. A wave takes whole tiles of TILE channels, so there are 128 n half
// filters (not 64); a turn of kChunk steps does whole taps, so a tap has one, two, four or eight (not 384).
bool TowerSupported(int filters, bool f32) { return f32 ? filters == 64 : filters == 128 || filters == 256; }

long long TowerFragments(int blocks, int filters) { return filters == 128 ? Fragments<128>(blocks) : Fragments<256>(blocks); }

long long TowerFragmentIndex(int blocks, int filters, int conv, int tap, int out, int in) {
  return filters == 128 ? FragmentIndex<128>(blocks, conv, tap, out, in) : FragmentIndex<256>(blocks, conv, tap, out, in);
}

// Where the kernel is faster than winograd convolutions, whose launches spread few positions over more CUs. us a batch through the
// interface, winograd / this. 20x256 halves 32 positions 850 / 702,
// 200 1426 / 840, 512 2146 / 1571, 1000 3505 / 3061; 10x256 without squeeze-and-excitation 13 299 / 309, 17 328 / 307, 64 454 / 319, 512
// 1158 / 876, 1000 1993 / 1606; 10x128 1 284 / 195, 8 302 / 199, 64 392 / 217, 256 655 / 319, 512 915 / 518, 1000 1338 / 963, mish without
// squeeze-and-excitation 8 261 / 183, 1000 1332 / 929; thousands of evals/s of two and of four threads, 20x256 halves 17 40 / 44 and 58 / 66, 64
// 120 / 163 and 156 / 247, 512 313 / 366 and 321 / 406.
// 64 floats: 6 blocks 1 position 172 / 124, 32 225 / 139, 256 509 / 269, 512 708 / 486, 1000 1133 / 892, of four threads 1 15.1 / 17.5, 32 349 / 519,
// 256 1267 / 2018, 1000 1602 / 2352; 2 blocks 1 102 / 86, 24 125 / 94, 1000 848 / 745. One block, more than half of it the input
// convolution, gains less (24 103 / 84, four threads 508 / 503; 257 263 / 234) and keeps to the batches of one round.
// 256 half filters with squeeze-and-excitation, since its weights are asked for ahead: 20 blocks 1 position 645 / 630, 4 662 / 667, 8 684 / 670, 16
// 740 / 660, of four threads 4.3 / 4.5, 8 30.4 / 33.4, 16 55 / 68; 10 blocks 1 337 / 321, 16 369 / 342, 2 blocks 8 126 / 125; without it 20 blocks 1
// 456 / 500, 16 514 / 528, 4 blocks 8 154 / 160.
bool TowerFaster(int batch, int filters, bool f32, int blocks, bool se) {
  if (f32) return blocks > 1 || (batch > 24 && batch <= 256);
  return filters <= 128 || batch > 16 || (se && blocks > 1);
}

namespace {
template <int C, int POS>
void LaunchTowerT(TowerArgs a, int first, int count, hipStream_t stream) {
  if (count <= 0) return;
  a.masks += 112LL * first;
  a.values += 112LL * first;
  a.out = static_cast<half_t*>(a.out) + 64LL * C * first;
  a.batch = count;
  resident_tower_kernel<C, POS><<<dim3((count + POS - 1) / POS), dim3(64 * kWaves), 0, stream>>>(a);
}
}  // namespace

// Full rounds of 256 workgroups with two positions each, then the rest, with one position each where that makes one round
// of cheaper workgroups (20x256: a round of one 0.8 ms, of two 1.4 ms).
void LaunchTower(const TowerArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  if (a.blocks < 1 || (a.act != kActMish && a.act != kActRelu) || !TowerSupported(a.filters, false)) {
    throw std::runtime_error("LaunchTower: no kernel");
  }
  const int rest = a.batch % 512, pairs = rest > 256 ? a.batch : a.batch - rest;
  if (a.filters == 128) {
    LaunchTowerT<128, 2>(a, 0, pairs, stream);
    LaunchTowerT<128, 1>(a, pairs, a.batch - pairs, stream);
  } else {
    LaunchTowerT<256, 2>(a, 0, pairs, stream);
    LaunchTowerT<256, 1>(a, pairs, a.batch - pairs, stream);
  }
}

}  // namespace lc0mi
