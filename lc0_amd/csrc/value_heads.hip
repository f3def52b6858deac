// Heads of 16-bit attention bodies: value and moves-left heads in one kernel (embedding layer, first and second dense layer), the
// attention policy from its query and key vectors on, and both in one launch.
// Replaces three calls of FullyConnectedLayer::Forward1D per head: blas/network_blas.cc:725-772, and the logits, promotion
// offsets and the gather of the policy: blas/network_blas.cc:850-914.
#include "kernel_common.h"
#include "row_panel.h"

#include <algorithm>

#include <stdexcept>

namespace lc0mi {

namespace {

constexpr int kHeadWaves = 8, kHeadCh = 32, kHeadFc = 16 * kHeadWaves, kHeadChunk = 256, kHeadAhead = 16;

// ---------------------------------------------------------------------------
// A workgroup does one head (blockIdx.y) of one position. Embedding: wave w multiplies 16 squares (w % 4) with 16 channels
// (w / 4), 256 columns at a time from LDS. First dense layer: 16 columns per wave, the one row broadcast from LDS, its weights
// sixteen fragments ahead and asked for before anything else is known. Second: one output per wave. Weights lie in
// fragments of 16 outputs x 32 inputs in the order of use (lane l: output l % 16, inputs 8 (l / 16) ... + 7).
//
// As launches of their own the six products are 4 to 5 us each in a chain of dependent ones, for operands of 0.1 to 0.5 MB.
// Bound by latency and by what a CU takes from L2: 0.7 MB a workgroup at width 1024, 0.5 MB of them the value head's
// first-layer weights. us back to back, both heads: width 256 1 position 8.5, 64 9.2, 256 12.1; width 1024 10.6, 11.5, 22.4.
// (A form that took row-major weights with the loads of row_panel.h spilled, and took 18 to 29 us at up to 64 positions.)
// ---------------------------------------------------------------------------
template <typename ET, int NC> struct ValueHeadLds {
  __attribute__((aligned(16))) ET rows[NC > 1 ? 2 : 1][64 * (kHeadChunk + 8)];
  __attribute__((aligned(16))) ET embedded[64 * kHeadCh];
  float hidden[kHeadFc];
};

template <typename ET, int NC>   // NC chunks of 256 columns of x
__device__ __forceinline__ void ValueHead(const ValueHeadsArgs& p, const HeadLayers& h, ValueHeadLds<ET, NC>& lds) {
  using ev8 = typename Vec16<ET>::v8;
  constexpr int LD = kHeadChunk + 8, VX = 64 * kHeadChunk / 8 / (64 * kHeadWaves), SC = kHeadChunk / 32;
  auto& rows = lds.rows;
  auto& embedded = lds.embedded;
  auto& hidden = lds.hidden;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int ch = h.ch;
  const half_t* x = p.x + (long long)blockIdx.x * 64 * p.ldx;

  intx4 xv[NC][VX];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int i = 0; i < VX; i++) {
      const int at = i * 64 * kHeadWaves + tid;
      xv[c][i] = *reinterpret_cast<const intx4*>(x + (long long)(at / 32) * p.ldx + c * kHeadChunk + at % 32 * 8);
    }
  const int tile = wave >> 2, sq = (wave & 3) * 16 + r;
  const intx4* we_src = reinterpret_cast<const intx4*>(h.w_embed) + tile * NC * SC * 64 + lane;
  intx4 we[SC];
#pragma unroll
  for (int s = 0; s < SC; s++) we[s] = we_src[s * 64];
  const int rounds = (ch + 7) / 8;   // of sixteen fragments
  const intx4* w1_src = reinterpret_cast<const intx4*>(h.w_fc1) + wave * rounds * kHeadAhead * 64 + lane;
  intx4 w1[kHeadAhead];
#pragma unroll
  for (int s = 0; s < kHeadAhead; s++) w1[s] = w1_src[s * 64];
  // (the flat row is square * ch + channel: zeros up to a whole round)
  for (int at = 64 * ch + tid; at < 512 * rounds; at += 64 * kHeadWaves) embedded[at] = (ET)0.0f;

  floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < NC; c++) {
#pragma unroll
    for (int i = 0; i < VX; i++) {
      const int at = i * 64 * kHeadWaves + tid;
      *reinterpret_cast<intx4*>(rows[c & 1] + at / 32 * LD + at % 32 * 8) = xv[c][i];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SC; s++) {
      const ev8 a = *reinterpret_cast<const ev8*>(rows[c & 1] + sq * LD + 32 * s + 8 * g);
      acc = Mfma16(__builtin_bit_cast(ev8, we[s]), a, acc);
      if (c + 1 < NC) we[s] = we_src[((c + 1) * SC + s) * 64];
    }
  }
  float bias[4];
  LoadBias4(h.b_embed, 16 * tile + 4 * g, ch, bias);
  DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int c = 16 * tile + 4 * g + e;
      if (c < ch) embedded[sq * ch + c] = (ET)act_fn(acc[e] + bias[e]);
    }
  });
  __syncthreads();

  floatx4 sum[2] = {};
  for (int n = 0; n < rounds; n++) {
    if (n + 1 < rounds) w1_src += kHeadAhead * 64;   // (after the last round its own weights once more)
#pragma unroll
    for (int s = 0; s < kHeadAhead; s++) {
      const ev8 a = *reinterpret_cast<const ev8*>(embedded + (n * kHeadAhead + s) * 32 + 8 * g);
      sum[s & 1] = Mfma16(__builtin_bit_cast(ev8, w1[s]), a, sum[s & 1]);
      w1[s] = w1_src[s * 64];
    }
  }
  if (r == 0) {   // (every row of the tile is the same one)
    const int n = 16 * wave + 4 * g;
    LoadBias4(h.b_fc1, n, h.fc, bias);
    DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
      for (int e = 0; e < 4; e++) hidden[n + e] = act_fn(sum[0][e] + sum[1][e] + bias[e]);
    });
  }
  __syncthreads();
  for (int o = wave; o < h.out_n; o += kHeadWaves) {
    const ET* w2 = reinterpret_cast<const ET*>(h.w_fc2) + (long long)o * h.ld_fc2;
    float v = 0.0f;
    for (int k = lane; k < h.fc; k += 64) v += hidden[k] * (float)w2[k];
    v = WaveSum(v) + (h.b_fc2 != nullptr ? h.b_fc2[o] : 0.0f);
    if (lane == 0) h.out[(long long)blockIdx.x * h.out_n + o] = Activate(v, h.out_act);
  }
}

// ---------------------------------------------------------------------------
// Policy of one position by a workgroup: logits[q][k] = scale Q_q . K_k (64 x 64, float), the offsets of the three promotion pieces from
// the last eight keys, and the 1858 moves' values gathered from both. The eight waves share the reduction, 128 columns at a time
// (with at most 256 columns in all two of them share it, and each of four takes 16 keys); operands straight from memory in the order
// of row_panel.h, sums of two waves each added in LDS, the four that remain where they are gathered.
// Bound by latency with few positions, where the products and the gather as launches of their own are 5 to 10 us each in the chain; beside
// the value heads it is hidden by them. us back to back, depth 1024: 1 position 9.0, 64 9.9, 256 15.8 (the products alone on tiles 14.9, the
// gather 10 more), 1024 54 (46 and 20); depth 256: 5.9, 6.5, 7.1, 26. us of a pass, three launches -> one: 15x1024 fp16 1 position 828 -> 809, 16
// 1239 -> 1224, 48 2082 -> 2066, bf16 64 2168 -> 2153, e4m3 16 918 -> 904; 10x256 1 272 -> 255, 64 365 -> 353; level from 100 positions on.
// ---------------------------------------------------------------------------
constexpr int kLogitStride = 64 + 4;
struct PolicyLds {
  __attribute__((aligned(16))) float part[4][64 * kLogitStride];
  float offset[4][8];
};

template <typename ET>
__device__ __forceinline__ void PolicyTail(const PolicyTailArgs& p, PolicyLds& lds) {
  using ev8 = typename Vec16<ET>::v8;
  constexpr int kMoves = 1858, kPerThread = (kMoves + 64 * kHeadWaves - 1) / (64 * kHeadWaves);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const half_t* rows = p.qk + (long long)blockIdx.x * 64 * p.ld;
  int source[kPerThread];
#pragma unroll
  for (int i = 0; i < kPerThread; i++) source[i] = p.inv_map[min(i * 64 * kHeadWaves + tid, kMoves - 1)];

  // Promotion offsets: key 56 + wave against the four rows of ppo.
  {
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const half_t* key = rows + (long long)(56 + wave) * p.ld + p.key_offset;
    for (int c = lane; c < p.depth / 8; c += 64) {
      const ev8 kv = *reinterpret_cast<const ev8*>(key + c * 8);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const floatx4 p0 = *reinterpret_cast<const floatx4*>(p.ppo + (long long)i * p.depth + c * 8);
        const floatx4 p1 = *reinterpret_cast<const floatx4*>(p.ppo + (long long)i * p.depth + c * 8 + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) s[i] += (float)kv[e] * p0[e] + (float)kv[4 + e] * p1[e];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float t = WaveSum(s[i]);
      if (lane == 0) lds.offset[i][wave] = t;
    }
  }

  const int row_bytes = 2 * p.depth, steps = (row_bytes + kStepBytes - 1) / kStepBytes;
  const char* queries = reinterpret_cast<const char*>(rows);
  const char* keys = reinterpret_cast<const char*>(rows + p.key_offset);
  TileOffsets at[4];
#pragma unroll
  for (int t = 0; t < 4; t++) at[t].Set(16 * t, 64, 2 * p.ld);
  auto left = [&](int step) { return min(kStepBytes, row_bytes - step * kStepBytes); };
  int parts = 4;
  if (steps > 2) {
    floatx4 acc[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int c = 0; c < 4; c++) acc[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = wave; s < steps; s += kHeadWaves)
      OneStep<4, 4>(queries + s * kStepBytes, at, keys + s * kStepBytes, at, left(s), acc, PanelOp<ET>{});
    // Accumulator lane (r, g) of tile (t, c): query 16 t + r, keys 16 c + 4 g + e.
    auto place = [&](int t, int c) { return reinterpret_cast<floatx4*>(&lds.part[wave & 3][(16 * t + r) * kLogitStride + 16 * c + 4 * g]); };
    if (wave >= 4) {
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) *place(t, c) = acc[t][c];
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) *place(t, c) = acc[t][c] + *place(t, c);
    }
  } else {
    parts = 2;
    const int s = wave >> 2, c = wave & 3;
    floatx4 acc[4][1];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t][0] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    TileOffsets mine[1];
    mine[0].Set(16 * c, 64, 2 * p.ld);
    if (s < steps) OneStep<4, 1>(queries + s * kStepBytes, at, keys + s * kStepBytes, mine, left(s), acc, PanelOp<ET>{});
#pragma unroll
    for (int t = 0; t < 4; t++) *reinterpret_cast<floatx4*>(&lds.part[s][(16 * t + r) * kLogitStride + 16 * c + 4 * g]) = acc[t][0];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPerThread; i++) {
    const int move = i * 64 * kHeadWaves + tid;
    const bool plain = source[i] < 4096;
    const int q = plain ? 0 : source[i] - 4096, k = q / 24, j = q % 24 / 3, piece = q % 3;   // promotion from file k to file j
    const int cell = plain ? (source[i] >> 6) * kLogitStride + (source[i] & 63) : (48 + k) * kLogitStride + 56 + j;
    float v = lds.part[0][cell] + lds.part[1][cell];
    if (parts == 4) v += lds.part[2][cell] + lds.part[3][cell];
    v *= p.scale;
    if (!plain) v = v + lds.offset[piece][j] + lds.offset[3][j];
    if (move < kMoves) p.out[(long long)blockIdx.x * kMoves + move] = v;
  }
}

// Value and moves-left head, and with `policy` the policy: a workgroup each per position.
template <typename ET, int NC>
__global__ __launch_bounds__(64 * kHeadWaves) void value_heads_kernel(ValueHeadsArgs p) {
  __shared__ union { ValueHeadLds<ET, NC> head; PolicyLds policy; } lds;
  if ((int)blockIdx.y < p.heads) ValueHead<ET, NC>(p, p.head[blockIdx.y], lds.head);
  else PolicyTail<ET>(p.policy, lds.policy);
}

template <typename ET>
__global__ __launch_bounds__(64 * kHeadWaves) void policy_tail_kernel(PolicyTailArgs p) {
  __shared__ PolicyLds lds;
  PolicyTail<ET>(p, lds);
}

template <typename ET>
void LaunchValueHeadsT(const ValueHeadsArgs& a, hipStream_t stream) {
  const dim3 grid(a.batch, a.heads + (a.policy.qk != nullptr ? 1 : 0)), block(64 * kHeadWaves);
  switch (a.emb / kHeadChunk) {
    case 1: hipLaunchKernelGGL((value_heads_kernel<ET, 1>), grid, block, 0, stream, a); break;
    case 2: hipLaunchKernelGGL((value_heads_kernel<ET, 2>), grid, block, 0, stream, a); break;
    case 3: hipLaunchKernelGGL((value_heads_kernel<ET, 3>), grid, block, 0, stream, a); break;
    default: hipLaunchKernelGGL((value_heads_kernel<ET, 4>), grid, block, 0, stream, a); break;
  }
}
}  // namespace

bool ValueHeadSupported(int emb, int ch, int fc, int out_n) {
  return emb % kHeadChunk == 0 && emb >= kHeadChunk && emb <= 4 * kHeadChunk && ch >= 1 && ch <= kHeadCh && fc >= 1 && fc <= kHeadFc &&
         out_n >= 1;
}

long long HeadFragments(bool embed, int emb, int ch) {
  return embed ? 2LL * emb / 32 * 512 : (long long)kHeadWaves * kHeadAhead * ((ch + 7) / 8) * 512;
}

long long HeadFragmentIndex(bool embed, int row, int col, int emb, int ch) {
  const int steps = embed ? emb / 32 : kHeadAhead * ((ch + 7) / 8);
  return ((long long)(row / 16 * steps + col / 32) * 64 + row % 16 + 16 * (col % 32 / 8)) * 8 + col % 8;
}

bool PolicyTailSupported(const PolicyTailArgs& a) {
  return a.depth >= 8 && a.depth % 8 == 0 && a.ld % 8 == 0 && a.key_offset % 8 == 0 && a.ld <= 1 << 20;
}

void LaunchPolicyTail(const PolicyTailArgs& a, int batch, bool bf16, hipStream_t stream) {
  if (batch <= 0) return;
  if (!PolicyTailSupported(a)) throw std::runtime_error("LaunchPolicyTail: unsupported shape");
  const dim3 grid(batch), block(64 * kHeadWaves);
  if (bf16) hipLaunchKernelGGL(policy_tail_kernel<bf16_t>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(policy_tail_kernel<half_t>, grid, block, 0, stream, a);
}

void LaunchValueHeads(const ValueHeadsArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  bool ok = a.heads >= 1 && a.heads <= 2 && a.ldx % 8 == 0;
  for (int i = 0; ok && i < a.heads; i++) ok = ValueHeadSupported(a.emb, a.head[i].ch, a.head[i].fc, a.head[i].out_n);
  if (a.policy.qk != nullptr) ok = ok && PolicyTailSupported(a.policy);
  if (!ok) throw std::runtime_error("LaunchValueHeads: unsupported shape");
  if (a.bf16) LaunchValueHeadsT<bf16_t>(a, stream);
  else LaunchValueHeadsT<half_t>(a, stream);
}

}  // namespace lc0mi
