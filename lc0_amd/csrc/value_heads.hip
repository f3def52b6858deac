// Value and moves-left heads of 16-bit attention bodies in one kernel: embedding layer, first and second dense layer.
// Replaces three calls of FullyConnectedLayer::Forward1D per head: blas/network_blas.cc:725-772.
#include "kernel_common.h"

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
template <typename ET, int NC>   // NC chunks of 256 columns of x
__global__ __launch_bounds__(64 * kHeadWaves) void value_heads_kernel(ValueHeadsArgs p) {
  using ev8 = typename Vec16<ET>::v8;
  constexpr int LD = kHeadChunk + 8, VX = 64 * kHeadChunk / 8 / (64 * kHeadWaves), SC = kHeadChunk / 32;
  __shared__ __attribute__((aligned(16))) ET rows[NC > 1 ? 2 : 1][64 * LD];
  __shared__ __attribute__((aligned(16))) ET embedded[64 * kHeadCh];
  __shared__ float hidden[kHeadFc];
  const HeadLayers& h = p.head[blockIdx.y];
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

template <typename ET>
void LaunchValueHeadsT(const ValueHeadsArgs& a, hipStream_t stream) {
  const dim3 grid(a.batch, a.heads), block(64 * kHeadWaves);
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

void LaunchValueHeads(const ValueHeadsArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  bool ok = a.heads >= 1 && a.heads <= 2 && a.ldx % 8 == 0;
  for (int i = 0; ok && i < a.heads; i++) ok = ValueHeadSupported(a.emb, a.head[i].ch, a.head[i].fc, a.head[i].out_n);
  if (!ok) throw std::runtime_error("LaunchValueHeads: unsupported shape");
  if (a.bf16) LaunchValueHeadsT<bf16_t>(a, stream);
  else LaunchValueHeadsT<half_t>(a, stream);
}

}  // namespace lc0mi
