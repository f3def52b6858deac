// Row norm, smolgen generator and attention in one kernel for few positions: head depth 32, generator vectors of 256, a
// multiple of four heads up to 32:
//   y = beta + gamma (gen[b] - mean) / sqrt(var + eps) over the heads x 256 values of a position, rounded to 16 bits,
//   logits[b][h][q][k] = scale * Q.K^T + sum_j W[q*64+k][j] * y[h][j],  out = softmax_k(logits) . V
// (blas/network_blas.cc:326-347 with blas/encoder.h:29-66, then the attention, network_blas.cc:352-439).
#include "kernel_common.h"
#include "row_panel.h"

#include <stdexcept>
#include <type_traits>

namespace lc0mi {

namespace {

constexpr int kGen = 256, kNks = kGen / 16;
constexpr int kYStride = kGen + 8;                       // 16-bit values per head in LDS
constexpr int kVStride = 256 + 32;                       // bytes per key: the eight rows that 32 lanes read meet different banks

// ---------------------------------------------------------------------------
// A workgroup of eight waves owns QUERIES (4, 8 or 16) queries of one position and all heads, or with one to four positions a group of them.
//   Generator: the 64 QUERIES (query, key) rows are QUERIES / 4 32-row tiles per wave over the 32 heads as columns; weights in
//     the fragment order of smolgen_attention_kernel, asked for first, and the norm of the vectors while they are on their way.
//   Attention: four heads per wave. K comes in by 64-byte rows of the four heads and leaves the 4 x 4 transpose of row_panel.h as
//     lane (key r, head g), chunk j of the depth in register j. With a second operand that is Q's chunk j where the column's
//     head is g and zero elsewhere, four matrix instructions give the scores of 16 keys for 16 columns = 4 queries x 4
//     heads: no lane is idle in the softmax. V^T comes from a staged tile by transposing LDS loads; its products, head by
//     head, take probabilities that are zero outside the head's columns. Four queries at a time, K and V^T stay in registers.
// Logits stay in float with up to 8 queries; with 16 they are rounded to 16 bits, as the generator layer of its own leaves them.
// Bound by latency and by what a workgroup takes from L2 (32 KiB of weights per query, K and V 256, gamma and beta 64): the
// fewest queries that give no CU two workgroups are the fastest (us back to back, 32 heads in one group: 4 queries 1 position 10.5, 16 11.6,
// 24 20.5; 8 queries 24 14.0, 32 15.1; 16 queries 33 20.1, 64 22.7).
// ---------------------------------------------------------------------------
template <typename ET, typename OutT, int QUERIES>
__global__ __launch_bounds__(512) void smolgen_attention_few_kernel(SmolgenFewArgs p) {
  using ev8 = typename Vec16<ET>::v8;
  using ev4 = typename Vec16<ET>::v4;
  using LT = std::conditional_t<QUERIES <= 8, float, ET>;   // logits: floats where they fit the LDS
  using lv4 = LT __attribute__((ext_vector_type(4)));
  constexpr int kLogitStride = QUERIES * 64 + (QUERIES <= 8 ? 4 : 8);
  constexpr int GROUPS = QUERIES / 4, SHIFT = QUERIES == 4 ? 4 : QUERIES == 8 ? 3 : 2;   // 64 / QUERIES = 1 << SHIFT workgroups a position
  __shared__ __attribute__((aligned(16))) ET y_lds[32 * kYStride];
  __shared__ __attribute__((aligned(16))) LT logits[32 * kLogitStride];
  __shared__ __attribute__((aligned(16))) unsigned char v_lds[8][32 * kVStride];
  __shared__ float part[2][8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups go to the 8 XCDs in turn. From 8 positions on those of a position share an XCD, whose L2 then holds its K and
  // V once; with fewer they are spread, or most of the chip's L2s would have nothing to fetch.
  // The last grid / groups workgroups do the last group of heads, and so on.
  const int per_group = gridDim.x / p.head_groups, group = blockIdx.x / per_group, id = blockIdx.x - group * per_group;
  constexpr int MASK = (1 << SHIFT) - 1;
  const int b = p.batch >= 8 ? (id >> (SHIFT + 3)) * 8 + (id & 7) : id >> SHIFT;
  const int q0 = QUERIES * (p.batch >= 8 ? (id >> 3) & MASK : id & MASK);
  if (b >= p.batch) return;
  const int heads = p.heads, d_model = 32 * heads, ld = 3 * d_model;
  const int first_head = group * (heads / p.head_groups), end_head = first_head + heads / p.head_groups;   // this workgroup's

  // What does not depend on anything: weights, generator vectors, gamma and beta, K and Q.
  const intx4* wp = reinterpret_cast<const intx4*>(p.wfrag) + (long long)(2 * q0 + GROUPS * wave) * kNks * 64 + lane;
  const int row0 = tid >> 5, kv = (tid & 31) * 8;        // rows (heads) row0 and row0 + 16, eight columns
  ev8 x[2];
  floatx4 gm[2][2], bt[2][2];
#pragma unroll
  for (int v = 0; v < 2; v++) {
    x[v] = *reinterpret_cast<const ev8*>(p.gen + ((long long)b * heads + min(row0 + 16 * v, heads - 1)) * kGen + kv);
    const int at = min(max(row0 + 16 * v, first_head), end_head - 1) * kGen + kv;   // (other heads' are not used)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      gm[v][h] = *reinterpret_cast<const floatx4*>(p.gamma + at + 4 * h);
      bt[v][h] = *reinterpret_cast<const floatx4*>(p.beta + at + 4 * h);
    }
  }
  intx4 w[kNks];
#pragma unroll
  for (int s = 0; s < kNks; s++) w[s] = wp[s * 64];
  const int r = lane & 15, g = lane >> 4;
  const int head0 = first_head + 4 * wave;
  const bool live = head0 < end_head;                    // (a multiple of four heads: whole waves)
  const half_t* base = p.qkv + (long long)b * 64 * ld + (live ? head0 : first_head) * 32;
  intx4 k[4][4];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int i = 0; i < 4; i++)
      k[t][i] = *reinterpret_cast<const intx4*>(base + d_model + (unsigned)(16 * t + 4 * ((lane >> 2) & 3) + i) * (unsigned)ld +
                                                32 * g + 8 * (lane & 3));  // Column c = lane % 16 of a group is its query c % 4 of head c / 4: Q's chunk j where that is this lane's head g, else zero.
  const int hh = r >> 2;
  const half_t* qp = base + (unsigned)(q0 + (r & 3)) * (unsigned)ld + 32 * hh;
  intx4 q[4];
#pragma unroll
  for (int j = 0; j < 4; j++) q[j] = *reinterpret_cast<const intx4*>(qp + 8 * j);

  // Norm of the position's vectors.
  {
    const float inv = 1.0f / (float)(heads * kGen);
    auto block_sum = [&](float v, float (&at)[8]) {
      v = WaveSum(v);
      if (lane == 0) at[wave] = v;
      __syncthreads();
      return ((at[0] + at[1]) + (at[2] + at[3])) + ((at[4] + at[5]) + (at[6] + at[7]));
    };
    float s = 0.0f;
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 8; e++) s += row0 + 16 * v < heads ? (float)x[v][e] : 0.0f;
    const float mean = block_sum(s, part[0]) * inv;
    float m2 = 0.0f;
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float d = row0 + 16 * v < heads ? (float)x[v][e] - mean : 0.0f;
        m2 = fmaf(d, d, m2);
      }
    const float rstd = 1.0f / sqrtf(block_sum(m2, part[1]) * inv + p.eps);
#pragma unroll
    for (int v = 0; v < 2; v++) {
      ev8 o;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float f = bt[v][e / 4][e % 4] + gm[v][e / 4][e % 4] * ((float)x[v][e] - mean) * rstd;
        o[e] = row0 + 16 * v < heads ? (ET)f : (ET)0.0f;
      }
      *reinterpret_cast<ev8*>(y_lds + (row0 + 16 * v) * kYStride + kv) = o;
    }
  }
  __syncthreads();

  // Generator: GROUPS times 32 (query, key) rows of this wave times 32 heads, the next rows' weights in place of used ones.
  {
    const int c = lane & 31, hi = lane >> 5;
#pragma unroll
    for (int i = 0; i < GROUPS; i++) {
      floatx16 acc;
#pragma unroll
      for (int e = 0; e < 16; e++) acc[e] = 0.0f;
#pragma unroll
      for (int s = 0; s < kNks; s++) {
        const ev8 y = *reinterpret_cast<const ev8*>(y_lds + c * kYStride + 16 * s + 8 * hi);
        acc = Mfma32(__builtin_bit_cast(ev8, w[s]), y, acc);
        if (i + 1 < GROUPS) w[s] = wp[((i + 1) * kNks + s) * 64];
      }
      // register 4 n + e of lane (head c, hi): row 8 n + 4 hi + e of the tile
      const int tile = GROUPS * wave + i;   // query tile / 2, keys from 32 (tile % 2)
#pragma unroll
      for (int n = 0; n < 4; n++)
        *reinterpret_cast<lv4*>(logits + c * kLogitStride + tile * 32 + 8 * n + 4 * hi) =
            lv4{(LT)acc[4 * n], (LT)acc[4 * n + 1], (LT)acc[4 * n + 2], (LT)acc[4 * n + 3]};
    }
  }
  // V by whole 256-byte rows of the four heads, sixteen lanes a row.
  intx4 vr[16];
#pragma unroll
  for (int i = 0; i < 16; i++)
    vr[i] = *reinterpret_cast<const intx4*>(base + 2 * d_model + (unsigned)(4 * i + g) * (unsigned)ld + 8 * r);
  const intx4 zero = {0, 0, 0, 0};
  __syncthreads();
  if (!live) return;
#pragma unroll
  for (int t = 0; t < 4; t++) QuadTranspose(k[t]);
  // V^T as operands, 32 keys at a time through this wave's LDS: [32 keys][head][depth half], keys 32 s + 4 g + e and 16 further.
  ev8 vt[2][4][2];
  typedef short short4v __attribute__((ext_vector_type(4)));
  unsigned char* stage = v_lds[wave];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 8; i++) *reinterpret_cast<intx4*>(stage + (4 * i + g) * kVStride + 16 * r) = vr[8 * s + i];
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
      for (int dt = 0; dt < 2; dt++) {
        // (the transposing load: lane i of 16 receives D[4 e + i / 4][i % 4] of the 16 x 4 block whose row n lane n points at, so
        // here the keys 16 u + 4 g + e of depth 16 dt + i)
        short4v half[2];
#pragma unroll
        for (int u = 0; u < 2; u++)
          half[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v*)(
              stage + (16 * u + 4 * g + (r >> 2)) * kVStride + 64 * h + 32 * dt + 8 * (r & 3)));
        vt[s][h][dt] = __builtin_bit_cast(ev8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
      }
  }

#pragma unroll 1
  for (int group = 0; group < GROUPS; group++) {
#pragma unroll
    for (int j = 0; j < 4; j++) q[j] = g == hh ? q[j] : zero;
    floatx4 st[4];   // keys 16 t + 4 g + e
#pragma unroll
    for (int t = 0; t < 4; t++) {
      st[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 4; j++) st[t] = Mfma16(__builtin_bit_cast(ev8, k[t][j]), __builtin_bit_cast(ev8, q[j]), st[t]);
    }
    qp += 4 * (unsigned)(group + 1 < GROUPS ? ld : 0);
#pragma unroll
    for (int j = 0; j < 4; j++) q[j] = *reinterpret_cast<const intx4*>(qp + 8 * j);
    const LT* lp = logits + (head0 + hh) * kLogitStride + (4 * group + (r & 3)) * 64 + 4 * g;
    float mx = -3.0e38f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const lv4 l = *reinterpret_cast<const lv4*>(lp + 16 * t);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        st[t][e] = st[t][e] * p.scale + (float)l[e];
        mx = fmaxf(mx, st[t][e]);
      }
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
    for (int s = 0; s < 2; s++) {
      ev8 pf;   // keys 32 s + 4 g + e and 32 s + 16 + 4 g + e
#pragma unroll
      for (int e = 0; e < 8; e++) pf[e] = (ET)(st[2 * s + e / 4][e % 4] * inv);
#pragma unroll
      for (int h = 0; h < 4; h++) {
        const ev8 ph = __builtin_bit_cast(ev8, hh == h ? __builtin_bit_cast(intx4, pf) : zero);
#pragma unroll
        for (int dt = 0; dt < 2; dt++) o[dt] = Mfma16(vt[s][h][dt], ph, o[dt]);
      }
    }
    // depth 16 dt + 4 g + e of the column's query and head
    const long long at = ((long long)b * 64 + q0 + 4 * group + (r & 3)) * d_model + (head0 + hh) * 32 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < 2; dt++) {
      if constexpr (sizeof(OutT) == 1) {
        *reinterpret_cast<unsigned*>(static_cast<uint8_t*>(p.out) + at + 16 * dt) =
            PackFp8x4(o[dt][0] * p.out_mul, o[dt][1] * p.out_mul, o[dt][2] * p.out_mul, o[dt][3] * p.out_mul);
      } else {
        *reinterpret_cast<ev4*>(static_cast<ET*>(p.out) + at + 16 * dt) =
            ev4{(ET)o[dt][0], (ET)o[dt][1], (ET)o[dt][2], (ET)o[dt][3]};
      }
    }
  }
}

// Workgroups that share the heads of the same queries: K, V, gamma and beta are then spread over as many CUs, weights and the rows of the
// norm repeated. As many as leave half of the CUs free: us of a 15x1024 pass, one -> shared, 1 position by eight 820 -> 777, 2 by four 890
// -> 850, 4 by two 994 -> 971, e4m3 1 713 -> 671. By two at 8 positions, on every CU, a pass alone is faster too (1122 -> 1098), but four
// threads lose 10 % (15.7k -> 14.1k evals/s; 4 positions by two 9.1k -> 9.1k).
int HeadGroups(int workgroups, int heads) {
  int groups = 1;
  while (groups < 8 && 2 * groups * workgroups <= 128 && heads % (8 * groups) == 0) groups *= 2;
  return groups;
}

template <int QUERIES>
void LaunchFew(const SmolgenFewArgs& args, hipStream_t stream) {
  SmolgenFewArgs a = args;
  constexpr int PER = 64 / QUERIES;
  a.head_groups = HeadGroups(a.batch * PER, a.heads);
  const dim3 grid((a.batch >= 8 ? (a.batch + 7) / 8 * 8 * PER : a.batch * PER) * a.head_groups), block(512);
  if (a.out_f8) hipLaunchKernelGGL((smolgen_attention_few_kernel<half_t, uint8_t, QUERIES>), grid, block, 0, stream, a);
  else if (a.bf16) hipLaunchKernelGGL((smolgen_attention_few_kernel<bf16_t, half_t, QUERIES>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((smolgen_attention_few_kernel<half_t, half_t, QUERIES>), grid, block, 0, stream, a);
}
}  // namespace

bool SmolgenAttentionFewSupported(int heads, int depth, int gen_sz) {
  return depth == 32 && heads >= 4 && heads <= 32 && heads % 4 == 0 && gen_sz == kGen;
}

void LaunchSmolgenAttentionFew(const SmolgenFewArgs& a, hipStream_t stream) {
  if (a.batch <= 0) return;
  if (!SmolgenAttentionFewSupported(a.heads, 32, kGen) || (a.out_f8 && a.bf16)) {
    throw std::runtime_error("LaunchSmolgenAttentionFew: unsupported shape");
  }
  // As few queries per workgroup as leave one workgroup for every CU.
  if (a.batch <= 16) LaunchFew<4>(a, stream);
  else if (a.batch <= 32) LaunchFew<8>(a, stream);
  else LaunchFew<16>(a, stream);
}

}  // namespace lc0mi
