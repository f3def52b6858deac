// Operand fragments of 16-row matrix-instruction tiles taken straight from global memory (device code shared by the
// row-panel products of every element type).
#pragma once

#include "kernel_common.h"

namespace lc0mi {
namespace {

// A 16-row tile of a row-major operand is read 256 bytes of every row at a time (a "step"), as four loads of 16 bytes
// per lane. A matrix instruction wants lane (r = lane % 16, g = lane / 16) to hold a 16-byte chunk of row r; loads in
// that order touch four rows with every four neighbouring lanes, and the address path, which takes one 64-byte segment
// from each group of four lanes per cycle, delivers 16 bytes per cycle and CU (measured: 64 rows x 8 KiB by one
// workgroup on every CU, 31 k cycles). Here four neighbouring lanes read 64 consecutive bytes of one row (10.5 k cycles,
// 50 bytes per cycle) and a 4 x 4 transpose between the four loads and the four lanes (data-parallel-primitive moves,
// no LDS) puts the chunks where the instruction wants them: load i brings rows 4 q + i (q = lane / 4 % 4), byte
// 64 g + 16 (lane % 4); afterwards register j of lane (r, g) holds row r, byte 64 g + 16 j. Which bytes of a step meet
// in one instruction does not matter as long as both operands use the same order.
constexpr int kStepBytes = 256;

// v[i] of lane 4 n + j <-> v[j] of lane 4 n + i, for every four neighbouring lanes. Two butterfly stages; a stage is one
// instruction per register, a selection whose first source comes from the partner lane: lanes in the mask keep their
// own value. (Written out because the compiler makes a move and a selection of each. The no-ops are the two wait states
// between a vector write and a lane move that reads it.)
__device__ __forceinline__ void QuadTranspose(intx4 (&v)[4]) {
#define LC0MI_SEL(dst, partner, own, perm) \
  "v_cndmask_b32_dpp %" #dst ", %" #partner ", %" #own ", vcc quad_perm:[" perm "] row_mask:0xf bank_mask:0xf\n\t"
#pragma unroll
  for (int d = 0; d < 4; d += 2) {
    int a[2], b[2], c[2], e[2];
    asm("s_nop 1\n\ts_mov_b32 vcc_lo, 0x55555555\n\ts_mov_b32 vcc_hi, 0x55555555\n\t"   // even lanes keep v0, v2
        LC0MI_SEL(0, 9, 8, "1,0,3,2") LC0MI_SEL(2, 11, 10, "1,0,3,2")
        LC0MI_SEL(4, 13, 12, "1,0,3,2") LC0MI_SEL(6, 15, 14, "1,0,3,2")
        "s_not_b64 vcc, vcc\n\t"                                                         // odd lanes keep v1, v3
        LC0MI_SEL(1, 8, 9, "1,0,3,2") LC0MI_SEL(3, 10, 11, "1,0,3,2")
        LC0MI_SEL(5, 12, 13, "1,0,3,2") LC0MI_SEL(7, 14, 15, "1,0,3,2")
        : "=&v"(a[0]), "=&v"(b[0]), "=&v"(c[0]), "=&v"(e[0]), "=&v"(a[1]), "=&v"(b[1]), "=&v"(c[1]), "=&v"(e[1])
        : "v"(v[0][d]), "v"(v[1][d]), "v"(v[2][d]), "v"(v[3][d]), "v"(v[0][d + 1]), "v"(v[1][d + 1]), "v"(v[2][d + 1]),
          "v"(v[3][d + 1])
        : "vcc", "scc");
    int a2[2], b2[2], c2[2], e2[2];
    asm("s_nop 1\n\ts_mov_b32 vcc_lo, 0x33333333\n\ts_mov_b32 vcc_hi, 0x33333333\n\t"   // lanes 0, 1 keep v0, v1
        LC0MI_SEL(0, 10, 8, "2,3,0,1") LC0MI_SEL(1, 11, 9, "2,3,0,1")
        LC0MI_SEL(4, 14, 12, "2,3,0,1") LC0MI_SEL(5, 15, 13, "2,3,0,1")
        "s_not_b64 vcc, vcc\n\t"                                                         // lanes 2, 3 keep v2, v3
        LC0MI_SEL(2, 8, 10, "2,3,0,1") LC0MI_SEL(3, 9, 11, "2,3,0,1")
        LC0MI_SEL(6, 12, 14, "2,3,0,1") LC0MI_SEL(7, 13, 15, "2,3,0,1")
        : "=&v"(a2[0]), "=&v"(b2[0]), "=&v"(c2[0]), "=&v"(e2[0]), "=&v"(a2[1]), "=&v"(b2[1]), "=&v"(c2[1]), "=&v"(e2[1])
        : "v"(a[0]), "v"(b[0]), "v"(c[0]), "v"(e[0]), "v"(a[1]), "v"(b[1]), "v"(c[1]), "v"(e[1])
        : "vcc", "scc");
#pragma unroll
    for (int q = 0; q < 2; q++) {
      v[0][d + q] = a2[q]; v[1][d + q] = b2[q]; v[2][d + q] = c2[q]; v[3][d + q] = e2[q];
    }
  }
#undef LC0MI_SEL
}

// This lane's four load addresses of one tile: byte offsets from the first of `rows` rows (the workgroup's first row to
// the operand's last, so that 32 bits do), rows past the last one clamped.
struct TileOffsets {
  unsigned off[4];
  __device__ __forceinline__ void Set(int row0, int rows, int row_bytes) {
    const int lane = threadIdx.x & 63;
    const int in_row = 64 * (lane >> 4) + 16 * (lane & 3);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = min(row0 + 4 * ((lane >> 2) & 3) + i, rows - 1);
      off[i] = (unsigned)(row * row_bytes + in_row);
    }
  }
};

// One step (four 16-byte chunks of both operands) of a 16x16 accumulator tile, by operand type.
template <typename ET> struct PanelOp {   // half_t, bf16_t: 128 values, v_mfma_f32_16x16x32
  __device__ __forceinline__ void operator()(const intx4 (&w)[4], const intx4 (&a)[4], floatx4& c) const {
    using ev8 = typename Vec16<ET>::v8;
#pragma unroll
    for (int j = 0; j < 4; j++) c = Mfma16(__builtin_bit_cast(ev8, w[j]), __builtin_bit_cast(ev8, a[j]), c);
  }
};
template <> struct PanelOp<uint8_t> {     // e4m3: 256 values, v_mfma_f32_16x16x128_f8f6f4
  __device__ __forceinline__ void operator()(const intx4 (&w)[4], const intx4 (&a)[4], floatx4& c) const {
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const intx8 fw = {w[j][0], w[j][1], w[j][2], w[j][3], w[j + 1][0], w[j + 1][1], w[j + 1][2], w[j + 1][3]};
      const intx8 fa = {a[j][0], a[j][1], a[j][2], a[j][3], a[j + 1][0], a[j + 1][1], a[j + 1][2], a[j + 1][3]};
      c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fw, fa, c, 0, 0, 0, 0, 0, 0);
    }
  }
};

// The products of a wave that has one step only, with one set of operand registers. `bytes` of every row exist (a multiple
// of 16, at least 16), masked as PanelProducts masks its last step. (A function of its own: the same code called from there
// made its loops 3 % slower, 33x3072x256 in halves 3.38 us against 3.25.)
template <int TA, int TW, typename Acc, typename Op>
__device__ __forceinline__ void OneStep(const char* pa, const TileOffsets (&ta)[TA], const char* pw,
                                        const TileOffsets (&tw)[TW], int bytes, Acc (&acc)[TA][TW], Op op) {
  const int lane = threadIdx.x & 63, in_row = 64 * (lane >> 4) + 16 * (lane & 3);
  const bool in = in_row < bytes;
  const unsigned back = in ? 0u : (unsigned)in_row;
  intx4 a[TA][4], w[TW][4];
#pragma unroll
  for (int c = 0; c < TW; c++)
#pragma unroll
    for (int i = 0; i < 4; i++) w[c][i] = *reinterpret_cast<const intx4*>(pw + (tw[c].off[i] - back));
#pragma unroll
  for (int t = 0; t < TA; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) a[t][i] = *reinterpret_cast<const intx4*>(pa + (ta[t].off[i] - back));
  if (bytes < kStepBytes) {
    const intx4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int c = 0; c < TW; c++) w[c][i] = in ? w[c][i] : zero;
#pragma unroll
      for (int t = 0; t < TA; t++) a[t][i] = in ? a[t][i] : zero;
    }
  }
#pragma unroll
  for (int c = 0; c < TW; c++) QuadTranspose(w[c]);
#pragma unroll
  for (int t = 0; t < TA; t++) {
    QuadTranspose(a[t]);
#pragma unroll
    for (int c = 0; c < TW; c++) op(w[c], a[t], acc[t][c]);
  }
}

// Sum over this wave's steps [begin, end) of the products of TA activation tiles with TW weight tiles: op(w, a, acc)
// multiplies one step (four chunks of either operand). A step beyond whole_bytes of the rows is read up to there only.
template <int TA, int TW, typename Acc, typename Op>
__device__ __forceinline__ void PanelProducts(const char* a_base, const TileOffsets (&ta)[TA], const char* w_base,
                                              const TileOffsets (&tw)[TW], int row_bytes, int begin, int end,
                                              Acc (&acc)[TA][TW], Op op) {
  const int whole = row_bytes / kStepBytes;
  auto load = [&](int step, intx4 (&a)[TA][4], intx4 (&w)[TW][4]) {
    const char* pa = a_base + step * kStepBytes;
    const char* pw = w_base + step * kStepBytes;
#pragma unroll
    for (int c = 0; c < TW; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) w[c][i] = *reinterpret_cast<const intx4*>(pw + tw[c].off[i]);
#pragma unroll
    for (int t = 0; t < TA; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) a[t][i] = *reinterpret_cast<const intx4*>(pa + ta[t].off[i]);
  };
  auto multiply = [&](intx4 (&a)[TA][4], intx4 (&w)[TW][4]) {
#pragma unroll
    for (int c = 0; c < TW; c++) QuadTranspose(w[c]);
#pragma unroll
    for (int t = 0; t < TA; t++) {
      QuadTranspose(a[t]);
#pragma unroll
      for (int c = 0; c < TW; c++) op(w[c], a[t], acc[t][c]);
    }
  };
  const int last = min(end, whole);
  intx4 a0[TA][4], w0[TW][4];
  if (begin < last) {
    // (no condition around a load of the loop: behind a branch the compiler waits for every load in flight)
    load(begin, a0, w0);
    intx4 a1[TA][4], w1[TW][4];
    int st = begin;
    for (; st + 2 < last; st += 2) {
      load(st + 1, a1, w1);
      multiply(a0, w0);
      load(st + 2, a0, w0);
      multiply(a1, w1);
    }
    if (st + 1 < last) {
      load(st + 1, a1, w1);
      multiply(a0, w0);
      multiply(a1, w1);
    } else {
      multiply(a0, w0);
    }
  }
  if (begin < end && end > whole) {
    // A lane without bytes in this step reads the step's first ones of its rows and takes zeros instead: no condition
    // around a load here either (with one, a rest of 8 halves made 256x256x264 2.83 us instead of 2.72).
    const int lane = threadIdx.x & 63, in_row = 64 * (lane >> 4) + 16 * (lane & 3);
    const bool in = in_row < row_bytes - whole * kStepBytes;
    const char* pa = a_base + whole * kStepBytes;
    const char* pw = w_base + whole * kStepBytes;
    const unsigned back = in ? 0u : (unsigned)in_row;
#pragma unroll
    for (int c = 0; c < TW; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) w0[c][i] = *reinterpret_cast<const intx4*>(pw + (tw[c].off[i] - back));
#pragma unroll
    for (int t = 0; t < TA; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) a0[t][i] = *reinterpret_cast<const intx4*>(pa + (ta[t].off[i] - back));
    const intx4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int c = 0; c < TW; c++) w0[c][i] = in ? w0[c][i] : zero;
#pragma unroll
      for (int t = 0; t < TA; t++) a0[t][i] = in ? a0[t][i] : zero;
    }
    multiply(a0, w0);
  }
}

}  // namespace
}  // namespace lc0mi
