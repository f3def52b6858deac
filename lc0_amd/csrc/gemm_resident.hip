// Batched matrix products whose weights fit the LDS (the winograd-domain products of a 256-wide residual tower).
#include "gemm_variants.h"
#include "kernel_common.h"
#include "row_panel.h"

namespace lc0mi {

namespace {

// ---------------------------------------------------------------------------
// C_z = scale * A_z . W_z^T with K = 256 and 256 columns, 16-bit operands: one workgroup of eight waves per CU stays
// with one product z, keeps its whole 256 x 256 weight matrix (128 KiB) in LDS and walks over row blocks of 128, while
// tiles of such short products spend most of their time on their first operands and their epilogue.
//
// A wave owns 32 rows x 128 columns (2 x 8 accumulator tiles of v_mfma_f32_16x16x32): its rows come straight from global
// memory (row_panel.h), all 256 values of them, and the next block's are on their way while this one's are multiplied.
// The weights come in by direct transfers of 64 bytes per four lanes and are read without bank conflicts; a CU needs
// 8 x 64 KiB of them per block (4096 cycles) and as many cycles of its matrix cores. Output rows go through 4 KiB of LDS per wave and leave as 256-byte pieces.
// What bounds it: about 9 us of launch, weights and first rows before the first output, then memory: 36 products of 4096
// rows move 156 MB in 32.2 us (37.3 on 128x64 tiles), of 2048 rows 80 MB in 21.8 (23.5 to 25.9), of 768 rows 10.6 (12.9).
// Consecutive workgroups run on the same XCD, so that its L2 serves the weights of a product to all of them, or to all of
// them on two XCDs where the share of an XCD (31 or 32 of 252 workgroups) ends within a product's seven.
// ---------------------------------------------------------------------------
constexpr int kResRows = 128, kResCols = 256, kResK = 256;

template <typename ET>
__global__ __launch_bounds__(512) void gemm_resident_kernel(GemmArgs p, int per_product) {
  using ev8 = typename Vec16<ET>::v8;
  __shared__ __attribute__((aligned(1024))) char wlds[kResCols * kResK * 2];
  __shared__ __attribute__((aligned(16))) char strips[8][16 * 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r = lane & 15, g = lane >> 4;
  // Workgroup i runs on XCD i % 8: consecutive ranks on the same one.
  const int total = gridDim.x, xcd = blockIdx.x & 7;
  const int rank = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  const int z = rank / per_product, part = rank - z * per_product;
  const ET* A = reinterpret_cast<const ET*>(p.A) + (long long)z * p.strideA;
  ET* C = reinterpret_cast<ET*>(p.C) + (long long)z * p.strideC;
  // Transfer f = (16 weight rows c, step s of 128 values, i): lane 16 g + 4 q + x brings row 16 c + 4 q + i, byte
  // 256 s + 64 g + 16 (x ^ i). Four neighbouring lanes read 64 bytes of a row, and quarter j of row r lies at slot
  // 16 g + 4 (r / 4) + (j ^ r % 4) of transfer r % 4, so the 16 rows of a fragment read lie in different banks.
  const char* W = reinterpret_cast<const char*>(p.W) + 2 * (long long)z * p.strideW;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int f = wave * 16 + i, c = f >> 3, s = (f >> 2) & 1, k = f & 3;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(W + (long long)(16 * c + 4 * (r >> 2) + k) * p.ldw * 2 + 256 * s +
                                                         64 * g + 16 * ((r & 3) ^ k)),
        (__attribute__((address_space(3))) void*)(wlds + f * 1024), 16, 0, 0);
  }
  int w_slot[4];
#pragma unroll
  for (int j = 0; j < 4; j++) w_slot[j] = (r & 3) * 1024 + (16 * g + 4 * (r >> 2) + (j ^ (r & 3))) * 16;
  const int M = p.M, blocks = (M + kResRows - 1) / kResRows;
  auto load = [&](int block, intx4 (&a)[2][2][4]) {
    const int m0 = min(block * kResRows + 32 * wm, M - 1);   // (a wave without rows reads the last one and stores nothing)
    const char* base = reinterpret_cast<const char*>(A + (long long)m0 * p.lda);
    TileOffsets off[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      off[t].Set(16 * t, M - m0, 2 * p.lda);
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) a[t][s][i] = *reinterpret_cast<const intx4*>(base + s * kStepBytes + off[t].off[i]);
    }
  };
  auto block_products = [&](int block, intx4 (&a)[2][2][4]) {
    floatx4 acc[2][8];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int c = 0; c < 8; c++) acc[t][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 2; s++) {
      QuadTranspose(a[0][s]);
      QuadTranspose(a[1][s]);
#pragma unroll
      for (int c = 0; c < 8; c++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const ev8 w = *reinterpret_cast<const ev8*>(wlds + ((8 * wn + c) * 2 + s) * 4096 + w_slot[j]);
          acc[0][c] = Mfma16(w, __builtin_bit_cast(ev8, a[0][s][j]), acc[0][c]);
          acc[1][c] = Mfma16(w, __builtin_bit_cast(ev8, a[1][s][j]), acc[1][c]);
        }
    }
    // Accumulator lane (r, g) of tile (t, c): row 16 t + r, columns 16 c + 4 g + e. 16-byte chunk q of strip row x lies
    // at slot q ^ x.
    char* strip = strips[wave];
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
      for (int c = 0; c < 8; c++) {
        using ov4 = typename Vec16<ET>::v4;
        ov4 h;
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = (ET)(acc[t][c][e] * p.scale);
        *reinterpret_cast<ov4*>(strip + r * 256 + ((2 * c + (g >> 1)) ^ r) * 16 + (g & 1) * 8) = h;
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); the strip is private to this wave
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int x = 4 * i + (lane >> 4), q = lane & 15;
        const int m = block * kResRows + 32 * wm + 16 * t + x;
        const intx4 v = *reinterpret_cast<const intx4*>(strip + x * 256 + (q ^ x) * 16);
        if (m < M) *reinterpret_cast<intx4*>(C + (long long)m * p.ldc + 128 * wn + 8 * q) = v;
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
    }
  };
  intx4 a0[2][2][4], a1[2][2][4];
  int block = part;                      // (part < per_product <= blocks)
  load(block, a0);
  __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0): the weights
  __syncthreads();
  for (;;) {
    // (the last block is loaded once more instead of nothing: no condition around the loads)
    load(min(block + per_product, blocks - 1), a1);
    block_products(block, a0);
    block += per_product;
    if (block >= blocks) break;
    load(min(block + per_product, blocks - 1), a0);
    block_products(block, a1);
    block += per_product;
    if (block >= blocks) break;
  }
}
}  // namespace

void LaunchGemmResident(const GemmArgs& a, hipStream_t stream) {
  const int per_product = GemmResidentWorkgroups(a);
  auto launch = [&](auto elem_tag) {
    hipLaunchKernelGGL((gemm_resident_kernel<decltype(elem_tag)>), dim3(per_product * a.batch), dim3(512), 0, stream, a,
                       per_product);
  };
  if (a.bf16) launch(bf16_t{});
  else launch(half_t{});
}

}  // namespace lc0mi
