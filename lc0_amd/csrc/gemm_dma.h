// Direct-to-LDS matrix product (device code), included by the sources that instantiate it per operand type.
#pragma once

#include "kernel_common.h"
#include "gemm_variants.h"

#include <stdexcept>
#include <type_traits>

namespace lc0mi {

namespace {
// ---------------------------------------------------------------------------
// Large-shape GEMM: same contract as gemm_kernel for K % BK == 0 and half output.
//
// Operand tiles travel from global memory straight into LDS (16 bytes per lane,
// global_load_lds_dwordx4), double-buffered, with one barrier per k-tile: the
// fetch of k-tile t+1 is in flight while the MFMAs of k-tile t run, and no VGPR
// is spent on staging. One such instruction fills 1 KiB of LDS in lane order, so
// LDS rows are unpadded; the 16-byte chunk c of tile row r is stored at chunk
// slot c ^ swizzle(r), which makes the ds_read_b128 fragment reads (32 rows x
// one chunk column) hit all banks evenly. The epilogue applies scale, bias and
// activation in registers, stages 32-row strips through LDS and writes rows of
// the output as 16-byte vectors.
// ---------------------------------------------------------------------------
#define LC0MI_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

// 16 bytes per lane from global memory into LDS at lds_base + lane * 16
// (lds_base must be wave-uniform). Completion is visible through vmcnt only:
// callers wait with s_waitcnt vmcnt(0) plus a barrier before reading the data.
// Two forms: inline assembly, which the compiler schedules nothing across, and the compiler's builtin, which sets M0
// itself and may be moved among the MFMAs and fragment reads of a k-tile (better for the 256-row tiles: +0.5 % of a
// pass at batch 256; worse for the small tiles: -1 % at batch 16).
template <bool BUILTIN>
__device__ __forceinline__ void DmaToLds16(const void* gptr, void* lds_base) {
  if constexpr (BUILTIN) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)gptr, LC0MI_LDS_PTR(lds_base), 16,
                                     0, 0);
  } else {
    // (the no-op is the wait state that the hardware needs between a scalar write of M0 and a load into LDS, which takes
    // its LDS address from it; the compiler adds it for its builtin and does not look into this)
    unsigned lds_addr = (unsigned)(size_t)LC0MI_LDS_PTR(lds_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_addr), "v"(gptr) : "memory", "m0");
  }
}

template <int STORES>
__device__ __forceinline__ void StoreOut16(void* dst, intx4 val) {
  if constexpr (STORES == 1) {
    __builtin_nontemporal_store(val, reinterpret_cast<intx4*>(dst));
  } else if constexpr (STORES == 2) {
    StoreThrough16(dst, val);
  } else {
    *reinterpret_cast<intx4*>(dst) = val;
  }
}

// The same kernel serves fp16 operands (Args = GemmArgs: BKB = 128 bytes = 64
// halves per tile row, v_mfma_f32_32x32x16_f16) and e4m3 operands (Args =
// GemmF8Args: 128 bytes = 128 values per row, v_mfma_f32_32x32x64_f8f6f4);
// BKB is the k-tile in bytes. OutT is half_t or uint8_t (e4m3, fp8 operands only).
// STORES: how the 16-byte output vectors are stored: 0 ordinary stores (the output stays in L2 and the memory-side
// cache), 1 streaming (non-temporal) stores, 2 stores written through at device scope (they leave L2 alone like the
// streaming ones, but what they wrote is found faster by the next kernel; plain epilogue only).
// EPI (fp16 operands only): 0 the plain epilogue, 1 the consumer and 2 the producer side of a folded layer norm
// (GemmArgs::row_stats / GemmArgs::skip).
// NSTAGES k-tiles of LDS: NSTAGES - 1 of them are in flight while one is consumed. Two stages suffice when the
// operands come from L2; with small tiles and operands that come from memory (a few hundred to a few thousand rows:
// every workgroup streams weights nobody has touched since the previous pass) a k-tile takes longer to arrive than
// to consume, and more stages hide that.
// ET (fp16-type operands only): half_t or bf16_t; the output type is then ET as well.
// ALONE: for a workgroup that has its CU to itself: the barrier of a k-tile stands before its last products.
//
// The small tiles are bound inside a workgroup, not by bandwidth: a wave stands still while the address path takes its
// transfers (14.5 cycles each, 32 per k-tile of a 128x128 tile, about as long as the products take), and after every
// barrier nothing runs until the first fragments are there. So the transfers go out one by one between the products
// (sched_barrier pins the order; inline assembly is not seen by the scheduling groups), and with ALONE the barrier and
// the first fragments of the next k-tile come before the last products of this one. us, transfers first -> spread ->
// with ALONE: 512x1024x1024 on 64x64 tiles 6.8 -> 6.2 -> 5.6, 512x1024x1536 8.9 -> 7.9 -> 6.9, on 128x64 tiles
// 512x3072x1024 9.5 -> 8.1 -> 7.7; 4096x1024x1024 on 128x128 13.9 -> 12.6, 4096x1024x1536 19.2 -> 17.2. Workgroups that
// share a CU fill each other's gaps and lose with ALONE (832x1536x1024 on 312 tiles of 64x64: 9.4 -> 11.1), and so do
// 128x128 tiles (1024x3072x1024 12.5 -> 14.4). With two stages a transfer sent later has too little time to arrive
// (3072x3072x1024 on 128x128 30.5 -> 32.5; 77 positions of the 15x1024 net 2830 -> 2874 a pass), and the 256-row tiles
// lose 2 to 5 % (16384x1024x1024 35.4 -> 36.7): both keep the transfers at the head of the k-tile.
template <int BM, int BN, int BKB, int WAVES_M, int WAVES_N, typename Args, typename OutT, int STORES = 0,
          int EPI = 0, int NSTAGES = 2, typename ET = half_t, bool ALONE = false, bool TWO = false>
// Second launch bound = waves per SIMD: with small wave tiles two workgroups share a CU
// (4 waves per SIMD, at most 128 VGPRs) and overlap each other's prologue and epilogue.
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64,
                             ((BM / WAVES_M / 32) * (BN / WAVES_N / 32) <= 4 && 2 * NSTAGES * (BM + BN) * BKB <= 160 * 1024)
                                 ? WAVES_M * WAVES_N / 2
                                 : WAVES_M * WAVES_N / 4)
void gemm_dma_kernel(Args p) {
  constexpr bool F8 = std::is_same<Args, GemmF8Args>::value;
  constexpr int ES = F8 ? 1 : 2;                  // bytes per operand element
  constexpr int NWAVES = WAVES_M * WAVES_N;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int CPR = BKB / 16;                   // 16-byte chunks per tile row
  constexpr int ROWS_PER_CHUNK = 64 / CPR;        // tile rows per 1 KiB transfer
  constexpr int SWZ_SHIFT = (BKB == 128) ? 1 : 2; // log2(rows per 256 bytes of LDS)
  constexpr int A_CPW = BM / ROWS_PER_CHUNK / NWAVES, W_CPW = BN / ROWS_PER_CHUNK / NWAVES;
  static_assert(BKB == 128 || BKB == 64, "k-tile must be 64 or 128 bytes");
  static_assert(F8 || sizeof(OutT) == 2, "fp8 output needs fp8 operands");
  static_assert(A_CPW >= 1 && W_CPW >= 1, "tile too small for the wave count");
  constexpr int STAGE = (BM + BN) * BKB;          // bytes
  constexpr int OV = 16 / sizeof(OutT);           // output elements per 16-byte vector
  constexpr int EPI_STRIDE = WN + OV;             // elements
  constexpr int EPI_BYTES = NWAVES * 32 * EPI_STRIDE * (int)sizeof(OutT);
  // Folded layer norm: (mean, rstd) of the tile's rows, and the producer's per-wave-column partial sums.
  constexpr int STAT_BYTES = (EPI != 0) ? BM * 8 : 0;
  constexpr int PART_BYTES = (EPI == 2) ? WAVES_N * BM * 8 : 0;
  constexpr int EPI_TOTAL = EPI_BYTES + STAT_BYTES + PART_BYTES;
  constexpr int SMEM = (NSTAGES * STAGE > EPI_TOTAL) ? NSTAGES * STAGE : EPI_TOTAL;
  static_assert(BKB >= (F8 ? 128 : 64), "at least two k-steps in a k-tile");
  static_assert(NSTAGES >= 2 && (NSTAGES - 2) * (A_CPW + W_CPW) <= 63, "transfers in flight must fit the counter");
  static_assert(EPI == 0 || (!F8 && std::is_same<OutT, half_t>::value && std::is_same<ET, half_t>::value),
                "folded layer norm: fp16 operands and output");
  static_assert(std::is_same<ET, half_t>::value || (!F8 && std::is_same<OutT, ET>::value),
                "bfloat16 operands go with bfloat16 output");
  // The tile's bias (and per-column scale, fp8 operands) waits in LDS behind the stages: fetched with the first k-tile,
  // so that the epilogue does not start with a round trip to memory.
  constexpr int COLV_BYTES = (F8 ? 2 : 1) * BN * 4;
  __shared__ __attribute__((aligned(1024))) char smem[SMEM + COLV_BYTES];
  float* colv = reinterpret_cast<float*>(smem + SMEM);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  // With TWO tiles past the columns of the first product belong to a second one. (An instance of its own: the choice costs launches
  // that have no second product, e4m3 19200x32x1024 on 128x64 tiles 11.5 us instead of 10.85, 300x8192x256 on 64x64 8.75 instead of 8.45.)
  static_assert(!TWO || (BM < 256 && EPI == 0 && sizeof(OutT) == 2), "small tiles, 16-bit output");
  const int col_tiles = TWO ? (p.N + BN - 1) / BN : 0;
  const int2 tile = TileOfWorkgroup(p.tile_order);
  const bool second = TWO && tile.y >= col_tiles;
  const int m0 = tile.x * BM, n0 = (second ? tile.y - col_tiles : tile.y) * BN;
  const int M = p.M, N = second ? p.N2 : p.N, K = p.K, ldw = second ? p.ldw2 : p.ldw;
  float my_bias = 0.0f;
  [[maybe_unused]] float my_cscale = 0.0f;
  if (tid < BN && n0 + tid < N) {
    if (p.bias != nullptr && !second) my_bias = p.bias[n0 + tid];
    if constexpr (F8) my_cscale = (second ? p.col_scale2 : p.col_scale)[n0 + tid];
  }
  const char* A = reinterpret_cast<const char*>(p.A);
  const char* W = second ? reinterpret_cast<const char*>(p.W2) : reinterpret_cast<const char*>(p.W);
  if constexpr (!F8) {
    A += (long long)blockIdx.z * p.strideA * ES;
    W += (long long)blockIdx.z * p.strideW * ES;
  }

  const char* a_ptr[A_CPW];
  const char* w_ptr[W_CPW];
#pragma unroll
  for (int i = 0; i < A_CPW; i++) {
    const int row = (wave * A_CPW + i) * ROWS_PER_CHUNK + lane / CPR;
    const int c = (lane % CPR) ^ ((row >> SWZ_SHIFT) % CPR);
    a_ptr[i] = A + (long long)min(m0 + row, M - 1) * p.lda * ES + c * 16;
  }
#pragma unroll
  for (int i = 0; i < W_CPW; i++) {
    const int row = (wave * W_CPW + i) * ROWS_PER_CHUNK + lane / CPR;
    const int c = (lane % CPR) ^ ((row >> SWZ_SHIFT) % CPR);
    w_ptr[i] = W + (long long)min(n0 + row, N - 1) * ldw * ES + c * 16;
  }
  auto issue = [&](char* As, char* Ws, int kbyte) {
#pragma unroll
    for (int i = 0; i < A_CPW; i++) DmaToLds16<BM == 256>(a_ptr[i] + kbyte, As + (wave * A_CPW + i) * 1024);
#pragma unroll
    for (int i = 0; i < W_CPW; i++) DmaToLds16<BM == 256>(w_ptr[i] + kbyte, Ws + (wave * W_CPW + i) * 1024);
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  const int r = lane & 31, g = lane >> 5;
  const int swz = (r >> SWZ_SHIFT) % CPR;
  const int a_row = (wm * WM + r) * BKB, w_row = (wn * WN + r) * BKB;

  const int nk = K * ES / BKB;
  issue(smem, smem + BM * BKB, 0);
#pragma unroll
  for (int st = 1; st < NSTAGES - 1; st++) {
    if (st < nk) issue(smem + st * STAGE, smem + st * STAGE + BM * BKB, st * BKB);
  }
  if (tid < BN) {
    colv[tid] = my_bias;
    if constexpr (F8) colv[BN + tid] = my_cscale;
  }
  // Folded layer norm: (mean, rstd) of tile row `tid` (of the A operand for a consumer, of the residual for a
  // producer), fetched while the first k-tile is on its way and kept in two registers until the epilogue.
  [[maybe_unused]] float2 my_ms = make_float2(0.0f, 1.0f);
  [[maybe_unused]] bool norm_skip = false;
  if constexpr (EPI != 0) {
    const float* st = (EPI == 1) ? p.row_stats : p.skip_stats;
    norm_skip = st != nullptr;
    if (st != nullptr && tid < BM) {
      RowMeanRstd(st, (EPI == 1) ? p.row_parts : p.skip_parts, min(m0 + tid, M - 1), p.norm_n, p.norm_eps, my_ms.x,
                  my_ms.y);
    }
  }
  // Producer: the residual tile is touched early (one dword per 128-byte line, values unused), so that the
  // epilogue finds it in cache instead of reading memory in the same burst in which every workgroup writes.
  [[maybe_unused]] int touch[(BM * BN * 2 / 128 + NWAVES * 64 - 1) / (NWAVES * 64)] = {};
  // One k-step of a k-tile: the fragments of this wave's rows, and their products.
  using Frag = std::conditional_t<F8, intx8, typename Vec16<std::conditional_t<F8, half_t, ET>>::v8>;
  constexpr int STEPS = BKB / (F8 ? 64 : 32);
  auto load_frags = [&](const char* As, const char* Ws, int ks, Frag (&af)[TM], Frag (&wf)[TN]) {
    if constexpr (F8) {
      // One MFMA consumes 64 k-values: lane half g holds 32 consecutive bytes = 2 chunks.
      const int c0 = ((4 * ks + 2 * g) ^ swz) * 16, c1 = ((4 * ks + 2 * g + 1) ^ swz) * 16;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const intx4 lo = *reinterpret_cast<const intx4*>(As + a_row + i * 32 * BKB + c0);
        const intx4 hi = *reinterpret_cast<const intx4*>(As + a_row + i * 32 * BKB + c1);
        af[i] = intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const intx4 lo = *reinterpret_cast<const intx4*>(Ws + w_row + j * 32 * BKB + c0);
        const intx4 hi = *reinterpret_cast<const intx4*>(Ws + w_row + j * 32 * BKB + c1);
        wf[j] = intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    } else {
      const int coff = ((2 * ks + g) ^ swz) * 16;
#pragma unroll
      for (int i = 0; i < TM; i++) af[i] = *reinterpret_cast<const Frag*>(As + a_row + i * 32 * BKB + coff);
#pragma unroll
      for (int j = 0; j < TN; j++) wf[j] = *reinterpret_cast<const Frag*>(Ws + w_row + j * 32 * BKB + coff);
    }
  };
  auto product = [&](const Frag& w, const Frag& a, floatx16& c) {
    if constexpr (F8) c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, 0, 0, 0, 0, 0, 0);
    else c = Mfma32(w, a, c);
  };
  // The 128- and 64-row tiles put the transfers of the k-tile fetched next between the products of this one (EARLY: all
  // before its last k-step).
  constexpr bool INTERLEAVE = BM < 256 && EPI == 0 && NSTAGES > 2;
  constexpr bool EARLY = INTERLEAVE && ALONE;
  static_assert(!ALONE || NSTAGES > 2, "the transfers of a k-tile need another k-tile's time to arrive");
  constexpr int IN_FLIGHT = (NSTAGES - 2) * (A_CPW + W_CPW);
  // This wave's pieces of k-tile kt have landed (the transfers of the NSTAGES - 2 k-tiles behind it may still be in
  // flight; near the end of K fewer are, and the wait is for all of them), and with the barrier everybody's have, and
  // everybody is done reading the stage that is filled next.
  auto arrive = [&](int kt) {
    if (NSTAGES > 2 && kt + NSTAGES - 2 < nk) {
      __builtin_amdgcn_s_waitcnt(0x0F70 | (IN_FLIGHT & 15) | ((IN_FLIGHT >> 4) << 14));
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    }
    __syncthreads();
  };
  [[maybe_unused]] Frag af[2][TM], wf[2][TN];
  auto stage = [&](int kt) { return smem + (NSTAGES == 2 ? (kt & 1) : kt % NSTAGES) * STAGE; };
  if constexpr (EARLY) {
    arrive(0);
    load_frags(smem, smem + BM * BKB, 0, af[0], wf[0]);
  }
  auto k_tile = [&](int kt, auto fetch_tag) {
    constexpr bool FETCH = decltype(fetch_tag)::value;   // there is a k-tile to fetch (k-tile kt + NSTAGES - 1)
    const char* As = stage(kt);
    const char* Ws = As + BM * BKB;
    char* nxt = stage(kt + NSTAGES - 1);
    if constexpr (!EARLY) arrive(kt);
    if constexpr (INTERLEAVE) {
      constexpr int MFMAS = (EARLY ? STEPS - 1 : STEPS) * TM * TN, PIECES = FETCH ? A_CPW + W_CPW : 0;
      if constexpr (!EARLY) load_frags(As, Ws, 0, af[0], wf[0]);
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) {
        if (ks + 1 < STEPS) {
          load_frags(As, Ws, ks + 1, af[(ks + 1) & 1], wf[(ks + 1) & 1]);
        } else if constexpr (EARLY) {
          if (kt + 1 < nk) {
            // Before the last products: the barrier and the first fragments of the next k-tile, whose latency they hide.
            arrive(kt + 1);
            const char* next = stage(kt + 1);
            load_frags(next, next + BM * BKB, 0, af[0], wf[0]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TM * TN; t++) {
          product(wf[ks & 1][t % TN], af[ks & 1][t / TN], acc[t / TN][t % TN]);
          const int at = ks * TM * TN + t;
          if (at >= MFMAS) continue;
#pragma unroll
          for (int q = at * PIECES / MFMAS; q < (at + 1) * PIECES / MFMAS; q++) {
            __builtin_amdgcn_sched_barrier(0);
            if (q < A_CPW) {
              DmaToLds16<false>(a_ptr[q < A_CPW ? q : 0] + (kt + NSTAGES - 1) * BKB, nxt + (wave * A_CPW + q) * 1024);
            } else {
              DmaToLds16<false>(w_ptr[q < A_CPW ? 0 : q - A_CPW] + (kt + NSTAGES - 1) * BKB,
                                nxt + BM * BKB + (wave * W_CPW + q - A_CPW) * 1024);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    } else {
      if constexpr (FETCH) issue(nxt, nxt + BM * BKB, (kt + NSTAGES - 1) * BKB);
      if constexpr (EPI == 2) {
        if (kt == 1) {
          constexpr int LINES_PER_ROW = (BN * 2 + 127) / 128;
          constexpr int LINES = BM * LINES_PER_ROW;
#pragma unroll
          for (int q = 0; q < (LINES + NWAVES * 64 - 1) / (NWAVES * 64); q++) {
            const int line = q * NWAVES * 64 + tid;
            const int row = line / LINES_PER_ROW, seg = line % LINES_PER_ROW;
            const half_t* src = p.skip + (long long)min(m0 + row, M - 1) * p.ldskip + min(n0 + seg * 64, N - 2);
            if (line < LINES) touch[q] = *reinterpret_cast<const volatile int*>(src);
          }
        }
      }
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) {
        load_frags(As, Ws, ks, af[0], wf[0]);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) product(wf[0][j], af[0][i], acc[i][j]);
      }
      if constexpr (!F8 && (BM / WAVES_M / 32) * (BN / WAVES_N / 32) >= (BM / WAVES_M / 32) + (BN / WAVES_N / 32) && EPI == 0) {
        // Order of the k-tile's 32 MFMAs and 24 fragment reads: the reads of a k-step one by one between the MFMAs
        // of the step before it.
        constexpr int KS = BKB / 32, RD = TM + TN, MF = TM * TN;
        __builtin_amdgcn_sched_group_barrier(0x100, RD, 0);
#pragma unroll
        for (int ks = 0; ks + 1 < KS; ks++) {
#pragma unroll
          for (int q = 0; q < RD; q++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, MF - RD, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
      }
    }
  };
  int kt = 0;
  for (; kt + NSTAGES - 1 < nk; kt++) k_tile(kt, std::true_type{});
  for (; kt < nk; kt++) k_tile(kt, std::false_type{});

  if constexpr (TWO) {
    if (second) {   // few columns: straight from the accumulators, four neighbouring columns of a row per lane
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int blk = 0; blk < 4; blk++) {
            const int m = m0 + wm * WM + i * 32 + r, col = wn * WN + j * 32 + blk * 8 + g * 4, n = n0 + col;
            if (m >= M || n >= N) continue;
            if constexpr (F8) {
              const floatx4 cs = *reinterpret_cast<const floatx4*>(colv + BN + col);
              float v[4];
#pragma unroll
              for (int rr = 0; rr < 4; rr++) v[rr] = acc[i][j][blk * 4 + rr] * cs[rr] * p.out_mul2;
              *reinterpret_cast<unsigned*>(reinterpret_cast<uint8_t*>(p.C2) + (long long)m * p.ldc2 + n) =
                  PackFp8x4(v[0], v[1], v[2], v[3]);
            } else {
              using ov4 = typename Vec16<ET>::v4;
              ov4 h;
#pragma unroll
              for (int rr = 0; rr < 4; rr++) h[rr] = (ET)acc[i][j][blk * 4 + rr];
              *reinterpret_cast<ov4*>(reinterpret_cast<ET*>(p.C2) + (long long)m * p.ldc2 + n) = h;
            }
          }
      return;
    }
  }
  // Epilogue through LDS (the stage buffers are free after the barrier).
  __syncthreads();
  if constexpr (EPI == 2) {
    // (the early touches are consumed here: every wait of the loop has covered them)
#pragma unroll
    for (int q = 0; q < (int)(sizeof(touch) / sizeof(touch[0])); q++) asm volatile("" ::"v"(touch[q]));
  }
  OutT* C = reinterpret_cast<OutT*>(p.C);
  if constexpr (!F8) C += (long long)blockIdx.z * p.strideC;
  OutT* strip = reinterpret_cast<OutT*>(smem) + wave * 32 * EPI_STRIDE;
  constexpr int CHUNKS_PER_ROW = WN / OV;
  constexpr int STRIP_CHUNKS = 32 * CHUNKS_PER_ROW;
  constexpr int NPASS = (STRIP_CHUNKS + 63) / 64;
  const bool vec_ok = (p.ldc % OV == 0);
  float bias_v[TN][4][4];
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int blk = 0; blk < 4; blk++) {
      const floatx4 b4 = *reinterpret_cast<const floatx4*>(colv + wn * WN + j * 32 + blk * 8 + g * 4);
#pragma unroll
      for (int rr = 0; rr < 4; rr++) bias_v[j][blk][rr] = b4[rr];
    }
  // Folded layer norm: statistics of this tile's rows (of the A operand for a consumer, of the residual for a
  // producer), one row per thread, shared through LDS.
  [[maybe_unused]] float2* row_ms = reinterpret_cast<float2*>(smem + EPI_BYTES);                 // [BM] (mean, rstd)
  [[maybe_unused]] float2* part_lds = reinterpret_cast<float2*>(smem + EPI_BYTES + STAT_BYTES);  // [WAVES_N][BM]
  [[maybe_unused]] float col_c[TN][4][4];
  auto load_skip = [&](int i, intx4 (&sk)[NPASS]) {
#pragma unroll
    for (int pass = 0; pass < NPASS; pass++) {
      const int idx = pass * 64 + lane;
      const int row = idx / CHUNKS_PER_ROW;
      const int ch = idx - row * CHUNKS_PER_ROW;
      const int m = m0 + wm * WM + i * 32 + row;
      const int n = n0 + wn * WN + ch * OV;
      if constexpr (EPI == 2) {
        sk[pass] = (idx < STRIP_CHUNKS && m < M && n + OV - 1 < N)
                       ? *reinterpret_cast<const intx4*>(p.skip + (long long)m * p.ldskip + n)
                       : intx4{0, 0, 0, 0};
      }
    }
  };
  // Producer: the residual chunks of a strip are fetched one strip ahead.
  [[maybe_unused]] intx4 sk_cur[NPASS], sk_nxt[NPASS];
  if constexpr (EPI == 2) load_skip(0, sk_cur);
  if constexpr (EPI != 0) {
    if (norm_skip) {
      if (tid < BM) row_ms[tid] = my_ms;
      __syncthreads();
    }
    if constexpr (EPI == 1) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int blk = 0; blk < 4; blk++) LoadBias4(p.col_c, n0 + wn * WN + j * 32 + blk * 8 + g * 4, N, col_c[j][blk]);
    }
  }
  // Producer: gamma and beta of the residual's layer norm for this lane's eight columns (the same in every pass).
  [[maybe_unused]] float sk_gamma[8], sk_beta[8];
  if constexpr (EPI == 2) {
    static_assert(64 % CHUNKS_PER_ROW == 0, "a lane must keep its columns over the passes of a strip");
    const int n = n0 + wn * WN + (lane % CHUNKS_PER_ROW) * OV;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      sk_gamma[e] = (norm_skip && n + e < N) ? p.skip_gamma[n + e] : 1.0f;
      sk_beta[e] = (norm_skip && n + e < N) ? p.skip_beta[n + e] : 0.0f;
    }
  }
  DispatchAct(p.act, [&](auto act_fn) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      // Consumer: v = rstd * (scale * acc - mean * c) + bias = acc * (rstd * scale) + (bias - (rstd * mean) * c)
      [[maybe_unused]] float rs_scale = 1.0f, rs_mean = 0.0f;
      if constexpr (EPI == 1) {
        const float2 ms = row_ms[wm * WM + i * 32 + r];
        rs_scale = ms.y * p.scale;
        rs_mean = -ms.y * ms.x;
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
          float v[4];
          if constexpr (F8) {
            // Per-column dequantisation factor (activation scale x weight-row scale).
            float cs[4];
            const floatx4 c4 = *reinterpret_cast<const floatx4*>(colv + BN + wn * WN + j * 32 + blk * 8 + g * 4);
#pragma unroll
            for (int rr = 0; rr < 4; rr++) cs[rr] = c4[rr];
#pragma unroll
            for (int rr = 0; rr < 4; rr++) v[rr] = act_fn(acc[i][j][blk * 4 + rr] * cs[rr] + bias_v[j][blk][rr]);
          } else if constexpr (EPI == 1) {
#pragma unroll
            for (int rr = 0; rr < 4; rr++)
              v[rr] = act_fn(fmaf(acc[i][j][blk * 4 + rr], rs_scale, fmaf(rs_mean, col_c[j][blk][rr], bias_v[j][blk][rr])));
          } else {
#pragma unroll
            for (int rr = 0; rr < 4; rr++) v[rr] = act_fn(acc[i][j][blk * 4 + rr] * p.scale + bias_v[j][blk][rr]);
          }
          OutT* dst = &strip[r * EPI_STRIDE + j * 32 + blk * 8 + g * 4];
          if constexpr (sizeof(OutT) == 1) {
            *reinterpret_cast<unsigned*>(dst) =
                PackFp8x4(v[0] * p.out_mul, v[1] * p.out_mul, v[2] * p.out_mul, v[3] * p.out_mul);
          } else {
            using ov4 = typename Vec16<OutT>::v4;
            ov4 h;
#pragma unroll
            for (int rr = 0; rr < 4; rr++) h[rr] = (OutT)v[rr];
            *reinterpret_cast<ov4*>(dst) = h;
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); the strip is private to this wave
      __builtin_amdgcn_wave_barrier();
      if constexpr (EPI == 2) {
        if (i + 1 < TM) load_skip(i + 1, sk_nxt);
      }
#pragma unroll
      for (int pass = 0; pass < NPASS; pass++) {
        const int idx = pass * 64 + lane;
        const int row = idx / CHUNKS_PER_ROW;
        const int ch = idx - row * CHUNKS_PER_ROW;
        const int m = m0 + wm * WM + i * 32 + row;
        const int n = n0 + wn * WN + ch * OV;
        if constexpr (EPI == 2) {
          // C = (scale * acc + bias, already rounded to half) + residual, the residual normalised on the way when
          // it is itself an un-normalised sum; then the partial sums of the stored values over this wave's columns.
          const bool ok = idx < STRIP_CHUNKS && m < M && n + OV - 1 < N;
          const half8 hv = *reinterpret_cast<const half8*>(&strip[row * EPI_STRIDE + ch * OV]);
          const half8 hs = __builtin_bit_cast(half8, sk_cur[pass]);
          float2 rm = make_float2(0.0f, 1.0f);
          if (norm_skip) rm = row_ms[wm * WM + i * 32 + min(row, 31)];
          const float neg_mean_rstd = -rm.x * rm.y;
          half8 o;
          float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float t = fmaf((float)hs[e], rm.y, neg_mean_rstd);
            const float u = fmaf(t, sk_gamma[e], sk_beta[e]) + (float)hv[e];
            o[e] = (half_t)u;
            s1 += u;            // (of the sums before rounding to half: the difference is far below the rounding
            s2 = fmaf(u, u, s2);   //  of the normalised values themselves)
          }
          // Columns past N (a last column tile that N does not fill) and rows past M hold products of clamped
          // operand rows: they are neither stored nor counted in the row statistics.
          if (!ok) s1 = s2 = 0.0f;
          if (ok) {
            half_t* dst = reinterpret_cast<half_t*>(C) + (long long)m * p.ldc + n;
            StoreOut16<STORES>(dst, __builtin_bit_cast(intx4, o));
          }
          // Sum over the CHUNKS_PER_ROW (4 or 8) neighbouring lanes of a row, with data-parallel-primitive moves.
          static_assert(CHUNKS_PER_ROW == 4 || CHUNKS_PER_ROW == 8, "row reduction written for 4 or 8 lanes per row");
          s1 += DppMove<0xB1>(s1);   // lane ^ 1
          s2 += DppMove<0xB1>(s2);
          s1 += DppMove<0x4E>(s1);   // lane ^ 2
          s2 += DppMove<0x4E>(s2);
          if constexpr (CHUNKS_PER_ROW == 8) {
            s1 += DppMove<0x141>(s1);   // mirror within 8 lanes: the other quad's sum
            s2 += DppMove<0x141>(s2);
          }
          if (ch == 0 && idx < STRIP_CHUNKS) part_lds[wn * BM + wm * WM + i * 32 + row] = make_float2(s1, s2);
          if (pass + 1 == NPASS && i + 1 < TM) {
#pragma unroll
            for (int q = 0; q < NPASS; q++) sk_cur[q] = sk_nxt[q];
          }
          continue;
        }
        if (idx < STRIP_CHUNKS && m < M && n < N) {
          OutT* dst = C + (long long)m * p.ldc + n;
          if (vec_ok && n + OV - 1 < N) {
            const intx4 val = *reinterpret_cast<const intx4*>(&strip[row * EPI_STRIDE + ch * OV]);
            StoreOut16<STORES>(dst, val);
          } else {
            for (int e = 0; e < OV && n + e < N; e++) dst[e] = strip[row * EPI_STRIDE + ch * OV + e];
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
    }
  });
  if constexpr (EPI == 2) {
    // Partial sums of this column tile: the WAVES_N wave columns added in a fixed order.
    if (p.stats_out != nullptr) {
      __syncthreads();
      if (tid < BM && m0 + tid < M) {
        float2 t = part_lds[tid];
#pragma unroll
        for (int w = 1; w < WAVES_N; w++) {
          t.x += part_lds[w * BM + tid].x;
          t.y += part_lds[w * BM + tid].y;
        }
        reinterpret_cast<float2*>(p.stats_out)[(long long)(m0 + tid) * gridDim.y + tile.y] = t;
      }
    }
  }
}

// Outputs of at least 64 MiB, or of 32 MiB (the size of L2) from at least 16384 rows, are written with streaming stores:
// cached, each round of output tiles would push out the operand rows that the next round reads again
// (measured on the same machine: BT4 batch 256 +0.7 %, fp8 batch 1024 +5 %). Smaller launches keep cached
// stores for the kernel that consumes the output (batch 128 loses 2.6 % with streaming, a 10x256 net at
// batch 64 loses 8 %). Only the BM = 256 tiles carry the variant: nothing else is picked for such outputs.
inline bool StreamOutput(long long m, long long n, long long batch, int elem_bytes) {
  const long long bytes = m * n * batch * elem_bytes;
  return bytes >= (64LL << 20) || (m >= 16384 && bytes >= (32LL << 20));
}

// The STORES instance for a launch: what the caller asked for (GemmArgs::out_stores), or by the size rule above.
inline int OutputStores(int requested, long long m, long long n, long long batch, int elem_bytes) {
  if (requested == kStoresCached) return 0;
  if (requested == kStoresStream) return 1;
  if (requested == kStoresWriteThrough) return 2;
  if (!StreamOutput(m, n, batch, elem_bytes)) return 0;
  return requested == kStoresAutoKeep ? 2 : 1;
}

template <typename ET, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int NSTAGES = 2, bool ALONE = false>
void LaunchGemmDma(const GemmArgs& args, hipStream_t stream) {
  GemmArgs a = args;
  dim3 grid((a.M + BM - 1) / BM, (a.N + BN - 1) / BN + (a.N2 + BN - 1) / BN, a.batch);
  a.tile_order = PickTileOrder(a.M, 1024, grid);
  const dim3 block(WAVES_M * WAVES_N * 64);
  auto launch = [&](auto stores_tag) {
    constexpr int S = decltype(stores_tag)::value;
    [[maybe_unused]] constexpr int SF = S == 2 ? 1 : S;   // (the folded-layer-norm epilogues know cached and streaming stores only)
    // The folded-layer-norm epilogues exist for halves and with two stages only (LaunchGemmDmaStaged sends them there).
    if constexpr (std::is_same<ET, half_t>::value && NSTAGES == 2) {
      if (a.skip != nullptr) {
        if constexpr ((BN / WAVES_N) % 64 == 0 || BN / WAVES_N == 32) {
          hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BK * 2, WAVES_M, WAVES_N, GemmArgs, half_t, SF, 2, 2>), grid, block,
                             0, stream, a);
        }
        return;
      }
      if (a.row_stats != nullptr) {
        hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BK * 2, WAVES_M, WAVES_N, GemmArgs, half_t, SF, 1, 2>), grid, block, 0,
                           stream, a);
        return;
      }
    }
    if constexpr (BM < 256 && BN >= 64) {
      if (a.N2 > 0) {
        hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BK * 2, WAVES_M, WAVES_N, GemmArgs, ET, S, 0, NSTAGES, ET, ALONE, true>), grid,
                           block, 0, stream, a);
        return;
      }
    }
    hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, BK * 2, WAVES_M, WAVES_N, GemmArgs, ET, S, 0, NSTAGES, ET, ALONE>), grid,
                       block, 0, stream, a);
  };
  if constexpr (BM == 256) {
    const int stores = OutputStores(a.out_stores, a.M, a.N, a.batch, 2);
    if (stores == 1) return launch(std::integral_constant<int, 1>{});
    if (stores == 2) return launch(std::integral_constant<int, 2>{});
  }
  launch(std::integral_constant<int, 0>{});
}

// As many LDS stages (2 to 4) as leave room on the CUs for all of the launch's workgroups at once: with one
// workgroup per CU nothing else hides the time a k-tile takes to arrive from memory, with several per CU they hide it
// for each other and more stages would only lower their number (15x1024 net, per pass: 16 positions 1.91 -> 1.67 ms
// with four stages; 64 positions 2.59 -> 2.93 ms if forced there).
// A count of stages is an instance only where it admits more workgroups than the one tried before it.
constexpr int WorkgroupsPerCu(int stages, int stage_bytes) { return 160 * 1024 / (stages * stage_bytes + 4096); }

template <typename ET, int BM, int BN, int BK, int WAVES_M, int WAVES_N>
void LaunchGemmDmaStaged(const GemmArgs& a, hipStream_t stream) {
  constexpr int kStage = (BM + BN) * BK * 2, kCus = 256;
  constexpr int kFour = WorkgroupsPerCu(4, kStage), kThree = WorkgroupsPerCu(3, kStage);
  constexpr bool kAlone = BM * BN <= 128 * 64;   // (an instance for one workgroup per CU, with four stages)
  const long long wgs = (long long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN + (a.N2 + BN - 1) / BN) * a.batch;
  if (a.skip != nullptr || a.row_stats != nullptr) return LaunchGemmDma<ET, BM, BN, BK, WAVES_M, WAVES_N, 2>(a, stream);
  if constexpr (kAlone) {
    if (wgs <= kCus) return LaunchGemmDma<ET, BM, BN, BK, WAVES_M, WAVES_N, 4, true>(a, stream);
  }
  if constexpr (kFour > (kAlone ? 1 : 0)) {
    if (wgs <= kCus * kFour) return LaunchGemmDma<ET, BM, BN, BK, WAVES_M, WAVES_N, 4>(a, stream);
  }
  if constexpr (kThree > kFour) {
    if (wgs <= kCus * kThree) return LaunchGemmDma<ET, BM, BN, BK, WAVES_M, WAVES_N, 3>(a, stream);
  }
  LaunchGemmDma<ET, BM, BN, BK, WAVES_M, WAVES_N, 2>(a, stream);
}

template <typename ET>
void LaunchGemmDmaVariant(GemmVariant v, const GemmArgs& a, hipStream_t stream) {
  switch (v) {
    case kDma256x256: LaunchGemmDma<ET, 256, 256, 64, 2, 4>(a, stream); break;
    case kDma256x192: LaunchGemmDma<ET, 256, 192, 64, 4, 2>(a, stream); break;
    case kDma256x128: LaunchGemmDmaStaged<ET, 256, 128, 32, 4, 2>(a, stream); break;
    case kDma128x128: LaunchGemmDmaStaged<ET, 128, 128, 64, 2, 2>(a, stream); break;
    case kDma128x64: LaunchGemmDmaStaged<ET, 128, 64, 64, 2, 2>(a, stream); break;
    case kDma128x32: LaunchGemmDma<ET, 128, 32, 64, 4, 1>(a, stream); break;
    case kDma64x64: LaunchGemmDmaStaged<ET, 64, 64, 64, 2, 2>(a, stream); break;
    default: throw std::runtime_error("LaunchGemmDmaVariant: not a direct-to-LDS variant");
  }
}

}  // namespace

}  // namespace lc0mi
