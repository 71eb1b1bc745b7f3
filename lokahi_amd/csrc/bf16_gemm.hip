// Dense bf16 linear for several rows: Y[M, N] = X[M, K] @ W[N, K]^T on bf16
// MFMA with fp32 accumulation (the unquantized `_linear` branch,
// src/ollm/llama_mlx.py:64-65, for the bf16 lm_head at 886-910).
//
// Bound by the weight stream up to ~150 rows (1.05 GB at 128256 x 4096) and
// by LDS bandwidth beyond, so every weight is read once per 160 x rows and a
// workgroup keeps two K steps of both operands in flight:
//   * Workgroup tile TM x rows x 256 W rows, 8 waves as 2 (x rows) x 4 (W
//     rows), K step 64; both operands go straight from global memory to LDS
//     (three stages, 16-byte chunks XOR-swizzled: chunk c of row r at
//     c ^ ((r >> 1) & 7), so an operand read of 16 rows meets 16 distinct
//     16-byte slots of the 64 banks).
//   * TM is a multiple of 32 up to 160, chosen by cost (pick_tm): padding
//     rows cost LDS reads and MFMAs, a second tile of rows re-reads W.
//   * W is the A operand and x the B operand, so a lane holds 4 consecutive
//     output columns of one x row (one 16-byte store).
//   * Workgroup b starts its K loop at step 5 (W tile) mod K/64: in lockstep
//     all workgroups would read addresses equal modulo the row size, 8 KB at
//     K = 4096, from a few channels (230 -> 173 us at 4 rows).
//   * Sums are built over chains of 2 K steps and added to the total with
//     compensation (the error of each addition starts the next chain), so the
//     result is no further from the exact product than the dot2 GEMV's:
//     6.6e-8 (2-norm, K = 4096) against 8.3e-8; one chain over all of K is
//     4.0e-7, plain sums of 4-step chains 1.2e-7 and 13% faster at 300 rows.
// Measured on MI355X, 128256 x 4096, fp32 logits (the 4-row GEMV passes ->
// this kernel): 8 rows 339 -> 172 us, 32 rows 1360 -> 182, 64 rows 2740 ->
// 191, 300 rows 13060 -> 438, 512 rows ~22000 -> 675 us.  At 300 rows the
// loads alone take 317 us and LDS reads and MFMAs alone 298 (W from L2).
#include <algorithm>

#include "strata_internal.h"

namespace {

constexpr int TN = 256, BK = 64;   // W rows and K per step of a workgroup tile
constexpr int NWAVE = 8;           // 2 (x rows) x 4 (W rows)
constexpr int ROWB = BK * 2;       // bytes per staged row
constexpr int kRotate = 5;         // K steps between the starts of neighbouring W tiles
constexpr int kChain = 2;          // K steps per accumulation chain

template <int TM>
struct BTile {
  static constexpr int kStage = (TN + TM) * ROWB;   // W tile, then x tile
  static constexpr int NST = 3;
  static constexpr size_t kLds = (size_t)NST * kStage;
};

__device__ __forceinline__ f32x4_t mfma16(const uint4& a, const uint4& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  const bf16x2_t v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// K % 64 == 0, ldx % 8 == 0, x and w 16-byte aligned.  Grid: the nm row tiles
// of one W tile run in consecutive slots of one XCD (block b runs on XCD
// b % 8), so the second reads W from that L2.
template <int TM, typename YT>
__global__ __launch_bounds__(NWAVE * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bf16_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int64_t ldx,
                      int M, int K, int N, int nm, int nnt, YT* __restrict__ y) {
  constexpr int kStage = BTile<TM>::kStage, NST = BTile<TM>::NST;
  constexpr int WM = TM / 2, MBW = WM / 16, NBW = 4;
  constexpr int WI = TN / 8 / NWAVE;                    // W loads per lane per step
  constexpr int XI = (TM / 8 + NWAVE - 1) / NWAVE;      // X loads per lane per step
  constexpr int D = WI + XI;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int nt = (slot / nm) * 8 + xcd, mt = slot % nm;
  if (nt >= nnt) return;
  const int n0 = nt * TN, m0 = mt * TM;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int c16 = lane & 15, q = lane >> 4;
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)lds);
  const uint32_t kb = (uint32_t)K * 2, xb = (uint32_t)ldx * 2;
  const v4i32_t rw = rsrc(w + (int64_t)n0 * K, (uint32_t)min(N - n0, TN) * kb);
  const v4i32_t rx = rsrc(x + (int64_t)m0 * ldx, (uint32_t)(min(M - m0, TM) - 1) * xb + kb);

  // Load idx of a tile fills the 1 KB of its rows 8 idx .. +7: lane l brings
  // row 8 idx + l / 8, chunk (l % 8) ^ swizzle, and the swizzle depends on
  // idx's parity only.  x tiles have TM / 8 loads for 8 waves: a wave left
  // over repeats another's (the same bytes to the same place).
  const uint32_t sw0 = ((lane & 7) ^ (lane >> 4)) << 4, sw1 = ((lane & 7) ^ (4 + (lane >> 4))) << 4;
  const uint32_t wv0 = (lane >> 3) * kb + sw0, wv1 = (lane >> 3) * kb + sw1;
  uint32_t xv[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i)
    xv[i] = (lane >> 3) * xb + ((((i * NWAVE + wave) % (TM / 8)) & 1) ? sw1 : sw0);
  auto issue = [&](int g, int st) {
    const uint32_t base = lds0 + st * kStage;
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int idx = wave * WI + i;
      dma16(base + idx * 1024, (i & 1) ? wv1 : wv0, rw, idx * 8 * kb + g * ROWB);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int idx = (i * NWAVE + wave) % (TM / 8);
      dma16(base + TN * ROWB + idx * 1024, xv[i], rx, idx * 8 * xb + g * ROWB);
    }
  };

  f32x4_t acc[NBW][MBW];
#pragma unroll
  for (int i = 0; i < NBW; ++i)
#pragma unroll
    for (int j = 0; j < MBW; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int G = K / BK;
  const int rot = (int)((uint32_t)nt * kRotate % (uint32_t)G);
  // step t of this workgroup's order; steps past the last repeat it (their
  // loads land in a stage that is not read again)
  auto kstep = [&](int t) { t = min(t, G - 1) + rot; return t < G ? t : t - G; };
  for (int s = 0; s < NST - 1; ++s) issue(kstep(s), s);
  const int a0 = (wn * 64 + c16) * ROWB, b0 = TN * ROWB + (wm * WM + c16) * ROWB;
  const int sk = (c16 >> 1) & 7;
  int st = 0;
  // in: the current chain, started at minus the rounding error of the last
  // addition to acc (compensated summation, the correction rides in the chain)
  f32x4_t in[NBW][MBW];
#pragma unroll
  for (int i = 0; i < NBW; ++i)
#pragma unroll
    for (int j = 0; j < MBW; ++j) in[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int gb = 0; gb < G; gb += kChain) {
    const int ge = min(G, gb + kChain);
    for (int g = gb; g < ge; ++g) {
      // this lane's loads of step g are done, then every lane's; the barrier
      // also means that all waves have read the stage refilled below
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NST - 2) * D) : "memory");
      __syncthreads();
      const uint8_t* sb = lds + st * kStage;
      uint4 a[2][NBW], b[2][MBW];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int ch = ((4 * kk + q) ^ sk) << 4;
#pragma unroll
        for (int i = 0; i < NBW; ++i)
          a[kk][i] = *reinterpret_cast<const uint4*>(sb + a0 + i * 16 * ROWB + ch);
#pragma unroll
        for (int j = 0; j < MBW; ++j)
          b[kk][j] = *reinterpret_cast<const uint4*>(sb + b0 + j * 16 * ROWB + ch);
      }
      __builtin_amdgcn_sched_barrier(0);
      issue(kstep(g + NST - 1), st == 0 ? NST - 1 : st - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int j = 0; j < MBW; ++j)
#pragma unroll
          for (int i = 0; i < NBW; ++i) in[i][j] = mfma16(a[kk][i], b[kk][j], in[i][j]);
      st = st == NST - 1 ? 0 : st + 1;
    }
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) {
        const f32x4_t t = acc[i][j] + in[i][j];
        in[i][j] -= t - acc[i][j];
        // once t is infinite the error is NaN: any finite start will do then
#pragma unroll
        for (int r = 0; r < 4; ++r) in[i][j][r] = __builtin_amdgcn_fmed3f(in[i][j][r], -1e30f, 1e30f);
        acc[i][j] = t;
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the wave

  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
  for (int j = 0; j < MBW; ++j) {
    const int m = m0 + wm * WM + 16 * j + c16;
    if (m >= M) continue;
    YT* yr = y + (int64_t)m * N;
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
      const int n = n0 + wn * 64 + 16 * i + 4 * q;
      if (vec) {
        if (n < N) {
          if constexpr (sizeof(YT) == 4)
            *reinterpret_cast<float4*>(yr + n) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
          else
            *reinterpret_cast<uint2*>(yr + n) = make_uint2(pk_bf16(acc[i][j][0], acc[i][j][1]),
                                                           pk_bf16(acc[i][j][2], acc[i][j][3]));
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) Elem<YT>::store(yr, n + r, acc[i][j][r]);
      }
    }
  }
}

template <int TM, typename YT>
void go_t(const uint16_t* x, const uint16_t* w, int64_t ldx, int M, int K, int N, void* y,
          hipStream_t s) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)bf16_gemm_kernel<TM, YT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, BTile<TM>::kLds);
    attr = true;
  }
  const int nm = (M + TM - 1) / TM, nnt = (N + TN - 1) / TN;
  hipLaunchKernelGGL((bf16_gemm_kernel<TM, YT>), dim3((nnt + 7) / 8 * 8 * nm), dim3(NWAVE * 64),
                     BTile<TM>::kLds, s, x, w, ldx, M, K, N, nm, nnt, static_cast<YT*>(y));
}

template <int TM>
void go(const uint16_t* x, const uint16_t* w, int64_t ldx, int M, int K, int N, void* y,
        int y_dtype, hipStream_t s) {
  if (y_dtype == STRATA_F32) go_t<TM, float>(x, w, ldx, M, K, N, y, s);
  else go_t<TM, bf16_t>(x, w, ldx, M, K, N, y, s);
}

// x rows per tile: one workgroup per CU takes ~0.25 + 0.0057 TM us per K step
// (MI355X, W from L2: 0.43 us at TM = 32, 0.91 at 128, 1.16 at 160), so the
// fewest rounds times that.
int pick_tm(int M, int N, int cus) {
  const int64_t nnt = (N + TN - 1) / TN;
  int best = 32;
  double least = 0;
  for (int tm = 32; tm <= 160; tm += 32) {
    const int64_t rounds = ((int64_t)((M + tm - 1) / tm) * nnt + cus - 1) / cus;
    const double cost = (double)rounds * (0.25 + 0.0057 * tm);
    if (tm == 32 || cost < least) {
      least = cost;
      best = tm;
    }
  }
  return best;
}

// The GEMV reads all of W once per 4 rows (2 rows when M < 4), the GEMM once per
// tile of up to 160 rows but walks K in ~0.7 us steps while its tiles leave CUs
// idle.  So it wins from a number of passes x N that grows with K as a pass of the
// GEMV gets cheaper per byte, up to K = 4096, where 64 lanes with 8 loads each
// are full.  Microseconds, GEMV | this kernel, weights from HBM:
//   rows, N:   8, 8192       16, 8192     32, 4096     3, 12288     64, 2048     8, 24576
//   K = 1024   14.2 | 13.1   25.5 | 13.6  24.5 | 14.5  13.9 | 13.2  22.7 | 13.9   34.3 | 14.8
//   K = 2048   18.4 | 23.4   32.6 | 24.0  32.4 | 25.6  18.0 | 23.5  29.2 | 24.5   44.8 | 26.6
//   K = 4096   22.6 | 43.5   40.7 | 45.3  37.9 | 47.5  31.4 | 44.4  41.4 | 46.0   62.4 | 50.5
//   K = 8192   50.3 | 84.5   94.0 | 86.8  94.4 | 89.4  63.3 | 78.9  95.1 | 86.6  136.4 | 94.1
// (K = 6144, 8 rows of 8192: 40 | 82).  One 4-row pass loses to the GEMM on large
// W only, and only where K leaves more than an eighth of the lanes' last step
// empty: 128256 x 3072 146 | 138, x 3584 157 | 160, x 4096 168 | 182, x 6144 274 |
// 269, x 8192 348 | 353; 32000 x 3072 41 | 46.
bool gemm_wins(int M, int K, int N) {
  if (M < 3) return false;
  if (M == 4) return N >= 65536 && (int64_t)K * 8 < (int64_t)(K + 4095) / 4096 * 4096 * 7;
  const int64_t passes = M > 4 ? (M + 3) / 4 : 2;
  return passes * N >= (K <= 4096 ? 16384 + 6 * K : K < 8192 ? 40960 : 32768);
}

}  // namespace

int strata_bf16_linear(strata_ctx* ctx, const void* x, int64_t ldx, int M, int K,
                       const uint16_t* w, int N, void* y, int y_dtype, void* stream) {
  const bool fits = K % BK == 0 && ldx % 8 == 0 && (uint64_t)ldx * 160 * 2 + (uint64_t)K * 2 < (1ull << 32) &&
                    (uint64_t)K * TN * 2 < (1ull << 32);
  bool gemm = fits && (gemm_wins(M, K, N) || !strata_bf16_gemv_fits(ctx, M, K));
  if (ldx != K && M > 1) gemm = fits;  // the GEMV takes contiguous rows
  if (gemm) {
    const uint16_t* xx = static_cast<const uint16_t*>(x);
    hipStream_t s = as_stream(stream);
    switch (pick_tm(M, N, ctx->num_cus)) {
      case 32: go<32>(xx, w, ldx, M, K, N, y, y_dtype, s); break;
      case 64: go<64>(xx, w, ldx, M, K, N, y, y_dtype, s); break;
      case 96: go<96>(xx, w, ldx, M, K, N, y, y_dtype, s); break;
      case 128: go<128>(xx, w, ldx, M, K, N, y, y_dtype, s); break;
      default: go<160>(xx, w, ldx, M, K, N, y, y_dtype, s);
    }
    STRATA_HIP_CHECK(hipGetLastError());
    return STRATA_OK;
  }
  if (ldx == K || M == 1) return strata_bf16_gemv(ctx, x, M, K, w, N, y, y_dtype, stream);
  for (int m = 0; m < M; ++m) {
    const int rc = strata_bf16_gemv(ctx, static_cast<const uint16_t*>(x) + (int64_t)m * ldx, 1, K, w, N,
                                    static_cast<char*>(y) + (int64_t)m * N * dtype_size(y_dtype),
                                    y_dtype, stream);
    if (rc) return rc;
  }
  return STRATA_OK;
}
