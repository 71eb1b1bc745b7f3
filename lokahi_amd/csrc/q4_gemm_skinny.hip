// q4 linear for a few rows (3 <= M < 40, narrow linears up to 64): Y[M, N] =
// X[M, K] @ dequant(W)[N, K]^T on bf16 16x16x32 MFMAs, every weight read once.
//
// Same maths as mx.quantized_matmul(transpose=True) (src/ollm/llama_mlx.py:
// 53-74, the prefill call at 393-432 with a short prompt): each weight is
// s * q + b in fp32, rounded once to bf16 (as the 256-tile GEMM does), and the
// products accumulate in fp32.
//
// Sizing for MI355X: the 128 x 128-tile kernel (q4_gemm.hip) covers a 6144 x
// 4096 projection at 16 rows with 48 workgroups and takes ~230 us; here every
// workgroup owns only NC x 16 output columns, so the same launch has 384-1536
// workgroups streaming their weight rows in parallel.
//   * Workgroup = 4 waves on the same NC x 16 columns; wave w reduces the K
//     quarter w, and the four partial sums meet in LDS at the end.
//   * Per 128-k chunk lane (c, g) needs, of each of its NC columns (row n0 +
//     16 cc + c), the 16-byte code run of k 32 g .. +32 with that group's scale
//     and bias, and of each of its MB x row blocks (row 16 mb + c) the 32 x
//     values of the same k.  Word j of the run is the B operand of MFMA k-step
//     j: the lane supplies k slots 8 g .. +7 of each 32-k step from k 32 g + 8 j
//     .. +8, and its A operand (x) uses the same k, so the dot products are
//     unchanged.
//   * All of it reaches LDS by direct global -> LDS loads into a ring private
//     to the wave (NST stages, no barrier), four x rows of 256 bytes or 16
//     weight rows of 64 bytes per instruction.  Loaded straight into
//     registers, an x instruction touched 32 cache lines (64-byte strides) and
//     those were most of the time (24 rows: 3B down, 3072 x 8192, 20.7 -> 11.9
//     us; 8B down 34.3 -> 20.2, q/k/v 21.1 -> 12.7, gate/up 49.8 -> 36.3).
//     16-byte slots are XOR-swizzled so that the operand reads of 16 lanes meet
//     16 distinct slots of the 64 banks.
//   * Outputs: lane (c, g) of the 16x16 accumulator holds column c and rows
//     4 g .. 4 g + 3.
#include "strata_internal.h"

namespace {

struct SkinnyProblem {
  const uint4* w;      // [n, K/32] uint4
  const uint16_t* s;   // [n, K/64]
  const uint16_t* b;
  void* y;             // [M, n]
  int n;
  int col0;            // first column of this linear in the launch
};

struct SkinnyBatch {
  SkinnyProblem p[kMaxGemmProblems];
  int count;
};

__device__ __forceinline__ f32x4_t mfma16x32(const uint4& a, const uint4& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  const bf16x2_t v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// 8 codes of one word (k order, nibble i = code i) -> 8 bf16 s*q + b
__device__ __forceinline__ uint4 dequant8(uint32_t w, float s, float b) {
  const uint32_t lo = w & 0x0f0f0f0fu;         // codes 0, 2, 4, 6
  const uint32_t hi = (w >> 4) & 0x0f0f0f0fu;  // codes 1, 3, 5, 7
  uint4 o;
  o.x = pk_bf16(fmaf(s, (float)(lo & 0xffu), b), fmaf(s, (float)(hi & 0xffu), b));
  o.y = pk_bf16(fmaf(s, (float)((lo >> 8) & 0xffu), b), fmaf(s, (float)((hi >> 8) & 0xffu), b));
  o.z = pk_bf16(fmaf(s, (float)((lo >> 16) & 0xffu), b), fmaf(s, (float)((hi >> 16) & 0xffu), b));
  o.w = pk_bf16(fmaf(s, (float)(lo >> 24), b), fmaf(s, (float)(hi >> 24), b));
  return o;
}

template <int MB, int NC>
struct SkinnyStage {
  static constexpr int kX = MB * 16 * 256, kW = NC * 16 * 64, kSB = NC * 2 * 256;
  static constexpr int kBytes = kX + kW + kSB;
  static constexpr int kLoads = MB * 4 + NC * 3;  // per lane and chunk
};

// EXACT (at most 8 rows of the decode linears, MB = 1): the weights are not
// rounded.  Codes enter the MFMA as the exact bf16 values 128 + q (a mask and
// an OR per pair, x permuted to the pairs' order), every 32 k sum on their own,
// and the group's scale and bias apply to the fp32 sums: y += s sum x (128 + q)
// + (b - 128 s) sum x, the sums of x from MFMAs against ones.  (Sums over the
// whole group of 64 are 15% further from the exact product than the GEMV's
// 32-element slices, these are not.)
template <int MB, int NC, int NST, bool EXACT, typename YT>
__global__ __launch_bounds__(256) void q4_gemm_skinny_kernel(const uint16_t* __restrict__ x, int M,
                                                             int K, SkinnyBatch bt) {
  using S = SkinnyStage<MB, NC>;
  constexpr int RING = NST * S::kBytes;
  static_assert(MB * NC * 64 * 16 <= RING, "a wave's ring holds its partial sums");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_all[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, kq = lane >> 4;
  const int col0 = blockIdx.x * (16 * NC);
  int p = 0;
#pragma unroll
  for (int t = 1; t < kMaxGemmProblems; ++t)
    if (t < bt.count && col0 >= bt.p[t].col0) p = t;
  const SkinnyProblem& P = bt.p[p];
  const int n0 = col0 - P.col0;
  const int kw = K >> 2, kbeg = wave * kw, nch = kw >> 7;
  const uint32_t xb = (uint32_t)K * 2, wb = (uint32_t)K / 2, sb = (uint32_t)K / 32;  // bytes per row
  // x rows at or past M read as zero
  const v4i32_t rx = rsrc(x, (uint32_t)M * xb);
  const v4i32_t rw = rsrc(reinterpret_cast<const uint8_t*>(P.w) + (int64_t)n0 * wb, 16 * NC * wb);
  const v4i32_t rs = rsrc(reinterpret_cast<const uint8_t*>(P.s) + (int64_t)n0 * sb, 16 * NC * sb);
  const v4i32_t rb = rsrc(reinterpret_cast<const uint8_t*>(P.b) + (int64_t)n0 * sb, 16 * NC * sb);
  uint8_t* lds = lds_all + wave * RING;
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)lds);
  // x load i fills rows 4 i .. +3: slot q of row r holds 16-byte chunk q ^ (r % 16)
  uint32_t xv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xv[i] = kq * xb + ((c ^ (4 * i + kq)) << 4);
  // a weight load fills 16 rows: slot q of row r holds piece q ^ (r / 4 % 4)
  const uint32_t wv = (lane >> 2) * wb + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  // the chunk's first group for kq < 2, its second for the others; 2-byte loads,
  // as scales and biases may start at any 2-byte address (as fast as the pairs in
  // 4-byte loads: 28672 x 4096, 24 rows 40 us, 5 rows 31)
  const uint32_t sv = c * sb + (kq >> 1) * 2;
  auto issue = [&](int ch, int st) {
    const uint32_t k = kbeg + (ch << 7), base = lds0 + st * S::kBytes;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      dma16(base + S::kX + cc * 1024, wv, rw, 16 * cc * wb + k / 2);
      dma2(base + S::kX + S::kW + cc * 512, sv, rs, 16 * cc * sb + k / 32);
      dma2(base + S::kX + S::kW + cc * 512 + 256, sv, rb, 16 * cc * sb + k / 32);
    }
#pragma unroll
    for (int i = 0; i < MB * 4; ++i) dma16(base + i * 1024, xv[i & 3], rx, 4 * i * xb + k * 2);
  };

  f32x4_t acc[MB][NC];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) acc[mb][cc] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (int s = 0; s < NST - 1; ++s) issue(min(s, nch - 1), s);
  int st = 0;
  for (int ch = 0; ch < nch; ++ch) {
    // The stage read last is refilled (past the end with the last chunk again,
    // which nothing reads): its LDS reads are done first.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(min(ch + NST - 1, nch - 1), st == 0 ? NST - 1 : st - 1);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NST - 1) * S::kLoads) : "memory");
    const uint8_t* sg = lds + st * S::kBytes;
    if constexpr (EXACT) {
      static_assert(MB == 1, "one block of rows");
      const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
      uint4 xp[4];  // k 32 s + 8 kq .. +7 in the order 0 4 1 5 2 6 3 7
      uint32_t wd[NC][4], sr[NC][2], br[NC][2];
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          sr[cc][g] = *reinterpret_cast<const uint32_t*>(sg + S::kX + S::kW + cc * 512 + (32 * g + c) * 4);
          br[cc][g] = *reinterpret_cast<const uint32_t*>(sg + S::kX + S::kW + cc * 512 + 256 + (32 * g + c) * 4);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          wd[cc][j] = *reinterpret_cast<const uint32_t*>(sg + S::kX + cc * 1024 + c * 64 +
                                                         ((j ^ (c >> 2)) << 4) + kq * 4);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 v = *reinterpret_cast<const uint4*>(sg + c * 256 + (((4 * j + kq) ^ c) << 4));
        xp[j] = make_uint4(__builtin_amdgcn_perm(v.z, v.x, 0x05040100), __builtin_amdgcn_perm(v.z, v.x, 0x07060302),
                           __builtin_amdgcn_perm(v.w, v.y, 0x05040100), __builtin_amdgcn_perm(v.w, v.y, 0x07060302));
      }
      const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t xs = mfma16x32(xp[j], ones, zero);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) {
          const uint32_t w = wd[cc][j];
          const f32x4_t d =
              mfma16x32(xp[j], make_uint4((w & 0x000f000fu) | 0x43004300u, ((w >> 4) & 0x000f000fu) | 0x43004300u,
                                          ((w >> 8) & 0x000f000fu) | 0x43004300u,
                                          ((w >> 12) & 0x000f000fu) | 0x43004300u), zero);
          const float s = __uint_as_float(sr[cc][j >> 1] << 16), b = __uint_as_float(br[cc][j >> 1] << 16);
          const float cb = fmaf(-128.f, s, b);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[0][cc][r] = fmaf(cb, xs[r], fmaf(s, d[r], acc[0][cc][r]));
        }
      }
    } else {
    uint4 xr[MB][4], wr[NC];
    uint32_t sr[NC], br[NC];
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      wr[cc] = *reinterpret_cast<const uint4*>(sg + S::kX + cc * 1024 + c * 64 + ((kq ^ (c >> 2)) << 4));
      sr[cc] = *reinterpret_cast<const uint32_t*>(sg + S::kX + S::kW + cc * 512 + lane * 4);
      br[cc] = *reinterpret_cast<const uint32_t*>(sg + S::kX + S::kW + cc * 512 + 256 + lane * 4);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xr[mb][j] = *reinterpret_cast<const uint4*>(sg + (16 * mb + c) * 256 + (((4 * kq + j) ^ c) << 4));
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      const float s = __uint_as_float(sr[cc] << 16), b = __uint_as_float(br[cc] << 16);
      const uint32_t ww[4] = {wr[cc].x, wr[cc].y, wr[cc].z, wr[cc].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 bw = dequant8(ww[j], s, b);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb][cc] = mfma16x32(xr[mb][j], bw, acc[mb][cc]);
      }
    }
    }
    st = st == NST - 1 ? 0 : st + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the ring is the wave's again

  // the four K quarters meet in LDS; wave 0 adds them in wave order and stores
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < MB * NC; ++i)
      reinterpret_cast<f32x4_t*>(lds)[i * 64 + lane] = acc[i / NC][i % NC];
  }
  __syncthreads();
  if (wave != 0) return;
  YT* y = static_cast<YT*>(P.y);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      f32x4_t v = acc[mb][cc];
#pragma unroll
      for (int w = 1; w < 4; ++w)
        v += reinterpret_cast<const f32x4_t*>(lds_all + w * RING)[(mb * NC + cc) * 64 + lane];
      const int n = n0 + 16 * cc + c;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * mb + 4 * kq + r;
        if (m < M) Elem<YT>::store(y, (int64_t)m * P.n + n, v[r]);
      }
    }
}

template <int MB, int NC, int NST, bool EXACT, typename YT>
void launch_skinny_t(const uint16_t* x, int M, int K, const SkinnyBatch& bt, int cols,
                     hipStream_t stream) {
  constexpr int lds = 4 * NST * SkinnyStage<MB, NC>::kBytes;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)q4_gemm_skinny_kernel<MB, NC, NST, EXACT, YT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  hipLaunchKernelGGL((q4_gemm_skinny_kernel<MB, NC, NST, EXACT, YT>), dim3(cols / (16 * NC)), dim3(256), lds,
                     stream, x, M, K, bt);
}
// Two stages: a third costs workgroups per CU (8B gate/up, 9 rows: 29 us
// against 33, down 24 rows 20 against 23).
template <int MB, int NC>
void launch_skinny(const uint16_t* x, int M, int K, const SkinnyBatch& bt, int cols, int y_dtype,
                   hipStream_t stream) {
  if (y_dtype == STRATA_BF16) launch_skinny_t<MB, NC, 2, false, bf16_t>(x, M, K, bt, cols, stream);
  else launch_skinny_t<MB, NC, 2, false, float>(x, M, K, bt, cols, stream);
}

}  // namespace

bool strata_q4_skinny_fits(int M, int K, const strata_q4_weight* ws, int count) {
  if (M < 1 || M > kSkinnyMaxRows || K % 512 != 0 || count < 1 || count > kMaxGemmProblems)
    return false;
  // byte offsets into x and into a workgroup's up to 64 weight rows are 32-bit
  if ((uint64_t)M * K * 2 >= (1ull << 32) || (uint64_t)64 * K / 2 >= (1ull << 32)) return false;
  for (int i = 0; i < count; ++i)
    if (ws[i].N % 16 != 0 || !aligned16(ws[i].w)) return false;
  return true;
}

// The GEMV spends 4 dots per code and row and takes rows in blocks of 4 (2 for 3
// rows, or where 4 rows of x exceed its LDS), in steps of 4096 k (64 lanes, two
// 16-byte loads of codes each): its time follows the row blocks and, up to K =
// 8192, the whole steps that K takes.  This kernel's depends on K and the columns
// only.  So up to 4 rows (one row block, or two of 2) stay with the GEMV where K
// fills its steps.  Microseconds, GEMV | this kernel, weights from HBM:
//   rows  columns x K:  4096 x 4096  6144 x 4096  28672 x 4096  28672 x 3584  8192 x 8192  28672 x 8192
//   3                   7.3 |  6.7  10.4 |  9.6   29.5 | 30.7   28.5 | 26.1  22.6 | 18.9   53.6 | 57.5
//   4                   7.3 |  6.8   9.0 |  9.8   27.6 | 30.4   26.9 | 26.1  22.4 | 19.1   54.3 | 58.2
//   8                  12.2 |  6.8  15.3 |  9.9   46.7 | 31.0   46.3 | 26.6  39.2 | 20.1  103.1 | 59.2
// and 4096 x 14336: 4 rows 32.5 | 18.4, 8 rows 60.7 | 18.7.  Both are as long as a
// chain over K for narrow linears, this one the longer (8 rows, 1024 columns: K =
// 3072 5.8 | 5.3, 8192 7.6 | 9.6; 4 rows, 14336 8.9 | 14.4); the columns are left
// out of the rule, as a linear gives the same bits in a fused call as alone and
// q/k/v are best in one launch.
bool strata_q4_few_rows_on_mfma(int M, int K) {
  const bool full = K % 4096 == 0 && K <= 8192;
  return M >= 3 && M <= 8 && !(M <= 4 && full);
}

int strata_q4_gemm_skinny(const void* x, int M, int K, const strata_q4_weight* ws, int count,
                          int y_dtype, void* stream, bool exact) {
  STRATA_REQUIRE(strata_q4_skinny_fits(M, K, ws, count),
                 "q4 skinny GEMM: needs 1 <= M <= %d, K %% 512 == 0, N %% 16 == 0, operands under 4 GiB",
                 kSkinnyMaxRows);
  STRATA_REQUIRE(aligned16(x), "q4 skinny GEMM: x must be 16-byte aligned");
  SkinnyBatch bt{};
  bt.count = count;
  int cols = 0;
  bool n64 = true;  // every linear a multiple of 64 columns
  for (int i = 0; i < count; ++i) {
    bt.p[i] = SkinnyProblem{reinterpret_cast<const uint4*>(ws[i].w), ws[i].scales, ws[i].biases,
                            ws[i].y, static_cast<int>(ws[i].N), cols};
    cols += static_cast<int>(ws[i].N);
    n64 = n64 && ws[i].N % 64 == 0;
  }
  hipStream_t s = as_stream(stream);
  const uint16_t* xx = static_cast<const uint16_t*>(x);
  if (exact) {
    STRATA_REQUIRE(M <= 16, "q4 skinny GEMM: at most 16 rows without rounding");
    const bool bf = y_dtype == STRATA_BF16;
    if (n64 && cols >= 16384) {
      if (bf) launch_skinny_t<1, 4, 2, true, bf16_t>(xx, M, K, bt, cols, s);
      else launch_skinny_t<1, 4, 2, true, float>(xx, M, K, bt, cols, s);
    } else {
      if (bf) launch_skinny_t<1, 1, 2, true, bf16_t>(xx, M, K, bt, cols, s);
      else launch_skinny_t<1, 1, 2, true, float>(xx, M, K, bt, cols, s);
    }
    STRATA_HIP_CHECK(hipGetLastError());
    return STRATA_OK;
  }
  // 64-column workgroups (4 column blocks share each x fragment) when that
  // still gives >= 256 workgroups, else 16-column workgroups; x row blocks of
  // 16 per wave up to 3 (64 columns) or 4 (16 columns) within LDS (39 rows, 64
  // against 16 columns: 8B gate/up 46 against 69 us, 3B 20 against 33).
  const bool wide = n64 && cols >= 16384 && M <= 48;
  if (wide) {
    if (M <= 16) launch_skinny<1, 4>(xx, M, K, bt, cols, y_dtype, s);
    else if (M <= 32) launch_skinny<2, 4>(xx, M, K, bt, cols, y_dtype, s);
    else launch_skinny<3, 4>(xx, M, K, bt, cols, y_dtype, s);
  } else {
    if (M <= 16) launch_skinny<1, 1>(xx, M, K, bt, cols, y_dtype, s);
    else if (M <= 32) launch_skinny<2, 1>(xx, M, K, bt, cols, y_dtype, s);
    else launch_skinny<4, 1>(xx, M, K, bt, cols, y_dtype, s);
  }
  STRATA_HIP_CHECK(hipGetLastError());
  return STRATA_OK;
}
