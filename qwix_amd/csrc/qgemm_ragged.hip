// Ragged GEMM (mixture of experts): the tile bodies of qgemm_tiles.h behind a group lookup on the device.
#include "common.h"
#include "qgemm_tiles.h"

namespace qwix {
namespace {

template <int QT, int BM, int BN, int WGM, int WGN, int OUT>
__global__ void __launch_bounds__(WGM * WGN * 64)
    qgemm_ragged_dma_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                            Ragged rg, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  int g, m0, m_lim, n0;
  const int kind = ragged_tile<BM, BN>(rg, M, N, &g, &m0, &m_lim, &n0);
  if (kind == 0) return;
  using OutT = typename std::conditional<OUT == QWIX_BF16, uint16_t, uint32_t>::type;
  if (kind == 2) {
    zero_tile<BM, BN, OutT>(out, ldo, m0, m_lim, n0, N, WGM * WGN * 64);
    return;
  }
  const Epilogue e = group_epilogue(ep, rg, g);
  qgemm_dma_tile<QT, BM, BN, WGM, WGN, OUT, (OUT == QWIX_I32 ? 0 : 2)>(A, lda, B + g * rg.b_group_stride, ldb, m0, n0,
                                                                        m_lim, N, K, e, out, ldo);
}

template <int QT, int OUT, int EPI, int TM>
__global__ void __launch_bounds__(512)
    qgemm_ragged_pp_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                           Ragged rg, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  int g, m0, m_lim, n0;
  const int kind = ragged_tile<64 * TM, 256>(rg, M, N, &g, &m0, &m_lim, &n0);
  if (kind == 0) return;
  using OutT = typename std::conditional<OUT == QWIX_BF16, uint16_t, uint32_t>::type;
  if (kind == 2) {
    zero_tile<64 * TM, 256, OutT>(out, ldo, m0, m_lim, n0, N, 512);
    return;
  }
  const Epilogue e = group_epilogue(ep, rg, g);
  // The last tile of a group is no higher than its rows need: 64, 128 or 192 rows cost 0.4, 0.6 and 0.8 of 256.  2843 rows in 32 groups, N 1984
  // over K 1792, int8 37.6 -> 29.2 us; 2097 in 8, N 13248 over K 1536 85.7 -> 72.1; where groups are many tiles high little is left to gain (8192
  // in 8, N 14336 over K 4096, four draws of the sizes, int8 484 to 496 -> 471 to 491).
  const uint8_t* bg = B + g * rg.b_group_stride;
  const int rows = m_lim - m0;
  if (rows <= 64) qgemm_pp_tile<QT, OUT, EPI, 1>(A, lda, bg, ldb, m0, n0, m_lim, N, K, e, out, ldo);
  else if (TM > 2 && rows <= 128) qgemm_pp_tile<QT, OUT, EPI, 2>(A, lda, bg, ldb, m0, n0, m_lim, N, K, e, out, ldo);
  else if (TM > 3 && rows <= 192) qgemm_pp_tile<QT, OUT, EPI, 3>(A, lda, bg, ldb, m0, n0, m_lim, N, K, e, out, ldo);
  else qgemm_pp_tile<QT, OUT, EPI, TM>(A, lda, bg, ldb, m0, n0, m_lim, N, K, e, out, ldo);
}

template <int QT, int OUT, int EPI, int TM>
int launch_ragged_pp_tile(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                         int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr size_t smem = (2 * 64 * TM + 3 * 256) * 128;
  auto kern = qgemm_ragged_pp_kernel<QT, OUT, EPI, TM>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  kern<<<dim3(ragged_grid(M, N, rg.G, 64 * TM, 256)), 512, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, rg, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("ragged qgemm (ping-pong)");
}
template <int QT, int OUT, int EPI>
int launch_ragged_pp_epi(int tm, const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                         int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  if (tm == 2) return launch_ragged_pp_tile<QT, OUT, EPI, 2>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  if (tm == 3) return launch_ragged_pp_tile<QT, OUT, EPI, 3>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  return launch_ragged_pp_tile<QT, OUT, EPI, 4>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
}
// Ping-pong tiles of 64 * tm rows for a ragged product of more than 48 rows per group (0: 128 x 128 tiles).  The sizes are on the device:
// each group is taken to end 0.45 of a tile early, and to have at least one.  Where 128 x 128 tiles are about one per CU and K is short
// their two small workgroups per CU start and finish sooner.  int8 / e4m3, 8 to 64 groups of uneven sizes, weights from HBM, 128 x 128
// tiles -> these, us: 4000 rows, 16 groups, N 4096 over K 2048 74.7 -> 56.0 / 72.4 -> 57.6 (192 rows); 4656, 16, N 1472, K 2816
// 57.7 -> 36.0 (192); 7974, 32, N 1088, K 2048 47.4 -> 34.7 (256); 930, 8, N 1280, K 1152 12.5 against 13.0 (128).  The choice is
// within 2 % of the best of the three on average; what it misses lies in the sizes (2871 rows, 16, N 3392, K 2688 57.1, 45.3 with 256).
inline int ragged_pp_rows(int64_t M, int64_t N, int64_t K, int64_t G, bool big) {
  auto tile_rows = [&](int64_t rows) {
    const double per_group = static_cast<double>(M) / static_cast<double>(G * rows) + 0.45;
    return static_cast<double>(G) * (per_group > 1.0 ? per_group : 1.0);
  };
  if (!big && K < 1536 && tile_rows(128) * static_cast<double>((N + 127) / 128) <= 256.0) return 0;
  int best = 4;
  double best_us = 0;
  for (int tm = 4; tm >= 2; --tm) {
    const double us = pp_us(tm, tile_rows(64 * tm) * static_cast<double>((N + 255) / 256), K);
    if (tm == 4 || us < best_us) { best = tm; best_us = us; }
  }
  return best;
}

// The epilogue's rounding flags at compile time when every step rounds to bf16 (bf16 scales, bf16 result) or none
// does (f32 throughout), as the dense dispatch does; at run time otherwise.
template <int QT, int OUT>
int launch_ragged_pp(int tm, const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                     int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const bool all = ep.r0 && ep.r1 && ep.r2, none = !ep.r0 && !ep.r1 && !ep.r2;
  if (OUT == QWIX_BF16 && all) return launch_ragged_pp_epi<QT, OUT, 1>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  if (OUT == QWIX_F32 && none) return launch_ragged_pp_epi<QT, OUT, 0>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  return launch_ragged_pp_epi<QT, OUT, 2>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
}

template <int QT, int BM, int BN, int BK>
__global__ void __launch_bounds__(256)
    qgemm_ragged_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                        Ragged rg, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  int g, m0, m_lim, n0;
  const int kind = ragged_tile<BM, BN>(rg, M, N, &g, &m0, &m_lim, &n0);
  if (kind == 0) return;
  if (kind == 2) {
    if (ep.out_dtype == QWIX_BF16) zero_tile<BM, BN, uint16_t>(out, ldo, m0, m_lim, n0, N, 256);
    else zero_tile<BM, BN, uint32_t>(out, ldo, m0, m_lim, n0, N, 256);
    return;
  }
  const Epilogue e = group_epilogue(ep, rg, g);
  qgemm_tile<QT, BM, BN, BK>(A, lda, B + g * rg.b_group_stride, ldb, m0, n0, m_lim, N, K, e, out, ldo);
}

template <int QT, int BM, int BN, int WGM, int WGN, int OUT>
int launch_ragged_dma(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                      int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr size_t smem = 2 * (BM + BN) * 128;
  auto kern = qgemm_ragged_dma_kernel<QT, BM, BN, WGM, WGN, OUT>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  kern<<<dim3(ragged_grid(M, N, rg.G, BM, BN)), WGM * WGN * 64, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, rg, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("ragged qgemm (dma)");
}

// The one-tile-row body (deep prefetch of the weights into registers) under the ragged grid, for groups of
// a few dozen rows: tiles of 64 rows x 128 columns waste fewer rows at the ragged end of a group than 128-row
// tiles do, and such groups are bound by the streaming of their weight panels.
template <int QT, int OUT, int TM, int DEPTH, int NW>
__global__ void __launch_bounds__(64 * NW)
    qgemm_ragged_mid_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                            Ragged rg, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  constexpr int BM = 32 * TM, BN = 32 * NW;
  int g, m0, m_lim, n0;
  const int kind = ragged_tile<BM, BN>(rg, M, N, &g, &m0, &m_lim, &n0);
  if (kind == 0) return;
  using OutT = typename std::conditional<OUT == QWIX_BF16, uint16_t, uint32_t>::type;
  if (kind == 2) {
    zero_tile<BM, BN, OutT>(out, ldo, m0, m_lim, n0, N, 64 * NW);
    return;
  }
  const Epilogue e = group_epilogue(ep, rg, g);
  const int kshift = static_cast<int>((blockIdx.x * 5u) % static_cast<unsigned>(K / 128));
  qgemm_mid_tile<QT, OUT, 2, TM, DEPTH, NW>(A, lda, B + g * rg.b_group_stride, ldb, m0, n0, m_lim, N, K, e, out, ldo,
                                            kshift);
}

template <int QT, int OUT>
int launch_ragged_mid(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                      int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr int TM = 2, NW = 4, kDepth = 8;
  constexpr size_t smem = kDepth * 32 * TM * 128;  // 64 KB of activation stages (the epilogue needs 18 KB)
  auto kern = qgemm_ragged_mid_kernel<QT, OUT, TM, kDepth, NW>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  kern<<<dim3(ragged_grid(M, N, rg.G, 32 * TM, 32 * NW)), 64 * NW, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, rg, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("ragged qgemm (one tile row per 64 rows)");
}

template <int QT, int BM, int BN, int WGM, int WGN>
int dispatch_ragged_dma(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                        int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  if (ep.out_dtype == QWIX_I32) {
    if constexpr (QT == QWIX_INT8) return launch_ragged_dma<QT, BM, BN, WGM, WGN, QWIX_I32>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    return fail(QWIX_ERR_INVALID_ARGUMENT, "int32 output needs int8 operands");
  }
  if (ep.out_dtype == QWIX_BF16) return launch_ragged_dma<QT, BM, BN, WGM, WGN, QWIX_BF16>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  return launch_ragged_dma<QT, BM, BN, WGM, WGN, QWIX_F32>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
}

template <int QT>
int launch_ragged(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                  int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr int BM = 128, BN = 128, BK = 128;
  constexpr size_t smem = 2 * (BM + BN) * (BK + kPad);
  auto kern = qgemm_ragged_kernel<QT, BM, BN, BK>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  kern<<<dim3(ragged_grid(M, N, rg.G, BM, BN)), 256, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, rg, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("ragged qgemm");
}

// Ragged variant for a few rows per group (mixture-of-experts decode): blockIdx.y is the group, whose rows are
// found from the group sizes by every wavefront for itself; the workgroup streams that group's weight columns
// once per 16 rows.  blockIdx.y == G clears the rows that belong to no group.
template <int QT, int NT, int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
    qgemm_ragged_skinny_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                               Ragged rg, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  const int g = blockIdx.y, lane = threadIdx.x & 63;
  const int n_base = blockIdx.x * (16 * NT);
  long long before = 0;
  for (int i = lane; i < g; i += 64) before += max(rg.group_sizes[i], 0);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) before += __shfl_xor(before, m, 64);
  const int start = static_cast<int>(min(before, static_cast<long long>(M)));
  if (g == rg.G) {  // rows past the last group: zeros
    const int cols = min(16 * NT, N - n_base);
    for (int idx = threadIdx.x; idx < (M - start) * cols; idx += WAVES * 64) {
      const int64_t at = static_cast<int64_t>(start + idx / cols) * ldo + n_base + idx % cols;
      if (ep.out_dtype == QWIX_BF16) reinterpret_cast<uint16_t*>(out)[at] = 0;
      else reinterpret_cast<uint32_t*>(out)[at] = 0;
    }
    return;
  }
  const int end = static_cast<int>(min(before + max(rg.group_sizes[g], 0), static_cast<long long>(M)));
  const Epilogue e = group_epilogue(ep, rg, g);
  const uint8_t* bg = B + g * rg.b_group_stride;
  for (int row0 = start; row0 < end; row0 += 16) {  // the trip count is the same for the whole workgroup
    skinny_block<QT, NT, WAVES>(A, lda, bg, ldb, row0, end, n_base, N, K, e, out, ldo);
    __syncthreads();  // the partial sums in LDS are reused by the next pass
  }
}

template <int QT>
int launch_ragged_skinny(const void* a, int64_t lda, const void* b, int64_t ldb, const Ragged& rg, int64_t M, int64_t N,
                         int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const unsigned gy = static_cast<unsigned>(rg.G + 1);
  // Small workgroups: 4 wavefronts, and the fewer rows a group has, the narrower the column group (the
  // activation fragment is re-read per column group, which costs as much as the weights once a group has 16
  // rows).  Measured at 64 groups x 4 rows, K 2048, N 4096, in GB/s of weights: 16 wavefronts x 64 columns
  // 4260, 8 x 32 4700, 4 x 64 4680, 4 x 32 4810, 4 x 16 5120, 2 x 16 5060, 1 x 16 4980.
  constexpr int kWaves = 4;
#define QWIX_RSKINNY(NTT)                                                                                          \
  qgemm_ragged_skinny_kernel<QT, NTT, kWaves><<<dim3(static_cast<unsigned>((N + 16 * NTT - 1) / (16 * NTT)), gy), \
                                                kWaves * 64, 0, st>>>(static_cast<const uint8_t*>(a), lda,          \
                                                                      static_cast<const uint8_t*>(b), ldb, rg,        \
                                                                      static_cast<int>(M), static_cast<int>(N),      \
                                                                      static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo)
  if (M <= 4 * static_cast<int64_t>(rg.G))
    QWIX_RSKINNY(1);
  else if (M <= 8 * static_cast<int64_t>(rg.G))
    QWIX_RSKINNY(2);
  else
    QWIX_RSKINNY(4);
#undef QWIX_RSKINNY
  return check_launch("ragged qgemm (skinny)");
}

}  // namespace
}  // namespace qwix

using namespace qwix;

extern "C" int qwix_hip_qgemm_ragged(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t b_group_stride,
                                     int qtype, int64_t M, int64_t N, int64_t K, const int32_t* group_sizes,
                                     int64_t G, const void* sa, int sa_dtype, const void* sb, int sb_dtype,
                                     int64_t sb_group_stride, int acc_dtype, void* out, int out_dtype, int64_t ldo,
                                     void* stream) {
  if (const int rc = check_gemm_args(a, lda, b, ldb, qtype, M, N, K, sa, sa_dtype, sb, sb_dtype, acc_dtype, out,
                                     out_dtype, ldo))
    return rc;
  if (!group_sizes || G <= 0 || G > 65536)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "ragged qgemm needs 1..65536 group sizes (G=%lld)", (long long)G);
  if (b_group_stride % 16 || b_group_stride < 0 || sb_group_stride < 0 || (sb_group_stride % 4 != 0 && N % 4 == 0))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad group strides (b: %lld bytes, sb: %lld elements)",
                (long long)b_group_stride, (long long)sb_group_stride);
  if (M * lda >= (int64_t{1} << 31) || N * ldb >= (int64_t{1} << 31) ||
      (M / 128 + G + 1) * ((N + 127) / 128) >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "ragged qgemm: operand too large for 32-bit offsets (M*lda=%lld N*ldb=%lld)",
                (long long)(M * lda), (long long)(N * ldb));
  const Epilogue ep = make_epilogue(qtype, sa, sa_dtype, sb, sb_dtype, acc_dtype, nullptr, nullptr, out_dtype);
  const Ragged rg{group_sizes, static_cast<int>(G), 0, b_group_stride, sb_group_stride};
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (K % 128 == 0 && M <= 16 * G && G + 1 <= 65535 && 64 * ldb < (int64_t{1} << 31)) {
    // at most 16 rows per group on average (decode): stream every group's weight once instead of tiling
    // (measured, 64 groups x 2048 x 4096: 146 -> 119 us; at 32 rows per group a second pass over the weights loses)
    if (qtype == QWIX_INT8) return launch_ragged_skinny<QWIX_INT8>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    return launch_ragged_skinny<QWIX_E4M3>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  }
  if (K % 128 == 0) {
    const bool big = M / G >= 768 && ((M + 255) / 256) * ((N + 255) / 256) >= 192;
    const int tm = ragged_pp_rows(M, N, K, G, big);
    // 17 to 48 rows per group on average: 64-row tiles with the deep weight prefetch (64 groups x 32 rows, K 2048,
    // N 4096: 131.7 against 144.8 us; from 64 rows per group on the 128-row tile wins again, 174 against 160 us)
    if (M <= 48 * G && out_dtype != QWIX_I32 &&
        (M / 64 + G + 1) * ((N + 127) / 128) < (int64_t{1} << 31)) {
      if (qtype == QWIX_INT8) {
        if (out_dtype == QWIX_BF16) return launch_ragged_mid<QWIX_INT8, QWIX_BF16>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
        return launch_ragged_mid<QWIX_INT8, QWIX_F32>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
      }
      if (out_dtype == QWIX_BF16) return launch_ragged_mid<QWIX_E4M3, QWIX_BF16>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
      return launch_ragged_mid<QWIX_E4M3, QWIX_F32>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    }
    if (tm && K >= 256 && out_dtype != QWIX_I32) {
      if (qtype == QWIX_INT8) {
        if (out_dtype == QWIX_BF16) return launch_ragged_pp<QWIX_INT8, QWIX_BF16>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
        return launch_ragged_pp<QWIX_INT8, QWIX_F32>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
      }
      if (out_dtype == QWIX_BF16) return launch_ragged_pp<QWIX_E4M3, QWIX_BF16>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
      return launch_ragged_pp<QWIX_E4M3, QWIX_F32>(tm, a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    }
    if (qtype == QWIX_INT8) {
      if (big) return dispatch_ragged_dma<QWIX_INT8, 256, 256, 2, 4>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
      return dispatch_ragged_dma<QWIX_INT8, 128, 128, 2, 2>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    }
    if (big) return dispatch_ragged_dma<QWIX_E4M3, 256, 256, 2, 4>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
    return dispatch_ragged_dma<QWIX_E4M3, 128, 128, 2, 2>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  }
  if (qtype == QWIX_INT8) return launch_ragged<QWIX_INT8>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
  return launch_ragged<QWIX_E4M3>(a, lda, b, ldb, rg, M, N, K, ep, out, ldo, st);
}
