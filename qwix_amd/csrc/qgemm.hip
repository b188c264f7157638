// Quantized GEMMs on the gfx950 matrix cores (MFMA), dequantize-on-output.
//
//   out[m,n] = epilogue( sum_k a[m,k] * b[n,k] )      a: (M,K), b: (N,K), both K-contiguous
//
// Kernels around the tile bodies of qgemm_tiles.h: dense (one tile per workgroup, XCD-aware tile order), batched
// (blockIdx.y selects the problem), a skinny kernel for M <= 32 that streams the weights once, and K splits.
#include <cstdlib>
#include <type_traits>

#include "common.h"
#include "qgemm_strips.h"
#include "qgemm_tiles.h"

namespace qwix {
namespace {

template <int QT, int BM, int BN, int BK>
__global__ void __launch_bounds__(256)
    qgemm_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                 int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  int tile_m, tile_n;
  tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, &tile_m, &tile_n);
  qgemm_tile<QT, BM, BN, BK>(A, lda, B, ldb, tile_m * BM, tile_n * BN, M, N, K, ep, out, ldo);
}

template <int QT, int BM, int BN, int WGM, int WGN, int OUT, int EPI, int NST = 2>
__global__ void __launch_bounds__(WGM * WGN * 64)
    qgemm_dma_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                     int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  int tile_m, tile_n;
  tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, &tile_m, &tile_n);
  qgemm_dma_tile<QT, BM, BN, WGM, WGN, OUT, EPI, NST>(A, lda, B, ldb, tile_m * BM, tile_n * BN, M, N, K, ep, out, ldo);
}

template <int QT, int BM, int BN, int WGM, int WGN, int OUT, int EPI, int NST = 2>
int launch_dma(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
               const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr size_t smem = NST * (BM + BN) * 128;
  auto kern = qgemm_dma_kernel<QT, BM, BN, WGM, WGN, OUT, EPI, NST>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  kern<<<dim3(static_cast<unsigned>(tiles)), WGM * WGN * 64, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("qgemm (dma)");
}

// Picks the epilogue specialisation: (bf16 out, all-bf16 rounding), (f32 out, no rounding), raw int32,
// or the run-time-flag version for mixed scale dtypes.
template <int QT, int BM, int BN, int WGM, int WGN, int NST = 2>
int dispatch_dma(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                 const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const bool all = ep.r0 && ep.r1 && ep.r2, none = !ep.r0 && !ep.r1 && !ep.r2;
  if (ep.out_dtype == QWIX_I32) {
    if constexpr (QT == QWIX_INT8) return launch_dma<QT, BM, BN, WGM, WGN, QWIX_I32, 0, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    return fail(QWIX_ERR_INVALID_ARGUMENT, "int32 output needs int8 operands");
  }
  if (ep.zu != nullptr) {
    if constexpr (QT == QWIX_INT8) {
      if (ep.out_dtype == QWIX_BF16) return launch_dma<QT, BM, BN, WGM, WGN, QWIX_BF16, 3, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      return launch_dma<QT, BM, BN, WGM, WGN, QWIX_F32, 3, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    }
    return fail(QWIX_ERR_UNSUPPORTED, "zero-point correction needs int8 operands");
  }
  if (ep.out_dtype == QWIX_BF16) {
    if (all) return launch_dma<QT, BM, BN, WGM, WGN, QWIX_BF16, 1, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    return launch_dma<QT, BM, BN, WGM, WGN, QWIX_BF16, 2, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  }
  if (none) return launch_dma<QT, BM, BN, WGM, WGN, QWIX_F32, 0, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  return launch_dma<QT, BM, BN, WGM, WGN, QWIX_F32, 2, NST>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
}

template <int QT, int OUT, int EPI, int TM, int DEPTH, int NW>
__global__ void __launch_bounds__(64 * NW)
    qgemm_mid_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb, int M,
                     int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo, int kmul) {
  const int kshift = static_cast<int>((blockIdx.x * static_cast<unsigned>(kmul)) % static_cast<unsigned>(K / 128));
  qgemm_mid_tile<QT, OUT, EPI, TM, DEPTH, NW>(A, lda, B, ldb, blockIdx.y * (32 * TM), blockIdx.x * (32 * NW), M, N, K,
                                              ep, out, ldo, kshift);
}

// ------------------------------------------------------------------------------------------------
// The same one tile row when N is so small that 32-column workgroups do not fill the chip (N up to 8192): the
// KW wavefronts of a workgroup share its 32 columns and split K instead, wavefront w taking slabs w, w + KW, ...
// Activations and weights both go from global memory straight into registers, in the same permuted K order
// (lane half h holds bytes 64 h .. 64 h + 63 of a row's 128-byte slab, for its activation rows as for its
// weight column), so the main loop touches no LDS and has no barrier: every wavefront runs its own pipeline
// of DEPTH register sets, waiting only on its own loads (explicit vmcnt, loads issued as asm as above).  At the
// end the partial accumulators meet in LDS, and wavefront i adds up and stores the i-th block of 32 rows.
// int32 partials add exactly; for e4m3 the f32 sums are those of K / (128 KW) slabs each, added in wavefront order.
template <int QT, int OUT, int EPI, int TM, int DEPTH, int KW>
__global__ void __launch_bounds__(64 * KW)
    qgemm_ksplit_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb, int M,
                        int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo, int kmul) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  constexpr int BK = 128;
  constexpr int NK = IS_INT ? 4 : 2;  // MFMAs per slab and 32-row block
  constexpr int G = 4 * TM + 4;       // loads per slab and lane
  static_assert((DEPTH - 2) * G <= 63, "vmcnt is a 6-bit counter");
  static_assert(DEPTH >= 3 && DEPTH <= 8 && TM <= KW, "the waits and the final reduction list these cases");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 32;

  using AccT = typename std::conditional<IS_INT, v16i, v16f>::type;
  using FragT = typename std::conditional<IS_INT, v4i, v8i>::type;
  AccT acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0;
  float sav[TM];
  float sbv[1][4][4];
  fetch_scales<OUT, TM, 1>(ep, 0, n0, M, N, lane, sav, sbv);  // oldest loads: done before any slab is used

  const int hx = lane >> 5;
  uint32_t aoff[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    aoff[i] = static_cast<uint32_t>(min(i * 32 + (lane & 31), M - 1)) * static_cast<uint32_t>(lda) + hx * 64;
  const uint32_t boff = static_cast<uint32_t>(min(n0 + (lane & 31), N - 1)) * static_cast<uint32_t>(ldb) + hx * 64;
  v4i areg[DEPTH][TM][4], breg[DEPTH][4];
  const int KT = K / BK;
  const int kshift = static_cast<int>((blockIdx.x * static_cast<unsigned>(kmul)) % static_cast<unsigned>(KT));
  auto issue_group = [&](int kt, int st) {  // 4 TM + 4 register loads per lane, not tracked by the compiler
    kt += kshift;
    if (kt >= KT) kt -= KT;
    const uint8_t* ga = A + kt * BK;
    const uint8_t* gb = B + kt * BK;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      asm volatile("global_load_dwordx4 %0, %4, %5\n\t"
                   "global_load_dwordx4 %1, %4, %5 offset:16\n\t"
                   "global_load_dwordx4 %2, %4, %5 offset:32\n\t"
                   "global_load_dwordx4 %3, %4, %5 offset:48"
                   : "=&v"(areg[st][i][0]), "=&v"(areg[st][i][1]), "=&v"(areg[st][i][2]), "=&v"(areg[st][i][3])
                   : "v"(aoff[i]), "s"(ga)
                   : "memory");
    asm volatile("global_load_dwordx4 %0, %4, %5\n\t"
                 "global_load_dwordx4 %1, %4, %5 offset:16\n\t"
                 "global_load_dwordx4 %2, %4, %5 offset:32\n\t"
                 "global_load_dwordx4 %3, %4, %5 offset:48"
                 : "=&v"(breg[st][0]), "=&v"(breg[st][1]), "=&v"(breg[st][2]), "=&v"(breg[st][3])
                 : "v"(boff), "s"(gb)
                 : "memory");
  };

  const int mine = KT > wave ? (KT - wave + KW - 1) / KW : 0;  // slabs of this wavefront: wave + j * KW
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < mine) issue_group(wave + d * KW, d);
  for (int j0 = 0; j0 < mine; j0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int j = j0 + d;
      if (j < mine) {  // the same for the whole wavefront
        const int rem = mine - 1 - j;  // the groups after j (at most DEPTH - 2 of them) may stay in flight
        __builtin_amdgcn_sched_barrier(0);
        switch (rem < DEPTH - 2 ? rem : DEPTH - 2) {
          case 0: wait_vmcnt<0>(); break;
          case 1: wait_vmcnt<G>(); break;
          case 2: wait_vmcnt<(2 * G < 63 ? 2 * G : 63)>(); break;
          case 3: wait_vmcnt<(3 * G < 63 ? 3 * G : 63)>(); break;
          case 4: wait_vmcnt<(4 * G < 63 ? 4 * G : 63)>(); break;
          case 5: wait_vmcnt<(5 * G < 63 ? 5 * G : 63)>(); break;
          default: wait_vmcnt<(6 * G < 63 ? 6 * G : 63)>(); break;
        }
        __builtin_amdgcn_sched_barrier(0);
        // pin the set that has just landed: nothing may read or copy it in front of the wait above
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          asm volatile("" : "+v"(breg[d][r]));
#pragma unroll
          for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(areg[d][i][r]));
        }
        // set (d - 1) was multiplied one slab ago: refill it DEPTH - 1 slabs ahead
        if (j + DEPTH - 1 < mine) issue_group(wave + (j + DEPTH - 1) * KW, (d + DEPTH - 1) % DEPTH);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
          FragT fb;
          if constexpr (IS_INT) {
            fb = breg[d][ks];
          } else {
            const v4i lo = breg[d][2 * ks], hi = breg[d][2 * ks + 1];
            fb = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          }
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            if constexpr (IS_INT) {
              acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, areg[d][i][ks], acc[i], 0, 0, 0);
            } else {
              const v4i lo = areg[d][i][2 * ks], hi = areg[d][i][2 * ks + 1];
              const v8i fa = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
              acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb, fa, acc[i], 0, 0, 0, 0, 0, 0);
            }
          }
        }
      }
    }
  }
  // partial accumulators -> LDS (behind the 20 KB that the epilogue stages through), [wave][block][register][lane]
  constexpr int kStage = 20480;
  using Word = typename std::conditional<IS_INT, int, float>::type;
  Word* part = reinterpret_cast<Word*>(smem + kStage);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[((wave * TM + i) * 16 + r) * 64 + lane] = acc[i][r];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (wave == i) {  // wavefront i finishes block i
      AccT total[1][1];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        Word t = part[((0 * TM + i) * 16 + r) * 64 + lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) t += part[((w * TM + i) * 16 + r) * 64 + lane];
        total[0][0][r] = t;
      }
      const float sav1[1] = {sav[i]};
      staged_epilogue<OUT, EPI, 1, 1, KW, kStage, false>(total, sav1, sbv, ep, i * 32, n0, M, N, out, ldo, smem, wave, lane);
    }
  }
}

template <int QT, int OUT, int EPI = 2>
int launch_mid(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
               const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  // LDS: kDepth stages of activations, and at least the 18 KB the epilogue stages through
#define QWIX_MID(TMM, NWW) QWIX_MID_D(TMM, NWW, ((4 * TMM / NWW + 4) * 6 <= 63 ? 8 : 6))
#define QWIX_MID_D(TMM, NWW, DD)                                                                                  \
  {                                                                                                               \
    constexpr int kDepth = DD; /* the groups in flight must stay under vmcnt's 63 */                               \
    constexpr size_t smem = kDepth * 32 * TMM * 128 > 20480 ? kDepth * 32 * TMM * 128 : 20480;                     \
    auto kern = qgemm_mid_kernel<QT, OUT, EPI, TMM, kDepth, NWW>;                                                 \
    static LdsGrant granted;                                                                                      \
    if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;                        \
    kern<<<dim3(static_cast<unsigned>((N + 32 * NWW - 1) / (32 * NWW)),                                           \
                static_cast<unsigned>((M + 32 * TMM - 1) / (32 * TMM))), 64 * NWW, smem, st>>>(                    \
        static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),            \
        static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo, kmul);                     \
  }
  // Workgroups of 2 wavefronts (64 columns) for up to 32 rows, and for 64 rows while 128-column workgroups
  // would leave CUs without one: twice the workgroups, twice the CUs that pull weights.  Measured, weights
  // from HBM, 2 / 4 wavefronts, K 4096, N 14336: 32 rows 17.5 / 23.4 us, 64 rows 20.3 / 26.4 us; K 8192,
  // N 8192: 23.9 / 37.4 and 30.5 / 42.8 us; K 8192, N 28672: 51.8 / 54.2 and 62.6 / 55.0 us.
  const bool narrow = (N + 127) / 128 < 192;
  // Up to N 8192 and 64 rows a workgroup is a single wavefront (32 columns): 10 to 15 % less again (64 rows,
  // K 4096, N 4096 / 6144: 16.6 / 16.3 against 19.6 / 18.7 us; K 14336, N 4096: 44.1 against 52.6 us).
  // Workgroup b starts at slab 5 b (mod K / 128) and wraps around: with a power-of-two row pitch all workgroups
  // would otherwise ask the same few memory channels for the same K offset of their rows at the same time
  // (K 8192, N 28672, 64 rows: 49.3 against 54.9 us; K 4096, N 14336, 32 rows: 16.2 against 17.6 us).  Integer
  // sums do not depend on the order; e4m3 sums are then added in an order that depends on the column block.
  constexpr int kmul = 5;
  // N up to 8192: four wavefronts split K over the same 32 columns (32 rows, K 4096, N 6144: 12.3 against 14.2 us
  // for single-wavefront workgroups, K 8192, N 8192: 19.5 against 22.0 us; 64 rows: 5 % less).
  if (M <= 64 && (N + 63) / 64 <= 128 && K >= 1024) {
#define QWIX_KSPLIT(TMM, DD)                                                                                      \
  {                                                                                                               \
    constexpr int kKW = 4;                                                                                        \
    constexpr size_t smem = 20480 + kKW * TMM * 4096;                                                             \
    auto kern = qgemm_ksplit_kernel<QT, OUT, EPI, TMM, DD, kKW>;                                                  \
    static LdsGrant granted;                                                                                      \
    if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;                        \
    kern<<<dim3(static_cast<unsigned>((N + 31) / 32)), 64 * kKW, smem, st>>>(                                     \
        static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),            \
        static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo, kmul);                     \
  }
    if (M <= 32) QWIX_KSPLIT(1, 6)
    else QWIX_KSPLIT(2, 4)
#undef QWIX_KSPLIT
  } else if (M <= 64 && (N + 63) / 64 <= 128) {
    if (M <= 32) QWIX_MID(1, 1)
    else QWIX_MID(2, 1)
  } else if (M <= 32) {
    QWIX_MID(1, 2)
  } else if (M > 128) {
    QWIX_MID_D(4, 2, 4)  // two tile rows side by side: four stages, 64 KB, two workgroups per CU
  } else if (M > 64) {
    if ((N + 63) / 64 <= 256) QWIX_MID(4, 2)
    else QWIX_MID(4, 4)
  } else {
    if (narrow) QWIX_MID(2, 2)
    else QWIX_MID(2, 4)
  }
#undef QWIX_MID
#undef QWIX_MID_D
  return check_launch("qgemm (one tile row)");
}

// Rows of the ping-pong tiles / 64 of a dense product (0: 128 x 128 tiles or less).  Up to one 128 x 128 tile per CU those have three slab
// stages and start sooner (1024 x 4096 over K 4096 24.8 against 27.8 us with 128 rows, 1500 x 1500 over K 8192 41.3 against 51.1), and
// up to two per CU they overlap a short K's start with the other tile's end (4096 x 2048 over K 1024, e4m3 15.0 against 17.4).  Beyond:
// int8 / e4m3, weights from HBM, 128 x 128 or (fifth on) 256 x 256 tiles -> these: 2048 x 4096 over K 4096 39.5 -> 35.9 / 36.3 -> 34.7
// (128 rows), 512 x 14336 over K 4096 43.6 -> 38.8 / 44.5 -> 39.0 (128), 5224 x 1776 over K 3584 53.7 -> 37.3 (192), 2186 x 4992 over
// K 9984 168 -> 100 (192); 3000 x 4096 over K 4096 50.6 -> 48.4 / 49.4 -> 44.6 (192), 2304 x 8192 over K 512 28.3 -> 23.9 / 32.7 -> 27.1.
inline int pp_rows(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128), tiles_n = (N + 255) / 256;
  const bool big = ((M + 255) / 256) * tiles_n >= 192;
  if (!big && (tiles128 <= 256 || (tiles128 <= 512 && K < 1536))) return 0;
  int best = 4;
  double best_us = 0;
  for (int tm = 4; tm >= 2; --tm) {
    const double us = pp_us(tm, static_cast<double>((M + 64 * tm - 1) / (64 * tm) * tiles_n), K);
    if (tm == 4 || us < best_us) { best = tm; best_us = us; }
  }
  return best;
}

template <int QT, int OUT, int EPI, int TM>
__global__ void __launch_bounds__(512)
    qgemm_pp_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb, int M,
                    int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  constexpr int BM = 64 * TM;
  int tile_m, tile_n;
  tile_coords((M + BM - 1) / BM, (N + 255) / 256, &tile_m, &tile_n);
  qgemm_pp_tile<QT, OUT, EPI, TM>(A, lda, B, ldb, tile_m * BM, tile_n * 256, M, N, K, ep, out, ldo);
}

template <int QT, int OUT, int EPI, int TM>
int launch_pp_tile(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                   const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr int BM = 64 * TM;
  constexpr size_t smem = (2 * BM + 3 * 256) * 128;
  auto kern = qgemm_pp_kernel<QT, OUT, EPI, TM>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + 255) / 256);
  kern<<<dim3(static_cast<unsigned>(tiles)), 512, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("qgemm (ping-pong)");
}
template <int QT, int OUT, int EPI>
int launch_pp(int tm, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
              const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  if (tm == 2) return launch_pp_tile<QT, OUT, EPI, 2>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  if (tm == 3) return launch_pp_tile<QT, OUT, EPI, 3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  return launch_pp_tile<QT, OUT, EPI, 4>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
}

template <int QT>
int dispatch_pp(int tm, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const bool all = ep.r0 && ep.r1 && ep.r2, none = !ep.r0 && !ep.r1 && !ep.r2;
  if (ep.zu != nullptr) {
    if constexpr (QT == QWIX_INT8) {
      if (ep.out_dtype == QWIX_BF16 && all) return launch_pp<QT, QWIX_BF16, 4>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      if (ep.out_dtype == QWIX_BF16) return launch_pp<QT, QWIX_BF16, 3>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      return launch_pp<QT, QWIX_F32, 3>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    }
    return fail(QWIX_ERR_UNSUPPORTED, "zero-point correction needs int8 operands");
  }
  if (ep.out_dtype == QWIX_BF16) {
    if (all) return launch_pp<QT, QWIX_BF16, 1>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    return launch_pp<QT, QWIX_BF16, 2>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  }
  if (none) return launch_pp<QT, QWIX_F32, 0>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  return launch_pp<QT, QWIX_F32, 2>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
}

template <int QT, int BM, int BN, int BK>
int launch_qgemm(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                 const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr size_t smem = 2 * (BM + BN) * (BK + kPad);
  auto kern = qgemm_kernel<QT, BM, BN, BK>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  kern<<<dim3(static_cast<unsigned>(tiles)), 256, smem, st>>>(static_cast<const uint8_t*>(a), lda,
                                                              static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),
                                                              static_cast<int>(N), static_cast<int>(K), ep,
                                                              static_cast<uint8_t*>(out), ldo);
  return check_launch("qgemm");
}

// ------------------------------------------------------------------------------------------------
// Batched GEMM: blockIdx.y selects one of `batch` independent problems of the same shape (the batch
// axes of dot_general); operands, scale vectors and outputs of consecutive problems are a fixed
// stride apart.  Same tile bodies as the dense kernels.
struct Batched {
  int64_t a_stride, b_stride;    // bytes
  int64_t sa_stride, sb_stride;  // elements (0: the vector is shared by all problems)
  int64_t out_stride;            // elements
};

__device__ __forceinline__ Epilogue batch_epilogue(const Epilogue& ep, const Batched& bs, int z) {
  Epilogue e = ep;
  if (ep.sa != nullptr)
    e.sa = static_cast<const uint8_t*>(ep.sa) + z * bs.sa_stride * (ep.sa_dtype == QWIX_BF16 ? 2 : 4);
  if (ep.sb != nullptr)
    e.sb = static_cast<const uint8_t*>(ep.sb) + z * bs.sb_stride * (ep.sb_dtype == QWIX_BF16 ? 2 : 4);
  return e;
}

template <int QT, int BM, int BN, int WGM, int WGN, int OUT>
__global__ void __launch_bounds__(WGM * WGN * 64)
    qgemm_batched_dma_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                             Batched bs, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  const int z = blockIdx.y;
  int tile_m, tile_n;
  tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, &tile_m, &tile_n);
  const Epilogue e = batch_epilogue(ep, bs, z);
  constexpr int ES = OUT == QWIX_BF16 ? 2 : 4;
  qgemm_dma_tile<QT, BM, BN, WGM, WGN, OUT, (OUT == QWIX_I32 ? 0 : 2)>(
      A + z * bs.a_stride, lda, B + z * bs.b_stride, ldb, tile_m * BM, tile_n * BN, M, N, K, e,
      out + z * bs.out_stride * ES, ldo);
}

template <int QT, int BM, int BN, int BK>
__global__ void __launch_bounds__(256)
    qgemm_batched_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                         Batched bs, int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  const int z = blockIdx.y;
  int tile_m, tile_n;
  tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, &tile_m, &tile_n);
  const Epilogue e = batch_epilogue(ep, bs, z);
  const int es = ep.out_dtype == QWIX_BF16 ? 2 : 4;
  qgemm_tile<QT, BM, BN, BK>(A + z * bs.a_stride, lda, B + z * bs.b_stride, ldb, tile_m * BM, tile_n * BN, M, N, K, e,
                             out + z * bs.out_stride * es, ldo);
}

template <int QT, int OUT>
int launch_batched_dma(const void* a, int64_t lda, const void* b, int64_t ldb, const Batched& bs, int64_t batch,
                       int64_t M, int64_t N, int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  constexpr int BM = 128, BN = 128;
  constexpr size_t kStage = (BM + BN) * 128;
  constexpr size_t kStaging = 4 * 32 * (64 * (OUT == QWIX_BF16 ? 2 : 4) + 16);  // epilogue: 4 wavefronts x 32 padded rows
  // A single slab (K = 128, e.g. the head dimension of attention scores) never touches the second stage:
  // half the LDS lets more workgroups share a CU, which is what hides the latency of such short tiles.
  const size_t smem = K == 128 ? (kStage > kStaging ? kStage : kStaging) : 2 * kStage;
  auto kern = qgemm_batched_dma_kernel<QT, BM, BN, 2, 2, OUT>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  kern<<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batch)), 256, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, bs, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("batched qgemm (dma)");
}

template <int QT>
int launch_batched(const void* a, int64_t lda, const void* b, int64_t ldb, const Batched& bs, int64_t batch,
                   int64_t M, int64_t N, int64_t K, const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  if (K % 128 == 0) {
    if (ep.out_dtype == QWIX_I32) {
      if constexpr (QT == QWIX_INT8) return launch_batched_dma<QT, QWIX_I32>(a, lda, b, ldb, bs, batch, M, N, K, ep, out, ldo, st);
      return fail(QWIX_ERR_INVALID_ARGUMENT, "int32 output needs int8 operands");
    }
    if (ep.out_dtype == QWIX_BF16) return launch_batched_dma<QT, QWIX_BF16>(a, lda, b, ldb, bs, batch, M, N, K, ep, out, ldo, st);
    return launch_batched_dma<QT, QWIX_F32>(a, lda, b, ldb, bs, batch, M, N, K, ep, out, ldo, st);
  }
  constexpr int BM = 128, BN = 128, BK = 128;
  constexpr size_t smem = 2 * (BM + BN) * (BK + kPad);
  auto kern = qgemm_batched_kernel<QT, BM, BN, BK>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  kern<<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batch)), 256, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, bs, static_cast<int>(M),
      static_cast<int>(N), static_cast<int>(K), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("batched qgemm");
}

}  // namespace
}  // namespace qwix

using namespace qwix;

namespace qwix {
namespace {

template <int QT, int NT>
__global__ void __launch_bounds__(kSkinnyWaves * 64)
    qgemm_skinny_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb, int M,
                        int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  skinny_block<QT, NT>(A, lda, B, ldb, blockIdx.y * 16, M, blockIdx.x * (16 * NT), N, K, ep, out, ldo);
}

// The same block with smaller workgroups, for weights of hundreds of megabytes (an output projection over a
// large vocabulary): once there are several rounds of workgroups per CU, small ones overlap each other's load,
// reduce and store phases (one row, K 4096, N 131072: 4.9 -> 6.0 TB/s with 4 wavefronts x 16 columns).  Taken for
// up to 4 rows only: with 16 rows the narrow column groups re-read the activation fragment too often (8 wavefronts
// x 32 columns: between -8 % and +10 % depending on K), and at decode sizes of tens of megabytes, where all
// workgroups fit the chip at once, the 16-wavefront shape stays ahead (58.7 MB: 4.1 TB/s against 3.2 - 3.9).
template <int QT, int NT, int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
    qgemm_skinny_small_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                              int M, int N, int K, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  skinny_block<QT, NT, WAVES>(A, lda, B, ldb, blockIdx.y * 16, M, blockIdx.x * (16 * NT), N, K, ep, out, ldo);
}

template <int QT>
int launch_skinny(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                  const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const unsigned gy = static_cast<unsigned>((M + 15) / 16);
  if (N * K >= (int64_t{192} << 20) && M <= 4) {
#define QWIX_SKINNY_SMALL(NTT, WVV)                                                                                \
  qgemm_skinny_small_kernel<QT, NTT, WVV><<<dim3(static_cast<unsigned>((N + 16 * NTT - 1) / (16 * NTT)), gy), WVV * 64, \
                                            0, st>>>(static_cast<const uint8_t*>(a), lda,                             \
                                                     static_cast<const uint8_t*>(b), ldb, static_cast<int>(M),        \
                                                     static_cast<int>(N), static_cast<int>(K), ep,                     \
                                                     static_cast<uint8_t*>(out), ldo)
    QWIX_SKINNY_SMALL(1, 4);
#undef QWIX_SKINNY_SMALL
    return check_launch("qgemm (skinny)");
  }
#define QWIX_SKINNY(NTT)                                                                                         \
  qgemm_skinny_kernel<QT, NTT><<<dim3(static_cast<unsigned>((N + 16 * NTT - 1) / (16 * NTT)), gy), kSkinnyWaves * 64, \
                                 0, st>>>(static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, \
                                          static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), ep,       \
                                          static_cast<uint8_t*>(out), ldo)
  // wider column groups reuse the activation fragments; narrower ones keep every CU busy
  if (N >= 192 * 64)
    QWIX_SKINNY(4);
  else if (N >= 192 * 32)
    QWIX_SKINNY(2);
  else
    QWIX_SKINNY(1);
#undef QWIX_SKINNY
  return check_launch("qgemm (skinny)");
}

// ------------------------------------------------------------------------------------------------
// Decode with the activation quantization folded in (int8, M <= 32 per call): the float activations are
// what the kernel reads.  Every workgroup keeps its 16 rows in registers (the 16 wavefronts split K as in
// the skinny kernel, a lane holds the 32 consecutive k of one row that its MFMA operand needs), finds the
// rows' absmax (lanes of a row by shuffle, wavefronts through LDS; a maximum does not depend on the order),
// derives the scale exactly as the stand-alone quantize kernel does, quantizes its registers and goes on
// as the skinny kernel.  The quantized values and scales are bit-identical to quantize-then-multiply; they
// are recomputed by every workgroup from L2 (16 x K activations against 16 * NT x K weights), which is
// cheaper than a kernel launch of its own as long as K is short.  KB: 128-wide K blocks per wavefront
// (K <= 2048 * KB; only KB = 1 is instantiated).
template <typename D, int NT, int KB>
__global__ void __launch_bounds__(kSkinnyWaves * 64)
    qgemm_skinny_fused_kernel(const uint8_t* __restrict__ X, int64_t ldx, const uint8_t* __restrict__ B, int64_t ldb,
                              int M, int N, int K, int relu, Epilogue ep, uint8_t* __restrict__ out, int64_t ldo) {
  constexpr int ES = D::kTag == QWIX_BF16 ? 2 : 4;   // bytes per activation
  constexpr int XV = 32 * ES / 16;                    // 16-byte loads per lane and K block (32 elements)
  __shared__ v4i red[kSkinnyWaves][NT][64];
  __shared__ float rowmax[kSkinnyWaves][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const int n_base = blockIdx.x * (16 * NT), row0 = blockIdx.y * 16;
  const int nblk = K / 128;
  const int kb0 = wave * KB, kb1 = min(nblk, kb0 + KB);  // nblk <= 16 * KB

  const uint8_t* x_base = X + static_cast<int64_t>(row0) * ldx * ES;
  const uint8_t* b_base = B + static_cast<int64_t>(n_base) * ldb;
  const uint32_t x_off = static_cast<uint32_t>(min(col, M - 1 - row0)) * static_cast<uint32_t>(ldx * ES) + kq * 32 * ES;
  uint32_t b_off[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    b_off[t] = static_cast<uint32_t>(min(t * 16 + col, N - 1 - n_base)) * static_cast<uint32_t>(ldb) + kq * 32;

  // ---- this lane's activations and weights for all of its K blocks
  uint4 xr[KB][XV];
  v4i w[KB][NT][2];
#pragma unroll
  for (int j = 0; j < KB; ++j) {
    const int kb = kb0 + j;
#pragma unroll
    for (int v = 0; v < XV; ++v) xr[j][v] = make_uint4(0, 0, 0, 0);
    if (kb < kb1) {
      const uint8_t* xp = x_base + static_cast<int64_t>(kb) * 128 * ES + x_off;
#pragma unroll
      for (int v = 0; v < XV; ++v) xr[j][v] = *reinterpret_cast<const uint4*>(xp + 16 * v);
      const uint8_t* bp = b_base + kb * 128;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        w[j][t][0] = *reinterpret_cast<const v4i*>(bp + b_off[t]);
        w[j][t][1] = *reinterpret_cast<const v4i*>(bp + b_off[t] + 16);
      }
    }
  }

  if (relu) {
#pragma unroll
    for (int j = 0; j < KB; ++j)
#pragma unroll
      for (int v = 0; v < XV; ++v) xr[j][v] = relu16<D>(xr[j][v]);
  }
  // ---- absmax of the 16 rows
  float mx = 0.f;
#pragma unroll
  for (int j = 0; j < KB; ++j)
#pragma unroll
    for (int v = 0; v < XV; ++v) {
      float f[D::kVec];
      unpack16<D>(xr[j][v], f);
#pragma unroll
      for (int e = 0; e < D::kVec; ++e) mx = fmaxf(mx, __builtin_fabsf(f[e]));
    }
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (lane < 16) rowmax[wave][lane] = mx;
  __syncthreads();
  mx = rowmax[0][col];
#pragma unroll
  for (int wv = 1; wv < kSkinnyWaves; ++wv) mx = fmaxf(mx, rowmax[wv][col]);
  const float s = sym_scale<D, QWIX_INT8>(mx);  // the scale of row `col`, as the quantize kernel derives it
  const Divider<D, false, false> div(s);

  // ---- quantize the registers, multiply
  v4i acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[t][e] = 0;
#pragma unroll
  for (int j = 0; j < KB; ++j) {
    if (kb0 + j < kb1) {
      uint32_t qw[8];  // 32 int8 values, 4 per word, in k order
      constexpr int PER = D::kVec / 4;  // words a 16-byte vector turns into
#pragma unroll
      for (int v = 0; v < XV; ++v) {
        float f[D::kVec];
        unpack16<D>(xr[j][v], f);
#pragma unroll
        for (int h = 0; h < PER; ++h)
          qw[v * PER + h] = pack4_low_bytes(rne_bits_clamped(div(f[4 * h]), -128.f, 127.f),
                                            rne_bits_clamped(div(f[4 * h + 1]), -128.f, 127.f),
                                            rne_bits_clamped(div(f[4 * h + 2]), -128.f, 127.f),
                                            rne_bits_clamped(div(f[4 * h + 3]), -128.f, 127.f));
      }
      const v4i x0 = {static_cast<int>(qw[0]), static_cast<int>(qw[1]), static_cast<int>(qw[2]), static_cast<int>(qw[3])};
      const v4i x1 = {static_cast<int>(qw[4]), static_cast<int>(qw[5]), static_cast<int>(qw[6]), static_cast<int>(qw[7])};
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, w[j][t][0], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, w[j][t][1], acc[t], 0, 0, 0);
      }
    }
  }

#pragma unroll
  for (int t = 0; t < NT; ++t) red[wave][t][lane] = acc[t];
  // the row scales in the result's lane layout: row m = 4 * (lane / 16) + e of the block
  __shared__ float srow[16];
  if (wave == 0 && lane < 16) srow[lane] = s;
  __syncthreads();
  const bool r0 = ep.r0 != 0, r1 = ep.r1 != 0, r2 = ep.r2 != 0;
  for (int idx = tid; idx < NT * 256; idx += kSkinnyWaves * 64) {
    const int t = idx >> 8, e = (idx >> 6) & 3, l = idx & 63;
    const int mr = 4 * (l >> 4) + e;
    const int m = row0 + mr, n = n_base + t * 16 + (l & 15);
    if (m >= M || n >= N) continue;
    int a = 0;
#pragma unroll
    for (int wv = 0; wv < kSkinnyWaves; ++wv) a += red[wv][t][l][e];
    float v = static_cast<float>(a);
    if (r0) v = round_bf16(v);
    v *= srow[mr];
    if (r1) v = round_bf16(v);
    if (ep.sb != nullptr) v *= load_scale(ep.sb, ep.sb_dtype, n);
    if (r2) v = round_bf16(v);
    if (ep.out_dtype == QWIX_BF16)
      reinterpret_cast<uint16_t*>(out)[static_cast<int64_t>(m) * ldo + n] = f32_to_bf16_bits(v);
    else
      reinterpret_cast<float*>(out)[static_cast<int64_t>(m) * ldo + n] = v;
  }
}

template <typename D, int KB>
int launch_skinny_fused(const void* x, int64_t ldx, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K, bool relu,
                        const Epilogue& ep, void* out, int64_t ldo, hipStream_t st) {
  const unsigned gy = static_cast<unsigned>((M + 15) / 16);
#define QWIX_FUSED(NTT)                                                                                              \
  qgemm_skinny_fused_kernel<D, NTT, KB><<<dim3(static_cast<unsigned>((N + 16 * NTT - 1) / (16 * NTT)), gy),         \
                                          kSkinnyWaves * 64, 0, st>>>(static_cast<const uint8_t*>(x), ldx,           \
                                                                      static_cast<const uint8_t*>(b), ldb,           \
                                                                      static_cast<int>(M), static_cast<int>(N),      \
                                                                      static_cast<int>(K), relu ? 1 : 0, ep, static_cast<uint8_t*>(out), ldo)
  if (N >= 192 * 32)
    QWIX_FUSED(2);
  else
    QWIX_FUSED(1);
#undef QWIX_FUSED
  return check_launch("qgemm (skinny, fused activation quantize)");
}

// out[r] = sum_k q[r, k] over int8 rows: one wavefront per row, 16 bytes per lane and trip.
__global__ void __launch_bounds__(256) ksum_i8_kernel(const int8_t* __restrict__ q, int64_t ld, int rows, int K,
                                                      int32_t* __restrict__ out) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int8_t* p = q + static_cast<int64_t>(row) * ld;
  int s = 0;
  for (int k = lane * 16; k < K; k += 64 * 16) {  // K % 16 == 0
    const int4 w = *reinterpret_cast<const int4*>(p + k);
    const int u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) s += (u[e] << 24 >> 24) + (u[e] << 16 >> 24) + (u[e] << 8 >> 24) + (u[e] >> 24);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  if (lane == 0) out[row] = s;
}

}  // namespace
}  // namespace qwix

extern "C" int qwix_hip_ksum_i8(const void* q, int64_t ld, int64_t rows, int64_t K, int32_t* out, void* stream) {
  if (!q || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null argument");
  if (rows <= 0 || K <= 0 || rows > INT32_MAX || K > INT32_MAX || K % 16 || ld % 16 || ld < K || !aligned16(q))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "ksum_i8 needs K and ld multiples of 16 and a 16-byte aligned base "
                "(rows=%lld K=%lld ld=%lld)", (long long)rows, (long long)K, (long long)ld);
  ksum_i8_kernel<<<dim3(static_cast<unsigned>((rows + 3) / 4)), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const int8_t*>(q), ld, static_cast<int>(rows), static_cast<int>(K), out);
  return check_launch("ksum_i8");
}

static int qgemm_impl(const void* a, int64_t lda, const void* b, int64_t ldb, int qtype, int64_t M, int64_t N, int64_t K,
                      const void* sa, int sa_dtype, const void* sb, int sb_dtype, int acc_dtype, const void* zu,
                      const int32_t* zv, void* out, int out_dtype, int64_t ldo, void* stream, void* workspace = nullptr,
                      size_t workspace_bytes = 0, bool zu8 = false);
static int splitk_plan(int64_t M, int64_t N, int64_t K, double other_us, double* model_us = nullptr);
static bool splits_in_workgroup(int64_t M, int64_t N, int64_t K, bool few_rows, double other_us);
// Problems of up to this many 128 x 128 tiles take 64 x 64 tiles (four times the workgroups).  Measured, int8 and
// e4m3, bf16 result, weights in the second-level cache / from HBM: 256 x 4096 over K 1024 9.5 -> 5.6 / 12.1 -> 8.4 us,
// 1024^3 9.3 -> 5.4 / 11.7 -> 8.2, 512 x 4096 over K 4096 23.5 -> 16.2 / 34.9 -> 26.8, 1536 x 2048 over K 2048 (192
// tiles) 16.0 -> 12.6 / 18.3 -> 14.6; level from 256 tiles on (2048 x 2048 over K 1024: 10.6 / 10.4 us), behind at 512
// (4096 x 2048 over K 1024: 13.0 / 17.1 us).
#ifndef QWIX_SMALL_TILES
#define QWIX_SMALL_TILES 200
#endif
constexpr int64_t kSmallTiles = QWIX_SMALL_TILES;

// What the unsplit tiled kernel takes, in us (the figure a split of K has to beat), with weights that come from HBM
// as a model's do (copies in rotation, 600 MB): 64 x 64 tiles with four stages 3.5 us + 0.29 us per 128 of K and round
// of 256 workgroups (256 x 1024 over K 4096 12.7 us, 512 x 512 over K 8192 21.8 us, 512 x 4096 over K 4096 21.0 us),
// 0.58 us per slab with two stages, 128 x 128 tiles beyond.
static double tiled_model_us(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128), tiles64 = ((M + 63) / 64) * ((N + 63) / 64);
  const double slabs = static_cast<double>(K / 128);
  if (M < 64 && N * K >= (int64_t{8} << 20)) return 5.0 + 0.55 * slabs;  // the one-tile-row kernel's range
  if (tiles128 <= kSmallTiles && tiles64 <= 512) return 3.5 + 0.29 * slabs * (tiles64 <= 256 ? 1.0 : tiles64 / 256.0);
  if (tiles128 <= kSmallTiles) return 3.5 + 0.58 * slabs;
  return 5.0 + 0.55 * slabs;
}

static bool streams_weights(int64_t M, int64_t N, int64_t K, bool one_tile_row = false);

static int fused_act_impl(const void* x, int x_dtype, int64_t ldx, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                          bool relu, const void* sb, int sb_dtype, void* out, int out_dtype, int64_t ldo, void* stream) {
  if (!x || !b || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null x/b/out");
  if (x_dtype != QWIX_BF16 && x_dtype != QWIX_F32) return fail(QWIX_ERR_INVALID_ARGUMENT, "activations must be bf16 or f32");
  if ((sb && sb_dtype != QWIX_BF16 && sb_dtype != QWIX_F32) || (out_dtype != QWIX_BF16 && out_dtype != QWIX_F32))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "scale and output dtypes must be f32 or bf16");
  const int es = x_dtype == QWIX_BF16 ? 2 : 4;
  // One 128-wide K block per wavefront: beyond K = 2048 the arithmetic of re-quantizing the rows in every
  // workgroup costs more than the launch of a separate quantize kernel saves (measured: K = 1024 runs in half
  // the time of the two launches, K = 4096 in the same time).
  constexpr int64_t kMaxK = 128 * kSkinnyWaves;
  if (M <= 0 || M > 32 || N <= 0 || N > INT32_MAX || K <= 0 || K % 128 || K > kMaxK)
    return fail(QWIX_ERR_UNSUPPORTED, "fused activation quantize needs 1..32 rows and K a multiple of 128 up to %lld "
                "(M=%lld K=%lld)", (long long)kMaxK, (long long)M, (long long)K);
  if (ldx < K || (ldx * es) % 16 || ldb < K || ldb % 16 || !aligned16(x) || !aligned16(b) || ldo < N ||
      32 * ldx * es >= (int64_t{1} << 31) || 64 * ldb >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "bad leading dimensions or alignment (ldx=%lld ldb=%lld ldo=%lld)", (long long)ldx,
                (long long)ldb, (long long)ldo);
  // the activation scale is computed in the activations' dtype, like the stand-alone quantize does
  const Epilogue ep = make_epilogue(QWIX_INT8, x, x_dtype, sb, sb_dtype, 0, nullptr, nullptr, out_dtype);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (x_dtype == QWIX_BF16) return launch_skinny_fused<BF16, 1>(x, ldx, b, ldb, M, N, K, relu, ep, out, ldo, st);
  return launch_skinny_fused<F32, 1>(x, ldx, b, ldb, M, N, K, relu, ep, out, ldo, st);
}

extern "C" int qwix_hip_qgemm_fused_act(const void* x, int x_dtype, int64_t ldx, const void* b, int64_t ldb,
                                        int64_t M, int64_t N, int64_t K, const void* sb, int sb_dtype, void* out,
                                        int out_dtype, int64_t ldo, void* stream) {
  return fused_act_impl(x, x_dtype, ldx, b, ldb, M, N, K, false, sb, sb_dtype, out, out_dtype, ldo, stream);
}

// Workspace of qwix_hip_qgemm_dynamic_act: the quantized rows, their scales, what the quantize kernel itself needs
// for rows too long for one workgroup, and the GEMM's split-K partials; each part 256-byte aligned.
static size_t dyn_align(size_t v) { return (v + 255) & ~size_t{255}; }
extern "C" size_t qwix_hip_qgemm_dynamic_act_workspace_bytes(int64_t M, int64_t N, int64_t K, int x_dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const size_t es = x_dtype == QWIX_BF16 ? 2 : 4;
  return dyn_align(static_cast<size_t>(M) * K) + dyn_align(static_cast<size_t>(M) * es) +
         dyn_align(qwix_hip_quantize_workspace_bytes(M, K, 1, K, QWIX_ABSMAX)) +
         dyn_align(qwix_hip_qgemm_workspace_bytes(M, N, K));
}

static int dynamic_act_impl(const void* x, int x_dtype, int64_t ldx, const void* b, int64_t ldb, int qtype, int64_t M, int64_t N,
                            int64_t K, bool relu, const void* sb, int sb_dtype, int acc_dtype, void* out, int out_dtype,
                            int64_t ldo, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !b || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null x/b/out");
  if (x_dtype != QWIX_BF16 && x_dtype != QWIX_F32) return fail(QWIX_ERR_INVALID_ARGUMENT, "activations must be bf16 or f32");
  if (qtype != QWIX_INT8 && qtype != QWIX_E4M3)
    return fail(QWIX_ERR_UNSUPPORTED, "dynamic activation quantization to int8 or e4m3 (got qtype %d)", qtype);
  if (M <= 0 || N <= 0 || K <= 0) return fail(QWIX_ERR_INVALID_ARGUMENT, "bad shape M=%lld N=%lld K=%lld", (long long)M,
                                             (long long)N, (long long)K);
  // decode-size int8 calls: one launch (the rows are quantized in the GEMM's prologue)
  if (qtype == QWIX_INT8 && M <= 32 && K % 128 == 0 && K <= 128 * kSkinnyWaves && sb != nullptr)
    return fused_act_impl(x, x_dtype, ldx, b, ldb, M, N, K, relu, sb, sb_dtype, out, out_dtype, ldo, stream);
  // otherwise: the quantize kernel, then the GEMM, on the caller's scratch memory
  if (ldx != K) return fail(QWIX_ERR_UNSUPPORTED, "the two-launch route needs dense activation rows (ldx=%lld K=%lld)",
                            (long long)ldx, (long long)K);
  const size_t need = qwix_hip_qgemm_dynamic_act_workspace_bytes(M, N, K, x_dtype);
  if (!workspace || workspace_bytes < need || !aligned16(workspace))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "workspace of %zu bytes required, got %zu", need, workspace_bytes);
  const size_t es = x_dtype == QWIX_BF16 ? 2 : 4;
  uint8_t* q = static_cast<uint8_t*>(workspace);
  uint8_t* sa = q + dyn_align(static_cast<size_t>(M) * K);
  uint8_t* qws = sa + dyn_align(static_cast<size_t>(M) * es);
  const size_t qws_bytes = qwix_hip_quantize_workspace_bytes(M, K, 1, K, QWIX_ABSMAX);
  uint8_t* gws = qws + dyn_align(qws_bytes);
  const size_t gws_bytes = qwix_hip_qgemm_workspace_bytes(M, N, K);
  if (relu && (K % 8 || K * static_cast<int64_t>(es) > 16 * 2048 || !aligned16(x)))
    return fail(QWIX_ERR_UNSUPPORTED, "a ReLU in front needs 16-byte aligned rows of at most 32 KB (K=%lld)", (long long)K);
  if (int e = relu ? quantize_relu_rows(x, x_dtype, M, K, qtype, q, sa, stream)
                   : qwix_hip_quantize(x, x_dtype, M, K, 1, K, qtype, QWIX_ABSMAX, 0.f, QWIX_LAYOUT_NATURAL, q, sa, nullptr,
                                       qws_bytes ? qws : nullptr, qws_bytes, stream))
    return e;
  return qgemm_impl(q, K, b, ldb, qtype, M, N, K, sa, x_dtype, sb, sb_dtype, acc_dtype, nullptr, nullptr, out, out_dtype,
                    ldo, stream, gws_bytes ? gws : nullptr, gws_bytes);
}

extern "C" int qwix_hip_qgemm_dynamic_act(const void* x, int x_dtype, int64_t ldx, const void* b, int64_t ldb, int qtype,
                                          int64_t M, int64_t N, int64_t K, const void* sb, int sb_dtype, int acc_dtype,
                                          void* out, int out_dtype, int64_t ldo, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  return dynamic_act_impl(x, x_dtype, ldx, b, ldb, qtype, M, N, K, false, sb, sb_dtype, acc_dtype, out, out_dtype, ldo, workspace,
                          workspace_bytes, stream);
}

extern "C" int qwix_hip_qgemm_dynamic_relu(const void* x, int x_dtype, int64_t ldx, const void* b, int64_t ldb, int qtype,
                                           int64_t M, int64_t N, int64_t K, const void* sb, int sb_dtype, int acc_dtype,
                                           void* out, int out_dtype, int64_t ldo, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  return dynamic_act_impl(x, x_dtype, ldx, b, ldb, qtype, M, N, K, true, sb, sb_dtype, acc_dtype, out, out_dtype, ldo, workspace,
                          workspace_bytes, stream);
}

extern "C" int qwix_hip_gemm_bf16(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                                  void* out, int out_dtype, int64_t ldo, void* stream) {
  if (!a || !b || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null a/b/out");
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || 2 * K > INT32_MAX)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad GEMM shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
                (long long)K);
  if (out_dtype != QWIX_BF16 && out_dtype != QWIX_F32) return fail(QWIX_ERR_INVALID_ARGUMENT, "bad out dtype %d", out_dtype);
  // rows are walked in 128-byte slabs that go to LDS directly
  if (K % 64 || lda % 8 || ldb % 8 || lda < K || ldb < K || !aligned16(a) || !aligned16(b))
    return fail(QWIX_ERR_UNSUPPORTED, "bf16 GEMM needs K a multiple of 64, row pitches multiples of 8 elements and "
                "16-byte aligned operands (K=%lld lda=%lld ldb=%lld)", (long long)K, (long long)lda, (long long)ldb);
  if (ldo < N || !aligned16(out) || (N % 4 == 0 && ldo % 4 != 0))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad output leading dimension %lld for N=%lld", (long long)ldo, (long long)N);
  const int64_t ldab = 2 * lda, ldbb = 2 * ldb, kb = 2 * K;  // the tile bodies count bytes
  if (M * ldab >= (int64_t{1} << 31) || N * ldbb >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "operands beyond 2 GiB are not supported by the bf16 GEMM");
  const Epilogue ep{nullptr, nullptr, 0, 0, out_dtype, 0, 0, 0, 0, nullptr, nullptr};
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool big = ((M + 255) / 256) * ((N + 255) / 256) >= 192;
  const int tm = pp_rows(M, N, kb);
  // Below that the rules of the quantized GEMM, which walks slabs of the same bytes: 64 x 64 tiles up to kSmallTiles tiles
  // of 128 x 128, four slab stages while they are at most two per CU; three stages for 128 x 128 tiles that are at
  // most one per CU.  With the dequantization in front, int4: 1300 x 1024 over K 1024 18.3 -> 12.6 us, 3000 x 1024 over K 7168
  // 87 -> 74, 1500 x 2048 over K 14336 167 -> 146, 2000 x 2048 over K 4096 (256 tiles) 54.3 -> 49.5.
  const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128), tiles64 = ((M + 63) / 64) * ((N + 63) / 64);
  auto run = [&](auto out_tag) {
    constexpr int OUT = decltype(out_tag)::value;
    if (tm && kb >= 256) return launch_pp<kOpBf16, OUT, 0>(tm, a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
    if (big) return launch_dma<kOpBf16, 256, 256, 2, 4, OUT, 0>(a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
    if (tiles128 <= kSmallTiles && tiles64 <= 512) return launch_dma<kOpBf16, 64, 64, 2, 2, OUT, 0, 4>(a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
    if (tiles128 <= kSmallTiles) return launch_dma<kOpBf16, 64, 64, 2, 2, OUT, 0>(a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
    if (tiles128 <= 256) return launch_dma<kOpBf16, 128, 128, 2, 2, OUT, 0, 3>(a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
    return launch_dma<kOpBf16, 128, 128, 2, 2, OUT, 0>(a, ldab, b, ldbb, M, N, kb, ep, out, ldo, st);
  };
  return out_dtype == QWIX_BF16 ? run(std::integral_constant<int, QWIX_BF16>{}) : run(std::integral_constant<int, QWIX_F32>{});
}

extern "C" int qwix_hip_qgemm(const void* a, int64_t lda, const void* b, int64_t ldb, int qtype, int64_t M,
                              int64_t N, int64_t K, const void* sa, int sa_dtype, const void* sb, int sb_dtype,
                              int acc_dtype, void* out, int out_dtype, int64_t ldo, void* stream) {
  return qgemm_impl(a, lda, b, ldb, qtype, M, N, K, sa, sa_dtype, sb, sb_dtype, acc_dtype, nullptr, nullptr, out,
                    out_dtype, ldo, stream);
}

extern "C" size_t qwix_hip_qgemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  // the split count qwix_hip_qgemm_ws would pick: the plan against the unsplit tiled kernel's model
  const int splits = streams_weights(M, N, K) ? 0 : splitk_plan(M, N, K, tiled_model_us(M, N, K));
  return splits > 0 ? static_cast<size_t>(splits) * M * N * 4 : 0;
}

extern "C" int qwix_hip_qgemm_ws(const void* a, int64_t lda, const void* b, int64_t ldb, int qtype, int64_t M,
                                 int64_t N, int64_t K, const void* sa, int sa_dtype, const void* sb, int sb_dtype,
                                 int acc_dtype, void* out, int out_dtype, int64_t ldo, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  return qgemm_impl(a, lda, b, ldb, qtype, M, N, K, sa, sa_dtype, sb, sb_dtype, acc_dtype, nullptr, nullptr, out,
                    out_dtype, ldo, stream, workspace, workspace_bytes);
}

extern "C" int qwix_hip_qgemm_zp(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N,
                                 int64_t K, const void* sa, int sa_dtype, const void* sb, int sb_dtype,
                                 const int32_t* zu, const int32_t* zv, void* out, int out_dtype, int64_t ldo,
                                 void* stream) {
  if (!zu || !zv) return fail(QWIX_ERR_INVALID_ARGUMENT, "null zero-point vectors");
  if (out_dtype != QWIX_F32 && out_dtype != QWIX_BF16)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "zero-point corrected output must be f32 or bf16");
  return qgemm_impl(a, lda, b, ldb, QWIX_INT8, M, N, K, sa, sa_dtype, sb, sb_dtype, 0, zu, zv, out, out_dtype, ldo,
                    stream);
}

extern "C" int qwix_hip_qgemm_zp_i8(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N,
                                    int64_t K, const void* sa, int sa_dtype, const void* sb, int sb_dtype,
                                    const int8_t* zu, const int32_t* zv, void* out, int out_dtype, int64_t ldo,
                                    void* stream) {
  if (!zu || !zv) return fail(QWIX_ERR_INVALID_ARGUMENT, "null zero-point vectors");
  if (out_dtype != QWIX_F32 && out_dtype != QWIX_BF16)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "zero-point corrected output must be f32 or bf16");
  return qgemm_impl(a, lda, b, ldb, QWIX_INT8, M, N, K, sa, sa_dtype, sb, sb_dtype, 0, zu, zv, out, out_dtype, ldo,
                    stream, nullptr, 0, true);
}

extern "C" int qwix_hip_qgemm_batched(const void* a, int64_t lda, int64_t a_batch_stride, const void* b, int64_t ldb,
                                      int64_t b_batch_stride, int qtype, int64_t batch, int64_t M, int64_t N,
                                      int64_t K, const void* sa, int sa_dtype, int64_t sa_batch_stride,
                                      const void* sb, int sb_dtype, int64_t sb_batch_stride, int acc_dtype,
                                      void* out, int out_dtype, int64_t ldo, int64_t out_batch_stride,
                                      void* stream) {
  if (const int rc = check_gemm_args(a, lda, b, ldb, qtype, M, N, K, sa, sa_dtype, sb, sb_dtype, acc_dtype, out,
                                     out_dtype, ldo))
    return rc;
  if (batch <= 0 || batch > 65535)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "batched qgemm needs 1..65535 problems (batch=%lld)", (long long)batch);
  if (a_batch_stride % 16 || b_batch_stride % 16 || a_batch_stride < 0 || b_batch_stride < 0 || sa_batch_stride < 0 ||
      sb_batch_stride < 0 || out_batch_stride < 0 || (N % 4 == 0 && (sb_batch_stride % 4 || out_batch_stride % 4)))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad batch strides (a %lld b %lld bytes; sa %lld sb %lld out %lld elements)",
                (long long)a_batch_stride, (long long)b_batch_stride, (long long)sa_batch_stride,
                (long long)sb_batch_stride, (long long)out_batch_stride);
  if (M * lda >= (int64_t{1} << 31) || N * ldb >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "batched qgemm: one problem must fit 32-bit offsets (M*lda=%lld N*ldb=%lld)",
                (long long)(M * lda), (long long)(N * ldb));
  const Epilogue ep = make_epilogue(qtype, sa, sa_dtype, sb, sb_dtype, acc_dtype, nullptr, nullptr, out_dtype);
  const Batched bs{a_batch_stride, b_batch_stride, sa_batch_stride, sb_batch_stride, out_batch_stride};
  // A short contraction: strips of rows instead of tiles (the result's traffic is all there is)
  const bool all_bf = ep.r0 && ep.r1 && ep.r2 && sa_dtype == QWIX_BF16 && sb_dtype == QWIX_BF16 && out_dtype == QWIX_BF16;
  const bool all_f32 = !ep.r0 && !ep.r1 && !ep.r2 && sa_dtype == QWIX_F32 && sb_dtype == QWIX_F32 && out_dtype == QWIX_F32;
  const int64_t piece = out_dtype == QWIX_BF16 ? 8 : 4;
  if ((K == 64 || K == 128) && sa && sb && (all_bf || all_f32) && N % piece == 0 && ldo % piece == 0 &&
      out_batch_stride % piece == 0 && sb_batch_stride % 4 == 0 && aligned16(sb) &&
      (M + 128) * ldo * (out_dtype == QWIX_BF16 ? 2 : 4) < (int64_t{1} << 31)) {
    const StripArgs p{static_cast<const uint8_t*>(a), lda, a_batch_stride, static_cast<const uint8_t*>(b), ldb, b_batch_stride,
                      sa, sa_batch_stride, sb, sb_batch_stride, static_cast<uint8_t*>(out), ldo, out_batch_stride,
                      static_cast<int>(M), static_cast<int>(N)};
    return qgemm_strips(qtype, K, all_bf, p, batch, stream);
  }
  // A long contraction and few tiles: workgroups that split it
  if (qgemm_long_takes(M, N, K, batch) && N % 4 == 0 && ldo % 4 == 0 && out_batch_stride % 4 == 0 && out_dtype != QWIX_I32) {
    const LongArgs p{static_cast<const uint8_t*>(a), lda, a_batch_stride, static_cast<const uint8_t*>(b), ldb, b_batch_stride,
                     sa, sa_dtype, sa_batch_stride, sb, sb_dtype, sb_batch_stride, ep.r0, ep.r1, ep.r2,
                     static_cast<uint8_t*>(out), out_dtype, ldo, out_batch_stride, static_cast<int>(M), static_cast<int>(N),
                     static_cast<int>(K)};
    return qgemm_long(qtype, p, batch, stream);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (qtype == QWIX_INT8) return launch_batched<QWIX_INT8>(a, lda, b, ldb, bs, batch, M, N, K, ep, out, ldo, st);
  return launch_batched<QWIX_E4M3>(a, lda, b, ldb, bs, batch, M, N, K, ep, out, ldo, st);
}

// Up to this many rows of x they are one strip, which quantizes its rows and the rows of y as it loads them: 64 x 1 x 240 x 64 e4m3
// 16.6 -> 7.9 us with the operator (three launches before).  Beyond it each strip would do y again; x quantized by the strips alone
// costs them more than a launch that does both (32 x 2048 x 2048 x 128: 94 us; two launches in front 91.6, one 84.5).
constexpr int64_t kActRows = 64;

extern "C" size_t qwix_hip_qgemm_batched_act_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (batch <= 0 || M <= kActRows || N <= 0 || K <= 0) return 0;
  return dyn_align(static_cast<size_t>(batch) * M * K) + dyn_align(static_cast<size_t>(batch) * N * K) +
         dyn_align(static_cast<size_t>(batch) * M * 2) + dyn_align(static_cast<size_t>(batch) * N * 2);
}

extern "C" int qwix_hip_qgemm_batched_act(const void* x, const void* y, int qtype, int64_t batch, int64_t M, int64_t N, int64_t K,
                                          void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !y || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null x/y/out");
  if (qtype != QWIX_INT8 && qtype != QWIX_E4M3) return fail(QWIX_ERR_UNSUPPORTED, "int8 or e4m3 (got qtype %d)", qtype);
  if (batch <= 0 || batch > 65535 || M <= 0 || N <= 0 || M > INT32_MAX || N > INT32_MAX)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad shape batch=%lld M=%lld N=%lld", (long long)batch, (long long)M, (long long)N);
  if ((K != 64 && K != 128) || N % 8 || (M + 128) * N * 2 >= (int64_t{1} << 31) || M * K * 2 >= (int64_t{1} << 31) ||
      N * K * 2 >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "K 64 or 128, N a multiple of 8, one problem within 32-bit offsets (M=%lld N=%lld K=%lld)",
                (long long)M, (long long)N, (long long)K);
  if (!aligned16(x) || !aligned16(y) || !aligned16(out)) return fail(QWIX_ERR_INVALID_ARGUMENT, "x, y and out must be 16-byte aligned");
  StripArgs p{static_cast<const uint8_t*>(x), 2 * K, 2 * M * K, static_cast<const uint8_t*>(y), 2 * K, 2 * N * K,
              nullptr, 0, nullptr, 0, static_cast<uint8_t*>(out), N, M * N, static_cast<int>(M), static_cast<int>(N)};
  if (M <= kActRows) return qgemm_strips_act(qtype, K, p, batch, stream);
  const size_t need = qwix_hip_qgemm_batched_act_workspace_bytes(batch, M, N, K);
  if (!workspace || workspace_bytes < need || !aligned16(workspace))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "workspace of %zu bytes required, got %zu", need, workspace_bytes);
  uint8_t* qx = static_cast<uint8_t*>(workspace);
  uint8_t* qy = qx + dyn_align(static_cast<size_t>(batch) * M * K);
  uint8_t* sx = qy + dyn_align(static_cast<size_t>(batch) * N * K);
  uint8_t* sy = sx + dyn_align(static_cast<size_t>(batch) * M * 2);
  if (int e = quantize_two_rows(x, batch * M, qx, sx, y, batch * N, qy, sy, K, qtype, stream)) return e;
  p.a = qx;
  p.b = qy;
  p.lda = p.ldb = K;
  p.a_stride = M * K;
  p.b_stride = N * K;
  p.sa = sx;
  p.sb = sy;
  p.sa_stride = M;
  p.sb_stride = N;
  return qgemm_strips(qtype, K, true, p, batch, stream);
}

// The product of probabilities and values: as above with the second operand's contracted axis in front (codes turned while they are
// quantized).  Quantization of both in one launch, then the batched GEMM.
static bool batched_act_kn_shape(int64_t batch, int64_t M, int64_t N, int64_t K) {
  return batch > 0 && batch <= 65535 && M > 0 && N > 0 && K > 0 && M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX &&
         M * K < (int64_t{1} << 30) && N * K < (int64_t{1} << 30) && M * N < (int64_t{1} << 30) && takes_rows_and_cols(batch, M, N, K);
}
extern "C" size_t qwix_hip_qgemm_batched_act_kn_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (!batched_act_kn_shape(batch, M, N, K)) return 0;
  return dyn_align(static_cast<size_t>(batch) * M * K) + dyn_align(static_cast<size_t>(batch) * N * K) +
         dyn_align(static_cast<size_t>(batch) * M * 2) + dyn_align(static_cast<size_t>(batch) * N * 2);
}

extern "C" int qwix_hip_qgemm_batched_act_kn(const void* x, const void* y, int qtype, int64_t batch, int64_t M, int64_t N, int64_t K,
                                             void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !y || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null x/y/out");
  if (qtype != QWIX_INT8 && qtype != QWIX_E4M3) return fail(QWIX_ERR_UNSUPPORTED, "int8 or e4m3 (got qtype %d)", qtype);
  const size_t need = qwix_hip_qgemm_batched_act_kn_workspace_bytes(batch, M, N, K);
  if (need == 0)
    return fail(QWIX_ERR_UNSUPPORTED, "K a multiple of 16, N of 8, columns short enough for strips (batch=%lld M=%lld N=%lld K=%lld)",
                (long long)batch, (long long)M, (long long)N, (long long)K);
  if (!aligned16(x) || !aligned16(y) || !aligned16(out)) return fail(QWIX_ERR_INVALID_ARGUMENT, "x, y and out must be 16-byte aligned");
  if (!workspace || workspace_bytes < need || !aligned16(workspace))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "workspace of %zu bytes required, got %zu", need, workspace_bytes);
  uint8_t* qx = static_cast<uint8_t*>(workspace);
  uint8_t* qy = qx + dyn_align(static_cast<size_t>(batch) * M * K);
  uint8_t* sx = qy + dyn_align(static_cast<size_t>(batch) * N * K);
  uint8_t* sy = sx + dyn_align(static_cast<size_t>(batch) * M * 2);
  if (int e = quantize_rows_and_cols(x, qx, sx, y, qy, sy, batch, M, N, K, qtype, stream)) return e;
  return qwix_hip_qgemm_batched(qx, K, M * K, qy, K, N * K, qtype, batch, M, N, K, sx, QWIX_BF16, M, sy, QWIX_BF16, N,
                                qtype == QWIX_INT8 ? 0 : QWIX_BF16, out, QWIX_BF16, N, M * N, stream);
}

// ------------------------------------------------------------------------------------------------
// Split-K for problems whose 128 x 128 tiles occupy a fraction of the chip while K is long (a few hundred
// rows against a narrow weight): the grid gets a second dimension over ranges of K slabs, every workgroup
// writes its raw partial tile (int32, or f32 for e4m3) to a caller workspace [split][M][N], and a second
// kernel sums the splits and applies the epilogue.  Integer partials add exactly, so int8 results are the
// bits of the unsplit kernels.
template <int QT>
__global__ void __launch_bounds__(256)
    qgemm_splitk_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb, int M,
                        int N, int K, int slabs_per_split, uint8_t* __restrict__ ws) {
  int tile_m, tile_n;
  tile_coords((M + 127) / 128, (N + 127) / 128, &tile_m, &tile_n);
  const int k0 = blockIdx.y * slabs_per_split * 128;
  const int klen = min(K - k0, slabs_per_split * 128);  // > 0: the host sizes the grid that way
  const Epilogue raw{nullptr, nullptr, 0, 0, QT == QWIX_INT8 ? QWIX_I32 : QWIX_F32, 0, 0, 0, 0, nullptr, nullptr};
  uint8_t* part = ws + static_cast<int64_t>(blockIdx.y) * M * N * 4;
  qgemm_dma_tile<QT, 128, 128, 2, 2, (QT == QWIX_INT8 ? QWIX_I32 : QWIX_F32), 0>(A + k0, lda, B + k0, ldb, tile_m * 128,
                                                                                tile_n * 128, M, N, klen, raw, part, N);
}

// The rule of qgemm_impl for taking the weight-streaming kernel (see there for the model).
static bool streams_weights(int64_t M, int64_t N, int64_t K, bool one_tile_row) {
  const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
  const double passes = static_cast<double>((M + 15) / 16);
  const double skinny_us = 4.0 + passes * (0.5 + static_cast<double>(N) * static_cast<double>(K) / 5.2e6);
  // The tiled kernels, with weights that come from HBM (measured with rotating weights, 32 rows: K 4096 35 us
  // whatever N up to 14336; K 8192, N 28672 71 us; K 4096, N 131072 148 us): about 0.95 us per 128-wide K slab
  // and round of two tiles per CU, and never faster than about 3.8 bytes/ns of weights.
  const double rounds = tiles128 <= 512 ? 1.0 : static_cast<double>(tiles128) / 512.0;
  const double slab_us = 0.95 * static_cast<double>(K / 128) * rounds;
  const double read_us = static_cast<double>(N) * static_cast<double>(K) / 3.8e6;
  const double tiled_us = 5.0 + (slab_us > read_us ? slab_us : read_us);
  if (M <= 16) {
    // One pass either way.  From about 100 MB of weights on, while one or two rounds of 64-column workgroups
    // cover N, the one-tile-row kernel streams them faster (16 rows, K 8192, N 28672: 47.4 against 53.0 us, the
    // rate of a plain device copy; K 4096, N 28672: 27.3 against 30.2 us); with more rounds it falls behind
    // (K 8192, N 57344: 126 against 100 us).
    return !(one_tile_row && N * K >= (int64_t{96} << 20) && N <= 32768);
  }
  if (M <= 32 && one_tile_row) {
    // The one-tile-row kernel is there for this call (qgemm_impl checks what it needs).  With 32 rows and
    // 64-column workgroups it was measured, weights from HBM, at K 4096, N 4096 / 14336 / 28672: 14.2 / 17.5 /
    // 29.5 us; K 8192, N 8192 / 28672: 23.9 / 51.8 us; K 2048, N 8192: 9.7 us (the two passes of the
    // weight-streaming kernel: 11.3 / 25.9 / 30.0, 33.4 / 54.1, 9.7 us): 0.29 us per slab of K while the
    // workgroups are few, 4.8 bytes/ns of weights once they fill the chip.
    // Single-wavefront workgroups (N up to 8192): 0.26 us per slab (K 4096, N 4096 / 6144: 13.1 / 13.0 us,
    // K 8192, N 8192: 22.2 us, K 14336, N 4096: 34.6 us against 11.6 / 14.5, 23.9, 28.9 us).
    const double slabs_us = (N <= 8192 ? 0.26 : 0.29) * static_cast<double>(K / 128);
    const double bytes_us = static_cast<double>(N) * static_cast<double>(K) / 4.8e6;
    return skinny_us < 5.0 + (slabs_us > bytes_us ? slabs_us : bytes_us);
  }
  if (M <= 64 && one_tile_row) {
    // 33 to 64 rows, the same comparison: 0.34 us per slab (K 4096 / 8192 / 14336, N 4096: 16.6 / 27.4 / 44.1
    // us, where three or four passes of the weight-streaming kernel took 19.6 / 31.9 / 52.6 us), 4 bytes/ns.
    const double slabs_us = 0.34 * static_cast<double>(K / 128);
    const double bytes_us = static_cast<double>(N) * static_cast<double>(K) / 4.0e6;
    return skinny_us < 5.8 + (slabs_us > bytes_us ? slabs_us : bytes_us);
  }
  if (M <= 32) return skinny_us < tiled_us;
  // more rows: against the tiled kernel this shape would get (64 x 64 tiles with four stages on small problems:
  // 256 rows over K 8192 against 1024 columns take 22 us there, 30.6 us in sixteen passes of the weight-streaming kernel)
  return M <= 256 && tiles128 <= 256 && skinny_us < tiled_model_us(M, N, K);
}

// Number of K ranges worth cutting the problem into (0: do not split).  Model, in microseconds, fitted to
// measurements (256 x 4096 x 1024: 21.6 unsplit, 15.4 in 8 ranges; 256 x 8192 x 2048: 39.4 and 21.1): a
// 128-wide K slab takes about 0.55, the two launches 9 together, and the partial tiles travel to the
// workspace and back at about 4 bytes/ns.  Splitting has to win by 15 % to be chosen.
static int splitk_plan(int64_t M, int64_t N, int64_t K, double other_us, double* model_us) {
  if (K % 128 != 0 || M <= 32) return 0;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), slabs = K / 128;
  if (tiles > 128 || slabs < 8) return 0;
  int best = 0;
  double best_us = 1e30;
  for (int s = 2; s <= 16 && s * 2 <= slabs && tiles * s <= 512; s *= 2) {
    const double per = static_cast<double>((slabs + s - 1) / s);
    const double waves = static_cast<double>((tiles * s + 255) / 256);
    const double us = 9.0 + 0.55 * per * waves + static_cast<double>(s) * M * N * 8.0 / 4.0e6;
    if (us < 0.85 * other_us && us < best_us) {
      best_us = us;
      best = s;
      if (model_us != nullptr) *model_us = us;
    }
  }
  return best;
}

// Whether the wavefronts of a workgroup should split K (qgemm_long), the tiles being at most one round of the CUs: 4.6 us +
// 0.53 us per four slabs for 32 x 64 tiles, 6.2 + 0.75 for 64 x 64, and the weights at 10 bytes/ns (int8, weights in rotation:
// 256 x 1024 over K 4096 9.4 us, 59 x 4096 over K 4096 9.5, 33 x 8192 over K 8192 18.3, 100 x 4096 over K 14336 25.3; 200 x 3072 over K
// 11264 25.3 with 64 rows).  Against several passes of the weight-streaming kernel over weights that do not stay in the
// caches (33 rows: K 8192, N 8192 25.1 us, K 14336, N 4096 36.2, K 11264, N 3072 28.0) it is ahead from three passes on;
// smaller weights are streamed faster (59 x 1024 over K 4096 7.0 us); otherwise the models decide: `other_us` is the tiled
// kernels', or where K can be split through a workspace that kernel's with 1.5 us on top (100 x 1024 over K 8192: 16.6 us, model 14.5).  Up to 32 rows, and up to 63 where only 64-row tiles are one round, the
// one-tile-row kernel is level or ahead (17 rows: N 8192 over K 8192 17.1 against 19.4 us; 33 rows, N 14336 over K 4096 17.1
// against 18.0).
static bool splits_in_workgroup(int64_t M, int64_t N, int64_t K, bool few_rows, double other_us) {
  if (M <= 16 || K <= 128) return false;
  const int64_t cols = (N + 63) / 64, low = (M + 31) / 32 * cols, high = (M + 63) / 64 * cols;
  if (K % 128 != 0) return qgemm_long_takes(M, N, K, 1);  // (the other way is the register-staged tile)
  if (M <= 32 || (M < 64 ? low : high) > 256) return false;
  if (few_rows) return N * K >= 12 << 20;
  const double steps = static_cast<double>((K / 128 + 3) / 4), read_us = static_cast<double>(N) * static_cast<double>(K) / 1.0e7;
  const double us = (low > 256 ? 6.2 + 0.75 * steps : 4.6 + 0.53 * steps) + read_us;
  return us < 0.95 * other_us;
}

template <int QT>
static int launch_splitk(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K, int splits,
                         const Epilogue& ep, void* out, int64_t ldo, void* ws, hipStream_t st) {
  constexpr size_t smem = 2 * (128 + 128) * 128;
  auto kern = qgemm_splitk_kernel<QT>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), slabs = K / 128;
  const int per = static_cast<int>((slabs + splits - 1) / splits);
  const int used = static_cast<int>((slabs + per - 1) / per);  // every range holds at least one slab
  kern<<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(used)), 256, smem, st>>>(
      static_cast<const uint8_t*>(a), lda, static_cast<const uint8_t*>(b), ldb, static_cast<int>(M), static_cast<int>(N),
      static_cast<int>(K), per, static_cast<uint8_t*>(ws));
  const int64_t threads = (M * N + 3) / 4;
  splitk_reduce_kernel<QT == QWIX_INT8><<<dim3(static_cast<unsigned>((threads + 255) / 256)), 256, 0, st>>>(
      static_cast<const uint8_t*>(ws), used, static_cast<int>(M), static_cast<int>(N), ep, static_cast<uint8_t*>(out), ldo);
  return check_launch("qgemm (split K)");
}

static int qgemm_impl(const void* a, int64_t lda, const void* b, int64_t ldb, int qtype, int64_t M, int64_t N, int64_t K,
                      const void* sa, int sa_dtype, const void* sb, int sb_dtype, int acc_dtype, const void* zu,
                      const int32_t* zv, void* out, int out_dtype, int64_t ldo, void* stream, void* workspace,
                      size_t workspace_bytes, bool zu8) {
  if (const int rc = check_gemm_args(a, lda, b, ldb, qtype, M, N, K, sa, sa_dtype, sb, sb_dtype, acc_dtype, out,
                                     out_dtype, ldo))
    return rc;
  const Epilogue ep = make_epilogue(qtype, sa, sa_dtype, sb, sb_dtype, acc_dtype, zu, zv, out_dtype, zu8);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // Few rows: stream the weights instead of tiling.  Up to 16 rows always; up to 256 rows while a rough cost
  // model favours it (streams_weights): the skinny kernel makes one pass over the weights per 16 rows (about
  // 0.5 us + 5.2 bytes/ns each) after a 4 us start; the tiled kernels walk K in 128-wide slabs after 5 us,
  // however few of the chip's CUs their 128 x 128 tiles occupy.
  const double tiled_us = tiled_model_us(M, N, K);
  // what the one-tile-row kernel (launch_mid) needs
  // (65 to 128 rows: one workgroup per CU for its 96 or 128 KB of LDS stages, so only while one round of
  // workgroups covers N: 64-column ones up to N 16384, 128-column ones up to N 32768.  Measured against the
  // 128 x 128 tile, int8, weights from HBM, K 4096, N 4096 / 14336: 25.9 / 29.3 against 37.1 / 38.7 us; K 8192,
  // N 8192: 43.1 against 67.7 us; K 8192, N 28672: 68.9 against 77.0 us with 128-column workgroups, 90.4 with
  // two rounds of 64-column ones.)
  // 129 to 256 rows, N up to 8192: two tile rows of 128 side by side (four stages, two workgroups per CU) where
  // the 128 x 128 tiles would occupy a quarter of the chip: 256 rows, K 4096, N 4096: 24.6 against 36.5 us;
  // K 8192, N 8192: 43.8 against 65.0 us; K 14336, N 4096: 67.3 against 112.8 us; no gain from N 14336 on.
  const bool mid_ok = (M > 16 || (N * K >= (int64_t{96} << 20) && N <= 32768)) && (M <= 64 || (M <= 128 && (N + 127) / 128 <= 256) ||
                                 (M <= 256 && (N + 63) / 64 <= 128)) && K % 128 == 0 && out_dtype != QWIX_I32 &&
                      (zu == nullptr || qtype == QWIX_INT8) &&
                      N * K >= (int64_t{8} << 20) && M * lda < (int64_t{1} << 31) && N * ldb < (int64_t{1} << 31);
  const bool few_rows = streams_weights(M, N, K, mid_ok);
  const bool off31 = M * lda < (int64_t{1} << 31) && N * ldb < (int64_t{1} << 31);
  // K in ranges through the workspace: only where the caller's holds them (a smaller one is as good as none, whichever kernel
  // is chosen), and only against the tiled kernels: where the weight-streaming kernel is chosen its own model has spoken
  double other_us = tiled_us;
  int splits = 0;
  if (workspace != nullptr && aligned16(workspace) && zu == nullptr && out_dtype != QWIX_I32 && off31 && !few_rows) {
    double split_us = 0;
    splits = splitk_plan(M, N, K, tiled_us, &split_us);
    if (workspace_bytes < static_cast<size_t>(splits) * M * N * 4) splits = 0;
    if (splits > 0) other_us = split_us + 1.5;
  }
  if (splits_in_workgroup(M, N, K, few_rows, other_us) && zu == nullptr && out_dtype != QWIX_I32 && off31 && N % 4 == 0 && ldo % 4 == 0) {
    const LongArgs p{static_cast<const uint8_t*>(a), lda, 0, static_cast<const uint8_t*>(b), ldb, 0, sa, sa_dtype, 0, sb, sb_dtype, 0,
                     ep.r0, ep.r1, ep.r2, static_cast<uint8_t*>(out), out_dtype, ldo, 0, static_cast<int>(M),
                     static_cast<int>(N), static_cast<int>(K)};
    return qgemm_long(qtype, p, 1, stream);
  }
  if (splits > 0) {
    if (qtype == QWIX_INT8) return launch_splitk<QWIX_INT8>(a, lda, b, ldb, M, N, K, splits, ep, out, ldo, workspace, st);
    return launch_splitk<QWIX_E4M3>(a, lda, b, ldb, M, N, K, splits, ep, out, ldo, workspace, st);
  }
  if (few_rows && K % 128 == 0 && M * lda < (int64_t{1} << 31) && 64 * ldb < (int64_t{1} << 31)) {
    if (qtype == QWIX_INT8) return launch_skinny<QWIX_INT8>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    return launch_skinny<QWIX_E4M3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  }
  // 256 x 256 tiles once they fill most of the chip's 256 CUs; smaller problems use the tiles of pp_rows, or 128 x 128 and less.
  const bool big = ((M + 255) / 256) * ((N + 255) / 256) >= 192;
  const int tm = big || !mid_ok ? pp_rows(M, N, K) : 0;
  const bool off32 = M * lda < (int64_t{1} << 31) && N * ldb < (int64_t{1} << 31);  // 32-bit lane offsets
  if (K % 128 == 0 && off32) {  // direct-to-LDS pipeline
    // the ping-pong schedule with 128, 192 or 256 rows (no raw-accumulator variant of it exists)
    if (tm && K >= 256 && out_dtype != QWIX_I32) {
      if (qtype == QWIX_INT8) return dispatch_pp<QWIX_INT8>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      return dispatch_pp<QWIX_E4M3>(tm, a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    }
    // 64 x 64 tiles with four slab stages, at most two per CU
    const bool small_deep = ((M + 127) / 128) * ((N + 127) / 128) <= kSmallTiles && ((M + 63) / 64) * ((N + 63) / 64) <= 512;
    // From 64 rows on those tiles take the shapes of the one-tile-row kernel faster (weights from HBM, 100 rows: K 4096,
    // N 4096 23.5 -> 12.9 us, K 14336, N 4096 68.3 -> 36.2, K 8192, N 8192 41.8 -> 23.5; 64 rows: 14.6 -> 13.2, 41.0 ->
    // 37.9, 25.5 -> 24.3; 256 rows, K 4096, N 4096: 22.5 -> 13.4; level at 48 rows, behind below).  Where they do not
    // apply (N 28672: 224 tiles of 128 x 128) the one-tile-row kernel stays ahead of 128 x 128 tiles (28.6 against 39.3 us
    // at 64 rows).
    if (mid_ok && !(small_deep && M >= 64)) {
      // up to 64 rows against a weight of megabytes (and too many rows, or too large a weight, for the
      // weight-streaming kernel): the tile that keeps three slabs of weights in flight per wavefront
      if (qtype == QWIX_INT8 && zu != nullptr) {  // zero-point correction in the epilogue
        if (out_dtype == QWIX_BF16) return launch_mid<QWIX_INT8, QWIX_BF16, 3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
        return launch_mid<QWIX_INT8, QWIX_F32, 3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      }
      // (the epilogue's rounding flags at compile time in the common case: bf16 scales, bf16 result)
      const bool all_round = ep.r0 && ep.r1 && ep.r2;
      if (qtype == QWIX_INT8) {
        if (out_dtype == QWIX_BF16 && all_round) return launch_mid<QWIX_INT8, QWIX_BF16, 1>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
        if (out_dtype == QWIX_BF16) return launch_mid<QWIX_INT8, QWIX_BF16>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
        return launch_mid<QWIX_INT8, QWIX_F32>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      }
      if (out_dtype == QWIX_BF16 && all_round) return launch_mid<QWIX_E4M3, QWIX_BF16, 1>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      if (out_dtype == QWIX_BF16) return launch_mid<QWIX_E4M3, QWIX_BF16>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      return launch_mid<QWIX_E4M3, QWIX_F32>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    }
    // 128 x 128 tiles that would occupy less than a third of the chip: 64 x 64 tiles, four times as many workgroups
    // (a layer of 256 tokens x 4096 features over K 1024 is 64 tiles of 128 x 128)
    const bool small = ((M + 127) / 128) * ((N + 127) / 128) <= kSmallTiles;
    // four slab stages (64 KB) while the 64 x 64 tiles are at most two per CU: weights from HBM, 256 x 1024 over
    // K 4096 21.8 -> 12.7 us, 512 x 512 over K 8192 40.7 -> 21.8, 512 x 4096 over K 4096 26.8 -> 21.0; with 768 tiles
    // (1536 x 2048 over K 2048) 14.6 -> 17.1 us, so those keep two stages
    const bool deep = ((M + 63) / 64) * ((N + 63) / 64) <= 512;
    // 128 x 128 tiles that are at most one per CU: three slab stages (96 KB).  Weights from HBM, 256 tiles: 1024 x 4096
    // over K 4096 34.8 -> 25.3 us, 2048 x 2048 over K 4096 31.8 -> 26.4, over K 1024 12.5 -> 11.3; with two tiles per CU
    // (512 tiles) the second workgroup hides more than the third stage does (4096 x 2048 over K 1024: 14.2 against 20.0 us)
    const bool one_round = ((M + 127) / 128) * ((N + 127) / 128) <= 256;
    if (qtype == QWIX_INT8) {
      if (big) return dispatch_dma<QWIX_INT8, 256, 256, 2, 4>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      if (small && deep) return dispatch_dma<QWIX_INT8, 64, 64, 2, 2, 4>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      if (small) return dispatch_dma<QWIX_INT8, 64, 64, 2, 2>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      if (one_round) return dispatch_dma<QWIX_INT8, 128, 128, 2, 2, 3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
      return dispatch_dma<QWIX_INT8, 128, 128, 2, 2>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    }
    if (big) return dispatch_dma<QWIX_E4M3, 256, 256, 2, 4>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    if (small && deep) return dispatch_dma<QWIX_E4M3, 64, 64, 2, 2, 4>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    if (small) return dispatch_dma<QWIX_E4M3, 64, 64, 2, 2>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    if (one_round) return dispatch_dma<QWIX_E4M3, 128, 128, 2, 2, 3>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
    return dispatch_dma<QWIX_E4M3, 128, 128, 2, 2>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  }
  // register-staged kernel: any K that is a multiple of 16
  if (qtype == QWIX_INT8) return launch_qgemm<QWIX_INT8, 128, 128, 128>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
  return launch_qgemm<QWIX_E4M3, 128, 128, 128>(a, lda, b, ldb, M, N, K, ep, out, ldo, st);
}
