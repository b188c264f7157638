// Tile bodies of the MFMA GEMMs and the host helpers around them, shared by qgemm.hip (dense and batched), qgemm_ragged.hip
// (rows in groups) and wgemm_wq.hip (bf16 activations x quantized weights).
//
//   qgemm_tile      register-staged 128 x 128 tile, any K that is a multiple of 16
//   qgemm_dma_tile  K % 128 == 0: 128-byte K slabs go global -> LDS directly, two stages (three or four where a
//                   problem's tiles are so few per CU that nothing else covers the latency of the loads)
//   qgemm_pp_tile   128, 192 or 256 x 256, long K: two wavefront groups half a slab out of phase (ping-pong)
//   qgemm_mid_tile  one tile row, weights straight into registers
//   skinny_block    up to 16 rows, K split over the wavefronts
// Each is a device function of a tile origin and a row limit.  K is walked in slabs through LDS; rows are stored so that
// the 16-byte operand reads of 8 consecutive lanes touch all 32 banks once (padding in the register-staged body, an
// XOR swizzle in the others); operands are read back as 16-byte fragments and fed to v_mfma_i32_32x32x32_i8 /
// v_mfma_f32_32x32x64_f8f6f4.  The MFMA "A" operand is fed from b and the "B" operand from a, so that each lane ends up
// with 4 consecutive n for a single m.
#pragma once
#include <type_traits>

#include "common.h"

namespace qwix {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kPad = 16;
// Operand tag of the tile bodies for bf16 x bf16 (the float contraction of the dequantize-first path); the
// byte geometry is that of int8: a 128-byte K slab is four MFMA k-steps of 32 bytes per row (16 bf16 values).
constexpr int kOpBf16 = 16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Swizzle key of the kernels in this file: 16-byte chunk c of the 128-byte LDS row r sits at chunk position
// c ^ swz8(r).  Eight consecutive rows then cover all eight chunk positions; over the sixteen rows that the LDS
// serves per clock for a ds_read_b128 this still leaves two-way bank conflicts, which the sixteen-row key of
// common.h (swz128) removes.  Measured side by side on one card, the conflict-free key is nevertheless 2-5 %
// SLOWER here (int8 4096^3: 72.1 against 70.3 us; 8192^3: 494 against 485 us; the 8-expert ragged GEMM 578
// against 551 us; e4m3 and the one-tile-row kernel unchanged): these kernels run at the board's power limit,
// where faster fragment reads buy nothing and cost clock.  So the eight-row key stays.
__device__ __forceinline__ int swz8(int row) { return row & 7; }

// Epilogue description.  The reference scales the accumulator as ((T(acc) * sa) * sb) with one
// rounding per step in the promoted dtype; which of those roundings are to bf16 is decided on the
// host (r0: the converted accumulator, r1: after the lhs scale, r2: after the rhs scale).
struct Epilogue {
  const void* sa;  // per m, or null
  const void* sb;  // per n, or null
  int sa_dtype, sb_dtype, out_dtype;
  int r0, r1;
  int16_t r2, zu8;  // (16 bits: a word more moves the kernels' last arguments into a third line, which every workgroup waits for)
  // Zero-point correction of an asymmetric operand (int8 only): acc[m,n] -= zu[m] * zv[n], where one
  // vector holds the zero points and the other the K-sums of the opposite operand's quantized values.
  const void* zu;  // int32, or int8 with zu8 (zero points as quantize writes them)
  const int32_t* zv;
};
static_assert(sizeof(Epilogue) == 56, "the argument blocks of the GEMM kernels");
__device__ __forceinline__ int zu_at(const Epilogue& ep, int m) {
  return ep.zu8 ? static_cast<int>(static_cast<const int8_t*>(ep.zu)[m]) : static_cast<const int32_t*>(ep.zu)[m];
}

// XCD-aware tile order: consecutive hardware workgroup ids go to different XCDs; give every XCD a
// contiguous run of logical ids, and walk tiles in column groups of 8 tile-rows for L2 reuse.
__device__ __forceinline__ void tile_coords(int tiles_m, int tiles_n, int* tm, int* tn) {
  const int nb = gridDim.x;
  int pid = blockIdx.x;
  if ((nb & 7) == 0) pid = (pid & 7) * (nb >> 3) + (pid >> 3);
  constexpr int GM = 8;
  const int per_group = GM * tiles_n;
  const int group = pid / per_group;
  const int first_m = group * GM;
  const int gsz = min(tiles_m - first_m, GM);
  *tm = first_m + (pid % per_group) % gsz;
  *tn = (pid % per_group) / gsz;
}

__device__ __forceinline__ float load_scale(const void* p, int dtype, int64_t i) {
  return dtype == QWIX_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i])
                            : reinterpret_cast<const float*>(p)[i];
}

// acc[i][j][r]: m = m_base + i*32 + lane%32,  n = n_base + j*32 + 8*(r/4) + 4*(lane/32) + r%4.
// All scales a lane needs are fetched before its first store, so that the stores (which the
// compiler must keep ordered with loads that may alias) do not serialise the global-load latency.
template <int OUT, int TM, int TN, typename AccT>
__device__ __forceinline__ void write_tile(const AccT (&acc)[TM][TN], const Epilogue& ep, int m_base, int n_base,
                                           int lane, int M, int N, uint8_t* __restrict__ out, int64_t ldo) {
  const bool vec_ok = (N % 4 == 0);
  const bool r0 = ep.r0 != 0, r1 = ep.r1 != 0, r2 = ep.r2 != 0;
  float sav[TM];
  float sbv[TN][4][4];
  if constexpr (OUT != QWIX_I32) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m_base + i * 32 + (lane & 31);
      sav[i] = (ep.sa != nullptr && m < M) ? load_scale(ep.sa, ep.sa_dtype, m) : 1.f;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int n = n_base + j * 32 + 8 * qd + 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 4; ++r) sbv[j][qd][r] = 1.f;
        if (ep.sb != nullptr) {
          if (vec_ok && n < N) {  // n % 4 == 0: one 8- or 16-byte load
            if (ep.sb_dtype == QWIX_BF16) {
              const uint2 w = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(ep.sb) + n);
              sbv[j][qd][0] = __uint_as_float(w.x << 16);
              sbv[j][qd][1] = __uint_as_float(w.x & 0xFFFF0000u);
              sbv[j][qd][2] = __uint_as_float(w.y << 16);
              sbv[j][qd][3] = __uint_as_float(w.y & 0xFFFF0000u);
            } else {
              const float4 w = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(ep.sb) + n);
              sbv[j][qd][0] = w.x; sbv[j][qd][1] = w.y; sbv[j][qd][2] = w.z; sbv[j][qd][3] = w.w;
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < N) sbv[j][qd][r] = load_scale(ep.sb, ep.sb_dtype, n + r);
          }
        }
      }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m_base + i * 32 + (lane & 31);
    const bool m_ok = m < M;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int n = n_base + j * 32 + 8 * qd + 4 * (lane >> 5);
        if (m_ok && n < N) {
          if constexpr (OUT == QWIX_I32) {
            int* o = reinterpret_cast<int*>(out) + static_cast<int64_t>(m) * ldo + n;
            if (vec_ok) {
              *reinterpret_cast<int4*>(o) = make_int4(static_cast<int>(acc[i][j][4 * qd]), static_cast<int>(acc[i][j][4 * qd + 1]),
                                                      static_cast<int>(acc[i][j][4 * qd + 2]), static_cast<int>(acc[i][j][4 * qd + 3]));
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (n + r < N) o[r] = static_cast<int>(acc[i][j][4 * qd + r]);
            }
          } else {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float t;
              if constexpr (std::is_same<AccT, v16i>::value) {
                int a = acc[i][j][4 * qd + r];
                if (ep.zu != nullptr) a -= zu_at(ep, m) * ep.zv[min(n + r, N - 1)];
                t = static_cast<float>(a);
              } else {
                t = static_cast<float>(acc[i][j][4 * qd + r]);
              }
              t = r0 ? round_bf16(t) : t;
              t *= sav[i];
              t = r1 ? round_bf16(t) : t;
              t *= sbv[j][qd][r];
              v[r] = r2 ? round_bf16(t) : t;
            }
            if constexpr (OUT == QWIX_BF16) {
              uint16_t* o = reinterpret_cast<uint16_t*>(out) + static_cast<int64_t>(m) * ldo + n;
              if (vec_ok) {
                *reinterpret_cast<uint2*>(o) =
                    make_uint2(f32_to_bf16_bits(v[0]) | (static_cast<uint32_t>(f32_to_bf16_bits(v[1])) << 16),
                               f32_to_bf16_bits(v[2]) | (static_cast<uint32_t>(f32_to_bf16_bits(v[3])) << 16));
              } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  if (n + r < N) o[r] = f32_to_bf16_bits(v[r]);
              }
            } else {
              float* o = reinterpret_cast<float*>(out) + static_cast<int64_t>(m) * ldo + n;
              if (vec_ok) {
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
              } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  if (n + r < N) o[r] = v[r];
              }
            }
          }
        }
      }
    }
  }
}

// QT: QWIX_INT8 or QWIX_E4M3.  Wave tile = (BM/2) x (BN/2) = TM x TN MFMA tiles of 32x32.
// Software pipeline: while the MFMAs of k-step s run, the fragments of k-step s+1 are read from
// LDS into a second register set; the slab for the next iteration is fetched from global memory
// at the top of the iteration, written to the other LDS stage before the last k-step, and the
// workgroup barrier plus the first fragment read of the next slab hide behind that last k-step.
// The tile at rows [m0, m0 + BM) x columns [n0, n0 + BN); rows from M on are neither read nor stored.
template <int QT, int BM, int BN, int BK>
__device__ __forceinline__ void qgemm_tile(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B,
                                           int64_t ldb, int m0, int n0, int M, int N, int K, const Epilogue& ep,
                                           uint8_t* __restrict__ out, int64_t ldo) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  constexpr int LDS_STRIDE = BK + kPad;
  constexpr int TM = BM / 64, TN = BN / 64;
  constexpr int KSTEP = IS_INT ? 32 : 64;         // K elements (= bytes) per MFMA
  constexpr int NK = BK / KSTEP;
  static_assert(NK >= 2 && NK % 2 == 0, "the fragment double buffer needs an even number of k-steps");
  constexpr int CH = BK / 16;                      // 16-byte chunks per tile row
  constexpr int A_CHUNKS = BM * CH / 256, B_CHUNKS = BN * CH / 256;
  static_assert(BM * CH % 256 == 0 && BN * CH % 256 == 0, "tile/thread mismatch");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int STAGE = (BM + BN) * LDS_STRIDE;  // stage s: A tile at s*STAGE, B tile right after it

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  using AccT = typename std::conditional<IS_INT, v16i, v16f>::type;
  using FragT = typename std::conditional<IS_INT, v4i, v8i>::type;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  uint4 ra[A_CHUNKS], rb[B_CHUNKS];
  auto load_global = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int c = tid + i * 256, row = c / CH, kc = c % CH;
      const int m = m0 + row, k = k0 + kc * 16;
      ra[i] = make_uint4(0, 0, 0, 0);
      if (m < M && k < K) ra[i] = *reinterpret_cast<const uint4*>(A + static_cast<int64_t>(m) * lda + k);
    }
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i) {
      const int c = tid + i * 256, row = c / CH, kc = c % CH;
      const int n = n0 + row, k = k0 + kc * 16;
      rb[i] = make_uint4(0, 0, 0, 0);
      if (n < N && k < K) rb[i] = *reinterpret_cast<const uint4*>(B + static_cast<int64_t>(n) * ldb + k);
    }
  };
  auto store_lds = [&](int s) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const int c = tid + i * 256, row = c / CH, kc = c % CH;
      *reinterpret_cast<uint4*>(smem + s * STAGE + row * LDS_STRIDE + kc * 16) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i) {
      const int c = tid + i * 256, row = c / CH, kc = c % CH;
      *reinterpret_cast<uint4*>(smem + s * STAGE + (BM + row) * LDS_STRIDE + kc * 16) = rb[i];
    }
  };

  FragT fa[2][TM], fb[2][TN];
  const int a_off = (wm * (BM / 2) + (lane & 31)) * LDS_STRIDE + (lane >> 5) * (KSTEP / 2);
  const int b_off = (BM + wn * (BN / 2) + (lane & 31)) * LDS_STRIDE + (lane >> 5) * (KSTEP / 2);
  auto read_frags = [&](int s, int ks, int buf) {
    const uint8_t* pa = smem + s * STAGE + a_off + ks * KSTEP;
    const uint8_t* pb = smem + s * STAGE + b_off + ks * KSTEP;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if constexpr (IS_INT) {
        fa[buf][i] = *reinterpret_cast<const v4i*>(pa + i * 32 * LDS_STRIDE);
      } else {
        const v4i lo = *reinterpret_cast<const v4i*>(pa + i * 32 * LDS_STRIDE);
        const v4i hi = *reinterpret_cast<const v4i*>(pa + i * 32 * LDS_STRIDE + 16);
        fa[buf][i] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (IS_INT) {
        fb[buf][j] = *reinterpret_cast<const v4i*>(pb + j * 32 * LDS_STRIDE);
      } else {
        const v4i lo = *reinterpret_cast<const v4i*>(pb + j * 32 * LDS_STRIDE);
        const v4i hi = *reinterpret_cast<const v4i*>(pb + j * 32 * LDS_STRIDE + 16);
        fb[buf][j] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  auto mfma_step = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (IS_INT)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[buf][j], fa[buf][i], acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[buf][j], fa[buf][i], acc[i][j], 0, 0, 0, 0, 0, 0);
      }
  };

  const int KT = (K + BK - 1) / BK;
  load_global(0);
  store_lds(0);
  __syncthreads();
  read_frags(0, 0, 0);
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    const bool has_next = kt + 1 < KT;
    if (has_next) load_global((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks + 1 < NK; ++ks) {
      read_frags(cur, ks + 1, (ks + 1) & 1);
      mfma_step(ks & 1);
    }
    if (has_next) store_lds(cur ^ 1);
    __syncthreads();
    if (has_next) read_frags(cur ^ 1, 0, 0);
    mfma_step((NK - 1) & 1);
  }

  const int m_base = m0 + wm * (BM / 2), n_base = n0 + wn * (BN / 2);
  if (ep.out_dtype == QWIX_BF16) {
    write_tile<QWIX_BF16, TM, TN>(acc, ep, m_base, n_base, lane, M, N, out, ldo);
  } else if (ep.out_dtype == QWIX_F32) {
    write_tile<QWIX_F32, TM, TN>(acc, ep, m_base, n_base, lane, M, N, out, ldo);
  } else {
    if constexpr (IS_INT) write_tile<QWIX_I32, TM, TN>(acc, ep, m_base, n_base, lane, M, N, out, ldo);
  }
}

// Fast path (K % 128 == 0): the slabs go from global memory straight into LDS
// (global_load_lds_dwordx4: no staging registers, no ds_write instructions).  Each wave-level load
// fills one contiguous KiB of LDS = 8 tile rows x 128 bytes; inside a row the eight 16-byte k-chunks
// are stored at position (chunk ^ swz8(row)), chosen by having each lane fetch the matching global
// chunk, so that the fragment reads of 16 consecutive rows hit all 64 banks.  Rows past M / N are
// clamped to the last valid row (their results are never stored).  Loads for slab kt+1 are issued
// while the MFMAs of slab kt run; the workgroup barrier at the end of the slab waits for them.
// The workgroup is WGM x WGN wavefronts; with 8 wavefronts (two per SIMD) the issue time of one
// wavefront's loads and fragment reads hides behind the other's MFMAs.
// EPI: 0 = no bf16 rounding in the epilogue, 1 = every step rounds to bf16, 2 = flags at run time,
// 3 = flags at run time and zero-point correction, 4 = every step rounds to bf16 and zero-point correction.
#define QWIX_GLDS16(gptr, lptr)                                                                       \
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gptr),             \
                                   (__attribute__((address_space(3))) void*)(lptr), 16, 0, 0)
// The same load from a wave-uniform base pointer plus a per-lane 32-bit byte offset.  The offset is made opaque next to
// the load: the address is then a scalar base register plus a 32-bit vector offset, where an offset that the compiler
// widens to 64 bits ahead of the loop occupies two registers for the whole kernel and costs a 64-bit vector add per load.
#define QWIX_GLDS16_AT(gbase, off32, lptr)                                                            \
  do {                                                                                                \
    uint32_t qwix_off_ = (off32);                                                                     \
    asm volatile("" : "+v"(qwix_off_));                                                               \
    QWIX_GLDS16((gbase) + qwix_off_, lptr);                                                           \
  } while (0)
// The same with the offset variable made opaque in its own register (no copy per load): measured 1 % faster in the
// ping-pong kernel's slab loop, and 20 % slower in the one-slab batched kernel, which therefore takes the form above.
#define QWIX_GLDS16_AT_INPLACE(gbase, off32, lptr)                                                    \
  do {                                                                                                \
    asm volatile("" : "+v"(off32));                                                                   \
    QWIX_GLDS16((gbase) + (off32), lptr);                                                             \
  } while (0)

// The per-row and per-column scales of one wavefront's part of the tile, in the accumulator layout
// (acc[i][j][r]: m = m_base + i*32 + lane%32, n = n_base + j*32 + 8*(r/4) + 4*(lane/32) + r%4).
template <int OUT, int TM, int TN>
__device__ __forceinline__ void fetch_scales(const Epilogue& ep, int m_base, int n_base, int M, int N, int lane,
                                             float (&sav)[TM], float (&sbv)[TN][4][4]) {
  if constexpr (OUT != QWIX_I32) {
    const bool vec_ok = (N % 4 == 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m_base + i * 32 + (lane & 31);
      sav[i] = (ep.sa != nullptr && m < M) ? load_scale(ep.sa, ep.sa_dtype, m) : 1.f;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int n = n_base + j * 32 + 8 * qd + 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 4; ++r) sbv[j][qd][r] = 1.f;
        if (ep.sb != nullptr) {
          if (vec_ok && n < N) {  // n % 4 == 0: one 8- or 16-byte load
            if (ep.sb_dtype == QWIX_BF16) {
              const uint2 w = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(ep.sb) + n);
              sbv[j][qd][0] = __uint_as_float(w.x << 16);
              sbv[j][qd][1] = __uint_as_float(w.x & 0xFFFF0000u);
              sbv[j][qd][2] = __uint_as_float(w.y << 16);
              sbv[j][qd][3] = __uint_as_float(w.y & 0xFFFF0000u);
            } else {
              const float4 w = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(ep.sb) + n);
              sbv[j][qd][0] = w.x; sbv[j][qd][1] = w.y; sbv[j][qd][2] = w.z; sbv[j][qd][3] = w.w;
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < N) sbv[j][qd][r] = load_scale(ep.sb, ep.sb_dtype, n + r);
          }
        }
      }
  }
}

template <int OUT, int EPI, int TM, int TN, int NWAVES, int LDS_BYTES, bool SYNC = true, typename AccT>
__device__ __forceinline__ void staged_epilogue(const AccT (&acc)[TM][TN], const float (&sav)[TM],
                                                const float (&sbv)[TN][4][4], const Epilogue& ep, int m_base,
                                                int n_base, int M, int N, uint8_t* __restrict__ out, int64_t ldo,
                                                uint8_t* smem, int wave, int lane) {
  constexpr int WTN = TN * 32;
  // ---- epilogue.  acc[i][j][r]: m = m_base + i*32 + lane%32, n = n_base + j*32 + 8*(r/4) + 4*(lane/32) + r%4.
  // The scaled values are staged through this wavefront's own slice of LDS, 32 rows at a time, and
  // leave with 16-byte stores that cover whole 128-byte row segments (a direct store from the MFMA
  // layout would write 16-byte pieces of 32 different rows per instruction).
  using OutT = typename std::conditional<OUT == QWIX_BF16, uint16_t, uint32_t>::type;
  constexpr int ES = sizeof(OutT);
  constexpr int ROWB = WTN * ES + 16;            // staged row pitch in bytes (padded against bank conflicts)
  constexpr int CPR = WTN * ES / 16;             // 16-byte chunks per staged row
  constexpr int EPC = 16 / ES;                   // elements per chunk
  static_assert(NWAVES * 32 * ROWB <= LDS_BYTES, "epilogue staging does not fit in LDS");
  constexpr bool ZP = (EPI == 3 || EPI == 4);  // zero-point correction
  constexpr bool ALL = (EPI == 1 || EPI == 4), RUNTIME = (EPI == 2 || EPI == 3);
  const bool r0 = RUNTIME ? ep.r0 != 0 : ALL, r1 = RUNTIME ? ep.r1 != 0 : ALL, r2 = RUNTIME ? ep.r2 != 0 : ALL;
  int zuv[TM];
  if constexpr (ZP) {
#pragma unroll
    for (int i = 0; i < TM; ++i) zuv[i] = zu_at(ep, min(m_base + i * 32 + (lane & 31), M - 1));
  }
  if constexpr (SYNC) __syncthreads();  // every wavefront is done with the slabs; LDS becomes staging space
  uint8_t* stg = smem + wave * (32 * ROWB);
  const bool row_vec = (reinterpret_cast<uintptr_t>(out) % 16 == 0) && ((ldo * ES) % 16 == 0);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    float sa = 1.f;
    if constexpr (OUT != QWIX_I32) sa = sav[i];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        uint8_t* dst = stg + (lane & 31) * ROWB + (j * 32 + 8 * qd + 4 * (lane >> 5)) * ES;
        if constexpr (OUT == QWIX_I32) {
          *reinterpret_cast<int4*>(dst) = make_int4(static_cast<int>(acc[i][j][4 * qd]), static_cast<int>(acc[i][j][4 * qd + 1]),
                                                    static_cast<int>(acc[i][j][4 * qd + 2]), static_cast<int>(acc[i][j][4 * qd + 3]));
        } else if constexpr (ALL && OUT == QWIX_BF16) {
          // Every step rounds to bf16 and the result is bf16: round two values per v_cvt_pk_bf16_f32,
          // and let the last rounding produce the packed output directly.
          uint32_t w[2];
          int zvv[4] = {0, 0, 0, 0};
          if constexpr (ZP) {
            const int n = n_base + j * 32 + 8 * qd + 4 * (lane >> 5);
#pragma unroll
            for (int r = 0; r < 4; ++r) zvv[r] = ep.zv[min(n + r, N - 1)];
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            uint32_t pk;
            if constexpr (ZP)
              pk = pack_bf16x2(static_cast<float>(static_cast<int>(acc[i][j][4 * qd + 2 * h]) - zuv[i] * zvv[2 * h]),
                               static_cast<float>(static_cast<int>(acc[i][j][4 * qd + 2 * h + 1]) - zuv[i] * zvv[2 * h + 1]));
            else
              pk = pack_bf16x2(static_cast<float>(acc[i][j][4 * qd + 2 * h]),
                               static_cast<float>(acc[i][j][4 * qd + 2 * h + 1]));
            pk = pack_bf16x2(__uint_as_float(pk << 16) * sa, __uint_as_float(pk & 0xFFFF0000u) * sa);
            w[h] = pack_bf16x2(__uint_as_float(pk << 16) * sbv[j][qd][2 * h],
                               __uint_as_float(pk & 0xFFFF0000u) * sbv[j][qd][2 * h + 1]);
          }
          *reinterpret_cast<uint2*>(dst) = make_uint2(w[0], w[1]);
        } else {
          float v[4];
          int zvv[4] = {0, 0, 0, 0};
          if constexpr (ZP) {
            const int n = n_base + j * 32 + 8 * qd + 4 * (lane >> 5);
#pragma unroll
            for (int r = 0; r < 4; ++r) zvv[r] = ep.zv[min(n + r, N - 1)];
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float t;
            if constexpr (ZP) t = static_cast<float>(static_cast<int>(acc[i][j][4 * qd + r]) - zuv[i] * zvv[r]);
            else t = static_cast<float>(acc[i][j][4 * qd + r]);
            if (r0) t = round_bf16(t);
            t *= sa;
            if (r1) t = round_bf16(t);
            t *= sbv[j][qd][r];
            if (r2) t = round_bf16(t);
            v[r] = t;
          }
          if constexpr (OUT == QWIX_BF16)
            *reinterpret_cast<uint2*>(dst) =
                make_uint2(f32_to_bf16_bits(v[0]) | (static_cast<uint32_t>(f32_to_bf16_bits(v[1])) << 16),
                           f32_to_bf16_bits(v[2]) | (static_cast<uint32_t>(f32_to_bf16_bits(v[3])) << 16));
          else
            *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    // read back row-major: chunk c of the 32 x CPR grid -> row c / CPR, 16-byte column c % CPR
#pragma unroll
    for (int c0 = 0; c0 < 32 * CPR; c0 += 64) {
      const int c = c0 + lane, row = c / CPR, cc = c % CPR;
      const uint4 v = *reinterpret_cast<const uint4*>(stg + row * ROWB + cc * 16);
      const int mo = m_base + i * 32 + row, no = n_base + cc * EPC;
      if (mo < M && no < N) {
        OutT* o = reinterpret_cast<OutT*>(out) + static_cast<int64_t>(mo) * ldo + no;
        if (row_vec && no + EPC <= N) {
          __builtin_nontemporal_store(__builtin_bit_cast(v4i, v), reinterpret_cast<v4i*>(o));
        } else {
          const OutT* e = reinterpret_cast<const OutT*>(&v);
#pragma unroll
          for (int t = 0; t < EPC; ++t)
            if (no + t < N) o[t] = e[t];
        }
      }
    }
  }
}

// NST: slab stages of the direct-to-LDS tile body.  Two by default; four for the 64 x 64 tile of small problems while
// its workgroups are at most two per CU: they have nothing else to cover the latency of weights that come from HBM
// (three slabs in flight instead of one; with more workgroups per CU the LDS the stages take costs more than it gives).
template <int QT, int BM, int BN, int WGM, int WGN, int OUT, int EPI, int NST = 2>
__device__ __forceinline__ void qgemm_dma_tile(const uint8_t* __restrict__ A, int64_t lda,
                                               const uint8_t* __restrict__ B, int64_t ldb, int m0, int n0, int M,
                                               int N, int K, const Epilogue& ep, uint8_t* __restrict__ out,
                                               int64_t ldo) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  constexpr bool IS_BF = (QT == kOpBf16);
  constexpr bool B16 = IS_INT || IS_BF;  // 16 bytes per lane and k-step
  constexpr int BK = 128;
  constexpr int NWAVES = WGM * WGN;
  constexpr int WTM = BM / WGM, WTN = BN / WGN;   // wave tile
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int KSTEP = B16 ? 32 : 64;
  constexpr int NK = BK / KSTEP;
  constexpr int ROWS = BM + BN;
  constexpr int STAGE = ROWS * BK;
  constexpr int LOADS = ROWS / 8 / NWAVES;  // 1 KiB loads per wavefront per slab
  static_assert(ROWS % (8 * NWAVES) == 0 && (BM / 8) % LOADS == 0, "each wavefront loads from one operand");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  using AccT = typename std::conditional<IS_INT, v16i, v16f>::type;
  using FragT = typename std::conditional<B16, v4i, v8i>::type;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // ---- loader: a wave-uniform base pointer plus this lane's 32-bit offset for each row group
  const int lr = lane >> 3;                       // row inside the 8-row group
  const bool from_a = (wave * LOADS * 8) < BM;    // wave-uniform
  const uint8_t* gbase = from_a ? A : B;
  const int64_t gld = from_a ? lda : ldb;
  const int glim = from_a ? (M - 1) : (N - 1);
  const int grow0 = from_a ? (m0 + wave * LOADS * 8) : (n0 + wave * LOADS * 8 - BM);
  uint32_t goff[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j)
    goff[j] = static_cast<uint32_t>(min(grow0 + j * 8 + lr, glim)) * static_cast<uint32_t>(gld) +
              (((lane & 7) ^ swz8((wave * LOADS + j) * 8 + lr)) << 4);  // the global k-chunk that lands at position lane & 7
  auto issue_loads = [&](int s, int k0) {
    const uint8_t* gk = gbase + k0;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) QWIX_GLDS16_AT(gk, goff[j], smem + s * STAGE + (wave * LOADS + j) * 1024);
  };

  // ---- fragment addresses: row r, k-chunk c lives at r*128 + ((c ^ swz8(r)) << 4); wave tiles start at multiples of 32
  const int a_row = (wm * WTM + (lane & 31)) * BK;
  const int b_row = (BM + wn * WTN + (lane & 31)) * BK;
  const int hx = lane >> 5, x7 = swz8(lane & 31);
  FragT fa[2][TM], fb[2][TN];
  auto read_frags = [&](int s, int ks, int buf) {
    const uint8_t* base = smem + s * STAGE;
    if constexpr (B16) {
      const int off = ((ks * 2 + hx) ^ x7) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[buf][i] = *reinterpret_cast<const v4i*>(base + a_row + i * 32 * BK + off);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[buf][j] = *reinterpret_cast<const v4i*>(base + b_row + j * 32 * BK + off);
    } else {
      const int off = ((ks * 4 + hx * 2) ^ x7) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(base + a_row + i * 32 * BK + off);
        const v4i hi = *reinterpret_cast<const v4i*>(base + a_row + i * 32 * BK + (off ^ 16));
        fa[buf][i] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const v4i lo = *reinterpret_cast<const v4i*>(base + b_row + j * 32 * BK + off);
        const v4i hi = *reinterpret_cast<const v4i*>(base + b_row + j * 32 * BK + (off ^ 16));
        fb[buf][j] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  auto mfma_step = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (IS_INT)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[buf][j], fa[buf][i], acc[i][j], 0, 0, 0);
        else if constexpr (IS_BF)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb[buf][j]),
                                                              __builtin_bit_cast(bf16x8, fa[buf][i]), acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[buf][j], fa[buf][i], acc[i][j], 0, 0, 0, 0, 0, 0);
      }
  };
  // Interleave hints for one k-step: MFMAs in pairs, a fragment read after each pair, and a slab load
  // after each pair while loads remain.
  auto hint_kstep = [&](int n_loads) {
    constexpr int MF = TM * TN, RD = (B16 ? 1 : 2) * (TM + TN);
#pragma unroll
    for (int g = 0; g < MF; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // MFMA
      if (g < RD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           // DS read
      if (g < n_loads) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);      // VMEM read (LDS DMA)
    }
  };

  const int m_base = m0 + wm * WTM, n_base = n0 + wn * WTN;
  float sbv[TN][4][4];
  // The scale vectors are fetched before the main loop: at the start of the epilogue they would be a
  // cold two-microsecond round trip with nothing to hide behind.
  float sav[TM];
  fetch_scales<OUT, TM, TN>(ep, m_base, n_base, M, N, lane, sav, sbv);
  const int KT = K / BK;
  if constexpr (NST > 2) {
    // Slabs kt + 1 .. kt + NST - 1 are in flight while slab kt is multiplied.  At the end of slab kt: wait until only
    // the loads of the slabs after kt + 1 are outstanding, barrier (everyone's part of slab kt + 1 has landed, everyone
    // is done reading slab kt), and the stage of slab kt is requested again at the start of slab kt + 1.
    auto wait_for = [&](int newer) __attribute__((always_inline)) {  // `newer`: slabs requested after the awaited one
      static_assert((NST == 3 || NST == 4) && 2 * LOADS < 64, "wait counts are written out for three or four stages");
      // vmcnt is a six-bit field in two pieces: bits 3:0 and 15:14
      constexpr int W2 = 0x0F70 | ((2 * LOADS) & 0xF) | (((2 * LOADS) >> 4) << 14);
      constexpr int W1 = 0x0F70 | (LOADS & 0xF) | ((LOADS >> 4) << 14);
      if (newer >= 2) __builtin_amdgcn_s_waitcnt(W2);
      else if (newer == 1) __builtin_amdgcn_s_waitcnt(W1);
      else __builtin_amdgcn_s_waitcnt(0x0F70);
    };
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
      if (s < KT) issue_loads(s, s * BK);
    wait_for(min(KT - 1, NST - 2));
    __builtin_amdgcn_s_barrier();
    read_frags(0, 0, 0);
    int cur = 0;
    for (int kt = 0; kt < KT; ++kt) {
      const int nxt = cur + 1 == NST ? 0 : cur + 1;
      if (kt + NST - 1 < KT) issue_loads(cur == 0 ? NST - 1 : cur - 1, (kt + NST - 1) * BK);  // the stage of slab kt - 1
#pragma unroll
      for (int ks = 0; ks + 1 < NK; ++ks) {
        read_frags(cur, ks + 1, (ks + 1) & 1);
        mfma_step(ks & 1);
        hint_kstep(ks == 0 ? LOADS : 0);
      }
      mfma_step((NK - 1) & 1);
      if (kt + 1 < KT) {
        wait_for(min(KT - 1, kt + NST - 1) - (kt + 1));
        __builtin_amdgcn_s_barrier();
        read_frags(nxt, 0, 0);
      }
      cur = nxt;
    }
    staged_epilogue<OUT, EPI, TM, TN, NWAVES, NST * STAGE>(acc, sav, sbv, ep, m_base, n_base, M, N, out, ldo, smem, wave,
                                                             lane);
    return;
  }
  issue_loads(0, 0);
  __syncthreads();
  read_frags(0, 0, 0);
  // All loads of a slab are issued during its first k-step, giving them the rest of the slab to land.
  for (int kt = 0; kt < KT - 1; ++kt) {
    const int cur = kt & 1;
    issue_loads(cur ^ 1, (kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks + 1 < NK; ++ks) {
      read_frags(cur, ks + 1, (ks + 1) & 1);
      mfma_step(ks & 1);
      hint_kstep(ks == 0 ? LOADS : 0);
    }
    mfma_step((NK - 1) & 1);
    __syncthreads();
    read_frags(cur ^ 1, 0, 0);
  }
  {  // last slab: nothing left to fetch
    const int cur = (KT - 1) & 1;
#pragma unroll
    for (int ks = 0; ks + 1 < NK; ++ks) {
      read_frags(cur, ks + 1, (ks + 1) & 1);
      mfma_step(ks & 1);
    }
    mfma_step((NK - 1) & 1);
  }

  staged_epilogue<OUT, EPI, TM, TN, NWAVES, 2 * STAGE>(acc, sav, sbv, ep, m_base, n_base, M, N, out, ldo, smem, wave,
                                                         lane);
}

// ------------------------------------------------------------------------------------------------
// One tile row of at most 64 rows against a wide weight (a batch of decode tokens): the weight bytes dominate
// and every one of them is needed once.  A workgroup is NW (2 or 4) wavefronts side by side along N, each with all
// 32 * TM rows and 32 columns of its own; since no two wavefronts share a weight column, the weights go from
// global memory straight into registers (64 contiguous bytes per lane and slab, K permuted to match: lane
// half h holds bytes 64 h .. 64 h + 63 of the 128-byte slab row, and k-step s multiplies bytes 64 h + 16 s ..),
// while the activations go through LDS by direct-to-LDS loads as in the other kernels.  Both are fetched
// DEPTH - 1 slabs ahead (DEPTH LDS stages, DEPTH register sets; 8 in the build): a wavefront waits until all
// but its newest DEPTH - 2 groups of loads have landed (vmcnt counts in order; 6 groups of at most 6 loads stay
// under the counter's limit of 63), meets the others at a barrier, issues the group DEPTH - 1 slabs ahead into
// the stage the barrier has just freed, and multiplies.  Measured with weights from HBM, K 4096, N 14336,
// against the 128 x 128 two-stage tile and the weight-streaming kernel: 32 rows 26.2 / 36.6 / 26.1 us, 64 rows
// 26.6 / 36.8 / 48.0 us; 64 rows, K 8192, N 28672: 57.0 / 73.6 / 156.6 us (with four stages and compiler-
// tracked loads: 31.5 and 65.0 us for the two 64-row cases).  Workgroups of 64 columns then brought the 64-row
// case at N 14336 to 20.4 us and the 32-row case to 17.6 us.  With 128 rows every wavefront reads all 128
// activation rows from LDS per slab for its 32 columns, and a workgroup's stages take 96 KB, one workgroup per
// CU: that variant (six stages) pays while one round of 64-column workgroups covers N, and not under the
// ragged grid (64 groups of 128 rows: 232 against 228 us for the two-stage tile).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {  // vmcnt only: expcnt 7 and lgkmcnt 15 stay open
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

template <int QT, int OUT, int EPI, int TM, int DEPTH, int NW>
__device__ __forceinline__ void qgemm_mid_tile(const uint8_t* __restrict__ A, int64_t lda,
                                               const uint8_t* __restrict__ B, int64_t ldb, int m0, int n0, int M,
                                               int N, int K, const Epilogue& ep, uint8_t* __restrict__ out,
                                               int64_t ldo, int kshift) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  constexpr int BK = 128, TN = 1;  // TM: 32-row blocks of the tile; DEPTH: slabs of loads kept going, plus one
  constexpr int KSTEP = IS_INT ? 32 : 64;
  constexpr int NK = BK / KSTEP;
  constexpr int ASTAGE = 32 * TM * BK;  // 4 KB of activations per 32 rows and slab
  constexpr int PW = 4 * TM / NW;       // 1 KB pieces (8 rows) of a slab of activations that a wavefront fetches
  static_assert(PW * NW == 4 * TM, "the wavefronts share the activation rows evenly");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  using AccT = typename std::conditional<IS_INT, v16i, v16f>::type;
  using FragT = typename std::conditional<IS_INT, v4i, v8i>::type;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][0][r] = 0;

  const int m_base = m0, n_base = n0 + wave * 32;
  float sav[TM];
  float sbv[TN][4][4];
  fetch_scales<OUT, TM, TN>(ep, m_base, n_base, M, N, lane, sav, sbv);  // oldest loads: done before any slab

  // activations: 32 * TM rows of 128 bytes per slab = 4 * TM pieces of 1 KB (8 rows), PW per wavefront
  const int lr = lane >> 3;
  uint32_t aoff[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j)
    aoff[j] = static_cast<uint32_t>(min(m0 + (wave * PW + j) * 8 + lr, M - 1)) * static_cast<uint32_t>(lda) +
              (((lane & 7) ^ swz8((wave * PW + j) * 8 + lr)) << 4);
  // weights: column n_base + lane % 32, bytes 64 * (lane / 32) .. of the slab
  const int hx = lane >> 5, x7 = swz8(lane & 31);
  const uint32_t boff = static_cast<uint32_t>(min(n_base + (lane & 31), N - 1)) * static_cast<uint32_t>(ldb) + hx * 64;
  v4i breg[DEPTH][4];
  const int KT = K / BK;
  auto issue_group = [&](int kt, int st) {  // PW direct-to-LDS loads + 4 register loads per lane
    kt += kshift;  // this workgroup's first slab (below KT): the slabs are walked from there, wrapping around
    if (kt >= KT) kt -= KT;
    const uint8_t* ga = A + kt * BK;
#pragma unroll
    for (int j = 0; j < PW; ++j) QWIX_GLDS16_AT(ga, aoff[j], smem + st * ASTAGE + (wave * PW + j) * 1024);
    // Issued as asm so that the compiler does not track them: its own waits for these registers, merged over
    // the loop's back edge, come out as vmcnt(0) once per trip and would drain every load in flight.  The
    // explicit waits below are what guarantees that a register set has landed before it is multiplied.
    const uint8_t* gb = B + kt * BK;
    asm volatile("global_load_dwordx4 %0, %4, %5\n\t"
                 "global_load_dwordx4 %1, %4, %5 offset:16\n\t"
                 "global_load_dwordx4 %2, %4, %5 offset:32\n\t"
                 "global_load_dwordx4 %3, %4, %5 offset:48"
                 : "=&v"(breg[st][0]), "=&v"(breg[st][1]), "=&v"(breg[st][2]), "=&v"(breg[st][3])
                 : "v"(boff), "s"(gb)
                 : "memory");
  };
  const int a_row = (lane & 31) * BK;
  FragT fa[2][TM];
  auto read_a = [&](int st, int ks, int buf) {
    const uint8_t* base = smem + st * ASTAGE + a_row;
    if constexpr (IS_INT) {
      const int off = ((hx * 4 + ks) ^ x7) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[buf][i] = *reinterpret_cast<const v4i*>(base + i * 32 * BK + off);
    } else {
      const int off = ((hx * 4 + ks * 2) ^ x7) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(base + i * 32 * BK + off);
        const v4i hi = *reinterpret_cast<const v4i*>(base + i * 32 * BK + (off ^ 16));
        fa[buf][i] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < KT) issue_group(d, d);
  for (int kt0 = 0; kt0 < KT; kt0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int kt = kt0 + d;
      if (kt < KT) {  // the same for the whole workgroup
        // the groups after kt (PW + 4 loads each, at most DEPTH - 2 of them) may stay in flight
        constexpr int G = PW + 4;
        static_assert((DEPTH - 2) * G <= 63, "vmcnt is a 6-bit counter");
        static_assert(DEPTH >= 4 && DEPTH <= 8, "the wait below lists the cases");
        const int rem = KT - 1 - kt;
        __builtin_amdgcn_sched_barrier(0);
        switch (rem < DEPTH - 2 ? rem : DEPTH - 2) {
          case 0: wait_vmcnt<0>(); break;
          case 1: wait_vmcnt<G>(); break;
          case 2: wait_vmcnt<2 * G>(); break;
          case 3: wait_vmcnt<3 * G>(); break;
          case 4: wait_vmcnt<4 * G>(); break;
          case 5: wait_vmcnt<(5 * G < 63 ? 5 * G : 63)>(); break;  // 5, 6: not reached unless DEPTH is 7, 8
          default: wait_vmcnt<(6 * G < 63 ? 6 * G : 63)>(); break;
        }
        barrier();  // slab kt is in LDS from every wavefront, and everyone is done reading slab kt - 1
        // The compiler does not know that these registers were in flight until the wait above: pin them here, so
        // that no read or copy of them can be scheduled (or have been hoisted) in front of that wait.
#pragma unroll
        for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(breg[d][r]));
        if (kt + DEPTH - 1 < KT) issue_group(kt + DEPTH - 1, (d + DEPTH - 1) % DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        read_a(d, 0, 0);
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
          if (ks + 1 < NK) read_a(d, ks + 1, (ks + 1) & 1);
          FragT fb;
          if constexpr (IS_INT) {
            fb = breg[d][ks];
          } else {
            const v4i lo = breg[d][2 * ks], hi = breg[d][2 * ks + 1];
            fb = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          }
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            if constexpr (IS_INT)
              acc[i][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, fa[ks & 1][i], acc[i][0], 0, 0, 0);
            else
              acc[i][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb, fa[ks & 1][i], acc[i][0], 0, 0, 0, 0, 0, 0);
          }
        }
      }
    }
  }
  constexpr int kLds = DEPTH * ASTAGE > 20480 ? DEPTH * ASTAGE : 20480;  // the launch provides at least 20 KB
  staged_epilogue<OUT, EPI, TM, TN, NW, kLds>(acc, sav, sbv, ep, m_base, n_base, M, N, out, ldo, smem, wave,
                                                         lane);
}

// Byte offset of the scale that a lane touches: element `i` of `count`, `es` bytes each, or the last one.  What is read there is the
// element's first two bytes: a wider load would reach behind a vector of one bf16, and is misaligned where a group's scales start at an
// odd element.
constexpr int64_t scale_touch(int64_t i, int64_t count, int64_t es) { return (i < count ? i : count - 1) * es; }
static_assert(scale_touch(0, 1, 2) == 0 && scale_touch(127, 1, 2) == 0 && scale_touch(126, 3, 2) + 2 == 3 * 2 && scale_touch(2, 3, 4) + 4 == 3 * 4 &&
              scale_touch(int64_t{1} << 30, int64_t{1} << 31, 4) == int64_t{1} << 32, "every touch lies in its vector");

// ------------------------------------------------------------------------------------------------
// Ping-pong variant of the 256 x 256 kernel for long K.  The eight wavefronts form two groups (the
// upper and the lower 128 rows of the tile; the two wavefronts that share a SIMD are in different
// groups) that run half a slab out of phase: while one group is in its memory phase (read all
// fragments of a slab from LDS into registers, issue its direct-to-LDS loads of A), the other is in
// its compute phase (the slab's MFMAs back to back at raised priority, one load of B after each
// k-step), so the matrix pipe of every SIMD always has a wavefront that does little else.  Two
// workgroup barriers per slab keep the phases aligned; one extra barrier at the start of the lower
// group and at the end of the upper group produces the offset.
//   LDS: A in two stages of 32 KB, B in three (160 KB in all).  A wavefront loads 32 rows of A (its
// group's half) for the next slab and 32 rows of B for the slab after that; the third B stage is
// what makes room for loading B two slabs ahead, which gives those loads three phases to land and
// lets them be issued from the compute phase without a wait behind them.  Every load is waited for
// by the wavefront that issued it (vmcnt, oldest first) before the barrier that publishes it.
//   TM: the tile has 64 * TM rows (128, 192 or 256).  Per slab the LDS moves 176, 216 or 256 KB at 128 bytes a clock against 1024, 1536
// or 2048 clocks of MFMAs per SIMD, so lower tiles are bound by the LDS and cost more per row; they pay where they leave less of the
// chip idle in the last round, or less of a tile empty (pp_us).
template <int QT, int OUT, int EPI, int TM = 4>
__device__ __forceinline__ void qgemm_pp_tile(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B,
                                              int64_t ldb, int m0, int n0, int M, int N, int K, const Epilogue& ep,
                                              uint8_t* __restrict__ out, int64_t ldo) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  constexpr bool IS_BF = (QT == kOpBf16);
  constexpr bool B16 = IS_INT || IS_BF;  // 16 bytes per lane and k-step
  constexpr int BM = 64 * TM, BN = 256, BK = 128, WGN = 4;
  constexpr int TN = 2;                         // wave tile 32 * TM x 64
  constexpr int KSTEP = B16 ? 32 : 64, NK = BK / KSTEP;
  constexpr int A_STAGE = BM * BK, B_STAGE = BN * BK, B_BASE = 2 * A_STAGE;
  constexpr int LDS_BYTES = 2 * A_STAGE + 3 * B_STAGE;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;   // wm is also the phase group

  using AccT = typename std::conditional<IS_INT, v16i, v16f>::type;
  using FragT = typename std::conditional<B16, v4i, v8i>::type;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // ---- loader: this wavefront brings 8 * TM rows of its group's half of A and rows [wm*128 + wn*32, +32) of B, 8 rows per
  // instruction
  const int lr = lane >> 3;
  const int lrow0 = wm * 128 + wn * 32;
  const int arow0 = wm * (32 * TM) + wn * (8 * TM);
  uint32_t goffa[TM], goffb[4];
  const uint32_t lc = static_cast<uint32_t>((lane & 7) ^ swz8(lr));  // the row groups start at multiples of 8
#pragma unroll
  for (int j = 0; j < TM; ++j)
    goffa[j] = static_cast<uint32_t>(min(m0 + arow0 + j * 8 + lr, M - 1)) * static_cast<uint32_t>(lda) + lc * 16;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    goffb[j] = static_cast<uint32_t>(min(n0 + lrow0 + j * 8 + lr, N - 1)) * static_cast<uint32_t>(ldb) + lc * 16;
  }
  auto load_a = [&](int kt) {  // own half of the A rows of slab kt
    const uint8_t* gk = A + kt * BK;
    uint8_t* dst = smem + (kt & 1) * A_STAGE + arow0 * BK;
#pragma unroll
    for (int j = 0; j < TM; ++j) QWIX_GLDS16_AT_INPLACE(gk, goffa[j], dst + j * 1024);
  };
  auto load_b = [&](int kt, int stage) {  // own half of the B rows of slab kt
    const uint8_t* gk = B + kt * BK;
    uint8_t* dst = smem + B_BASE + stage * B_STAGE + lrow0 * BK;
#pragma unroll
    for (int j = 0; j < 4; ++j) QWIX_GLDS16_AT_INPLACE(gk, goffb[j], dst + j * 1024);
  };

  // ---- fragments of a whole slab
  const int a_row = (wm * (32 * TM) + (lane & 31)) * BK;
  const int b_row = B_BASE + (wn * 64 + (lane & 31)) * BK;
  const int hx = lane >> 5, x7 = swz8(lane & 31);
  FragT fa[NK][TM], fb[NK][TN];
  auto read_slab = [&](int a_stage, int b_stage) {
    const uint8_t* pa = smem + a_stage * A_STAGE + a_row;
    const uint8_t* pb = smem + b_stage * B_STAGE + b_row;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      if constexpr (B16) {
        const int off = ((ks * 2 + hx) ^ x7) << 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[ks][i] = *reinterpret_cast<const v4i*>(pa + i * 32 * BK + off);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[ks][j] = *reinterpret_cast<const v4i*>(pb + j * 32 * BK + off);
      } else {
        const int off = ((ks * 4 + hx * 2) ^ x7) << 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const v4i lo = *reinterpret_cast<const v4i*>(pa + i * 32 * BK + off);
          const v4i hi = *reinterpret_cast<const v4i*>(pa + i * 32 * BK + (off ^ 16));
          fa[ks][i] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const v4i lo = *reinterpret_cast<const v4i*>(pb + j * 32 * BK + off);
          const v4i hi = *reinterpret_cast<const v4i*>(pb + j * 32 * BK + (off ^ 16));
          fb[ks][j] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
    }
  };
  // s_waitcnt on vmcnt only (expcnt 7, lgkmcnt 15 stay open): all but the newest `left` direct-to-LDS
  // loads of this wavefront have landed
  auto wait_loads = [&](auto left) { __builtin_amdgcn_s_waitcnt(0x0F70 | decltype(left)::value); };
  using None = std::integral_constant<int, 0>;
  using NewA = std::integral_constant<int, TM>;
  using NewB = std::integral_constant<int, 4>;
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  const int KT = K / BK;  // >= 2
  // The scale vectors are first needed in the epilogue, where a cold fetch (address translation plus a trip
  // to HBM) would stall every wavefront with nothing to hide behind.  Touch this wavefront's pieces of them
  // now, under the equally cold first slab loads: every second of up to 128 row scales, each of 64 column scales.
  uint32_t warm_a = 0, warm_b = 0;
  if constexpr (OUT != QWIX_I32) {
    if (ep.sa != nullptr)
      warm_a = *reinterpret_cast<const uint16_t*>(static_cast<const uint8_t*>(ep.sa) +
                                                  scale_touch(m0 + wm * (32 * TM) + 2 * lane, M, ep.sa_dtype == QWIX_BF16 ? 2 : 4));
    if (ep.sb != nullptr)
      warm_b = *reinterpret_cast<const uint16_t*>(static_cast<const uint8_t*>(ep.sb) +
                                                  scale_touch(n0 + wn * 64 + lane, N, ep.sb_dtype == QWIX_BF16 ? 2 : 4));
  }
  // ---- prologue: A of slab 0, B of slabs 0 and 1 (each wavefront its rows)
  load_a(0);
  load_b(0, 0);
  load_b(1, 1);
  wait_loads(None{});
  asm volatile("" ::"v"(warm_a), "v"(warm_b));  // the touches above have landed too; their values are not used
  barrier();
  if (wm == 1) barrier();  // the lower group starts half a slab late

  // B is loaded two slabs ahead, during the compute phase, one load after each k-step's MFMAs (those
  // loads have three phases to land); A one slab ahead, in the memory phase.  The waits before the
  // barriers leave the loads just issued in flight and cover those issued one phase earlier.
  int bst = 0;  // B stage of slab kt = kt % 3
  // One slab; whether A of the next slab and B of the one after it are still to be requested is known at compile time,
  // so that the steady state is one basic block (a branch would end the scheduling regions that the fences below
  // delimit): the loop runs the slabs that request both, the last two slabs follow it.
  auto slab = [&](int kt, auto more_a_tag, auto more_b_tag) __attribute__((always_inline)) {
    constexpr bool more_a = decltype(more_a_tag)::value, more_b = decltype(more_b_tag)::value;
    // memory phase
    read_slab(kt & 1, bst);
    __builtin_amdgcn_sched_barrier(0);  // fragment reads first: the loads below may not slip in front of them
    if constexpr (more_a) {
      load_a(kt + 1);
      wait_loads(NewA{});
    } else {
      wait_loads(None{});
    }
    barrier();
    // compute phase
    const int bst2 = bst == 0 ? 2 : bst - 1;  // (kt + 2) % 3
    const uint8_t* gkb = B + (kt + 2) * BK;
    uint8_t* dstb = smem + B_BASE + bst2 * B_STAGE + lrow0 * BK;
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (IS_INT)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ks][j], fa[ks][i], acc[i][j], 0, 0, 0);
          else if constexpr (IS_BF)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb[ks][j]),
                                                                __builtin_bit_cast(bf16x8, fa[ks][i]), acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[ks][j], fa[ks][i], acc[i][j], 0, 0, 0, 0, 0, 0);
        }
      if constexpr (more_b) {
#pragma unroll
        for (int j = ks * (4 / NK); j < (ks + 1) * (4 / NK); ++j) QWIX_GLDS16_AT_INPLACE(gkb, goffb[j], dstb + j * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    if constexpr (more_b) wait_loads(NewB{}); else wait_loads(None{});
    barrier();
    bst = bst == 2 ? 0 : bst + 1;
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  int kt = 0;
  for (; kt + 2 < KT; ++kt) slab(kt, T_{}, T_{});
  if (kt + 1 < KT) {
    slab(kt, T_{}, F_{});
    ++kt;
  }
  slab(kt, F_{}, F_{});
  if (wm == 0) barrier();

  const int m_base = m0 + wm * (32 * TM), n_base = n0 + wn * 64;
  float sav[TM];
  float sbv[TN][4][4];
  fetch_scales<OUT, TM, TN>(ep, m_base, n_base, M, N, lane, sav, sbv);
  staged_epilogue<OUT, EPI, TM, TN, 8, LDS_BYTES>(acc, sav, sbv, ep, m_base, n_base, M, N, out, ldo, smem, wave, lane);
}

// us that `tiles` ping-pong tiles of 64 * tm rows take over K, one tile per CU at a time: a round's start and end, and its slabs, which
// cost more the more CUs are at work (clock, L2).  Fitted to 130 dense and 130 ragged shapes, int8 and e4m3, weights from HBM: the
// choice it makes is within 1 % (dense) and 2 % (ragged, sizes unknown) of the best of the three on average.
inline double pp_us(int tm, double tiles, int64_t K) {
  const double ends = 3.0 + tm, fixed = tm == 2 ? 0.44 : tm == 3 ? 0.55 : 0.64, busy = tm == 2 ? 0.5 : tm == 3 ? 0.65 : 0.8;
  const double slabs = static_cast<double>(K / 128), rounds = tiles / 256.0;
  const double full = static_cast<double>(static_cast<int64_t>(rounds + 1e-9)), rest = rounds - full;
  return full * (ends + slabs * (fixed + busy)) + (rest > 1e-6 ? ends + slabs * (fixed + busy * rest) : 0.0);
}

// ------------------------------------------------------------------------------------------------
// Ragged GEMM (mixture-of-experts): the rows of A are split into consecutive groups whose sizes are
// read from device memory; the rows of group g meet B_g, the g-th (N, K) panel.  Rows that belong
// to no group (past the sum of the sizes) come out as zeros.  No host synchronisation: the grid
// is sized for the worst case, floor(M / BM) + G + 1 tile rows, and every workgroup finds its
// tile by walking the group sizes (wave-uniform scalar work); workgroups past the last tile exit.
struct Ragged {
  const int32_t* group_sizes;  // G entries
  int G;
  int skip;                 // groups of up to this many rows have no tiles here (another launch does them)
  int64_t b_group_stride;   // bytes between consecutive B panels
  int64_t sb_group_stride;  // elements between the rhs scale vectors of consecutive groups (0: one shared vector)
};

constexpr int kRaggedChunk = 16;  // consecutive tile ids that run on one XCD

// Inclusive scan over the 64 lanes of a wavefront, x = min(x + y, most) (most < 2^31): six DPP adds.
__device__ __forceinline__ uint32_t scan_add(uint32_t x, uint32_t most) {
#define QWIX_SCAN_STEP(ctrl, rows) \
  x = min(x + static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), ctrl, rows, 0xF, false)), most)
  QWIX_SCAN_STEP(0x111, 0xF);  // row_shr:1, 2, 4, 8: inside the rows of 16 lanes
  QWIX_SCAN_STEP(0x112, 0xF);
  QWIX_SCAN_STEP(0x114, 0xF);
  QWIX_SCAN_STEP(0x118, 0xF);
  QWIX_SCAN_STEP(0x142, 0xA);  // row_bcast:15: rows 1 and 3
  QWIX_SCAN_STEP(0x143, 0xC);  // row_bcast:31: rows 2 and 3
#undef QWIX_SCAN_STEP
  return x;
}

// Returns 0: no tile, 1: a tile of group *g, 2: a tile of rows that belong to no group.
// Tile ids are numbered group by group; inside a group they walk 8 tile rows per column so that
// tiles that run together share operand panels.  Runs of kRaggedChunk ids are dealt out to the 8
// XCDs in turn, which also spreads the unused ids at the end over all of them.
// Every wavefront looks at 64 groups at once, a lane each: two scans (rows, tiles) and a ballot.  A walk from group to group
// is a chain of scalar loads, 0.17 us each in front of every tile (two rounds of tiles behind 64 groups: 90 us, scanned 65 us).
template <int BM, int BN>
__device__ __forceinline__ int ragged_tile(const Ragged& rg, int M, int N, int* g, int* m0, int* m_lim, int* n0) {
  int pid = blockIdx.x;  // gridDim.x % (8 * kRaggedChunk) == 0
  {
    const int k = pid >> 3, x = pid & 7;
    pid = ((k / kRaggedChunk) * 8 + x) * kRaggedChunk + k % kRaggedChunk;
  }
  const int tiles_n = (N + BN - 1) / BN;
  const int lane = threadIdx.x & 63;
  int row = 0, first = 0;  // rows and tiles of the groups before this chunk
  int start, size, before;
  int found = -1;
  for (int base = 0; base < rg.G; base += 64) {
    // sizes are clamped so that no group reaches past row M
    const int want = base + lane < rg.G ? min(max(rg.group_sizes[base + lane], 0), M) : 0;
    const int end = static_cast<int>(min(scan_add(want, M) + row, static_cast<uint32_t>(M)));
    const int prev = __shfl_up(end, 1, 64);
    start = lane == 0 ? row : prev;
    size = end - start;
    const int cnt = size > rg.skip ? (size + BM - 1) / BM * tiles_n : 0;
    const int last = first + static_cast<int>(scan_add(cnt, INT32_MAX));
    before = last - cnt;
    const uint64_t here = __ballot(pid >= before && pid < last);
    if (here != 0) {
      const int l = __builtin_ctzll(here);
      found = base + l;
      start = __builtin_amdgcn_readlane(start, l);
      size = __builtin_amdgcn_readlane(size, l);
      before = __builtin_amdgcn_readlane(before, l);
      break;
    }
    row = __builtin_amdgcn_readlane(end, 63);
    first = __builtin_amdgcn_readlane(last, 63);
  }
  if (found < 0) {  // the rows left over
    start = row;
    size = M - row;
    before = first;
    if (pid >= before + (size + BM - 1) / BM * tiles_n) return 0;
  }
  const int nt = (size + BM - 1) / BM;
  constexpr int GM = 8;
  const int r = pid - before, per = GM * tiles_n;
  const int fm = (r / per) * GM, gsz = min(nt - fm, GM);
  *g = found;
  *m0 = start + (fm + (r % per) % gsz) * BM;
  *m_lim = start + size;
  *n0 = ((r % per) / gsz) * BN;
  return found < 0 ? 2 : 1;
}

template <int BM, int BN, typename OutT>
__device__ __forceinline__ void zero_tile(uint8_t* out, int64_t ldo, int m0, int m_lim, int n0, int N, int nthreads) {
  const int rows = min(BM, m_lim - m0), cols = min(BN, N - n0);
  for (int idx = threadIdx.x; idx < rows * cols; idx += nthreads)
    reinterpret_cast<OutT*>(out)[static_cast<int64_t>(m0 + idx / cols) * ldo + n0 + idx % cols] = 0;
}

__device__ __forceinline__ Epilogue group_epilogue(const Epilogue& ep, const Ragged& rg, int g) {
  Epilogue e = ep;
  if (ep.sb != nullptr)
    e.sb = static_cast<const uint8_t*>(ep.sb) + g * rg.sb_group_stride * (ep.sb_dtype == QWIX_BF16 ? 2 : 4);
  return e;
}

inline unsigned ragged_grid(int64_t M, int64_t N, int64_t G, int BM, int BN) {
  const int64_t tiles = (M / BM + G + 1) * ((N + BN - 1) / BN);
  const int64_t unit = 8 * kRaggedChunk;
  return static_cast<unsigned>((tiles + unit - 1) / unit * unit);
}

// ------------------------------------------------------------------------------------------------
// Skinny GEMM (decode: a handful of tokens against a whole weight matrix).  The 128 x 128 tiles of
// the kernels above would leave most CUs idle and most MFMA rows empty; here the weight matrix is
// streamed exactly once: a workgroup owns NT tiles of 16 output columns, its 16 wavefronts split
// K, each with two 128-byte blocks of loads in flight, and the int32 (or f32) partial tiles meet
// in LDS.  int8: v_mfma_i32_16x16x64_i8, a lane holds 32 consecutive k of one row (two MFMAs);
// e4m3: one v_mfma_f32_16x16x128_f8f6f4.  The int32 sum does not depend on the split, so results
// are bit-identical to the tiled kernels'; the epilogue is the same rounding chain.
typedef int v8i_s __attribute__((ext_vector_type(8)));
typedef float v4f_s __attribute__((ext_vector_type(4)));
constexpr int kSkinnyWaves = 16;

// One 16-row block of the weight-streaming GEMM: rows row0 .. row0 + 15 (below M) against columns n_base ..
// n_base + 16 * NT - 1, by a workgroup of WAVES wavefronts that split K.
template <int QT, int NT, int WAVES = kSkinnyWaves>
__device__ __forceinline__ void skinny_block(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B,
                                             int64_t ldb, int row0, int M, int n_base, int N, int K, const Epilogue& ep,
                                             uint8_t* __restrict__ out, int64_t ldo) {
  constexpr bool IS_INT = (QT == QWIX_INT8);
  using AccT = typename std::conditional<IS_INT, v4i, v4f_s>::type;
  __shared__ AccT red[WAVES][NT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const int nblk = K / 128;
  const int per_wave = (nblk + WAVES - 1) / WAVES;
  // Which slice of K a wavefront takes rotates with the workgroup: in step, all workgroups would ask the same few
  // memory channels for the same K offset of their rows at the same time (4096 x 14336 int8, 16 rows: 14.5 -> 13.9 us).
  const int slice = (wave + static_cast<int>(blockIdx.x)) % WAVES;
  const int kb0 = min(nblk, slice * per_wave), kb1 = min(nblk, kb0 + per_wave);

  // wave-uniform bases + fixed 32-bit lane offsets; rows of A past M and columns past N are clamped
  const uint8_t* a_base = A + static_cast<int64_t>(row0) * lda;
  const uint8_t* b_base = B + static_cast<int64_t>(n_base) * ldb;
  const uint32_t a_off = static_cast<uint32_t>(min(col, M - 1 - row0)) * static_cast<uint32_t>(lda) + kq * 32;
  uint32_t b_off[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    b_off[t] = static_cast<uint32_t>(min(t * 16 + col, N - 1 - n_base)) * static_cast<uint32_t>(ldb) + kq * 32;

  AccT acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[t][r] = 0;

  struct Blk {
    v4i x[2];
    v4i w[NT][2];
  };
  auto load_blk = [&](int kb, Blk* b) {
    const uint8_t* ap = a_base + kb * 128 + a_off;
    b->x[0] = *reinterpret_cast<const v4i*>(ap);
    b->x[1] = *reinterpret_cast<const v4i*>(ap + 16);
    const uint8_t* bp = b_base + kb * 128;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      b->w[t][0] = *reinterpret_cast<const v4i*>(bp + b_off[t]);
      b->w[t][1] = *reinterpret_cast<const v4i*>(bp + b_off[t] + 16);
    }
  };
  auto compute_blk = [&](const Blk& b) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (IS_INT) {
        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b.x[0], b.w[t][0], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b.x[1], b.w[t][1], acc[t], 0, 0, 0);
      } else {
        const v8i_s xa = {b.x[0][0], b.x[0][1], b.x[0][2], b.x[0][3], b.x[1][0], b.x[1][1], b.x[1][2], b.x[1][3]};
        const v8i_s wb = {b.w[t][0][0], b.w[t][0][1], b.w[t][0][2], b.w[t][0][3],
                          b.w[t][1][0], b.w[t][1][1], b.w[t][1][2], b.w[t][1][3]};
        acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(xa, wb, acc[t], 0, 0, 0, 0, 0, 0);
      }
    }
  };
  for (int kb = kb0; kb < kb1; kb += 2) {
    Blk b0, b1;
    const bool two = kb + 1 < kb1;
    load_blk(kb, &b0);
    if (two) load_blk(kb + 1, &b1);
    compute_blk(b0);
    if (two) compute_blk(b1);
  }

#pragma unroll
  for (int t = 0; t < NT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  // result lane layout: column n = lane % 16, row m = 4 * (lane / 16) + r
  const bool r0 = ep.r0 != 0, r1 = ep.r1 != 0, r2 = ep.r2 != 0;
  for (int idx = tid; idx < NT * 256; idx += WAVES * 64) {
    const int t = idx >> 8, r = (idx >> 6) & 3, l = idx & 63;
    const int m = row0 + 4 * (l >> 4) + r, n = n_base + t * 16 + (l & 15);
    if (m >= M || n >= N) continue;
    float v;
    if constexpr (IS_INT) {
      int a = 0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) a += red[w][t][l][r];
      if (ep.out_dtype == QWIX_I32) {
        reinterpret_cast<int*>(out)[static_cast<int64_t>(m) * ldo + n] = a;
        continue;
      }
      if (ep.zu != nullptr) a -= zu_at(ep, m) * ep.zv[n];
      v = static_cast<float>(a);
    } else {
      v = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += red[w][t][l][r];
    }
    if (r0) v = round_bf16(v);
    if (ep.sa != nullptr) v *= load_scale(ep.sa, ep.sa_dtype, m);
    if (r1) v = round_bf16(v);
    if (ep.sb != nullptr) v *= load_scale(ep.sb, ep.sb_dtype, n);
    if (r2) v = round_bf16(v);
    if (ep.out_dtype == QWIX_BF16)
      reinterpret_cast<uint16_t*>(out)[static_cast<int64_t>(m) * ldo + n] = f32_to_bf16_bits(v);
    else
      reinterpret_cast<float*>(out)[static_cast<int64_t>(m) * ldo + n] = v;
  }
}

// Dtype chain of the reference epilogue: int32 adopts the first scale's dtype (through f32); a
// float accumulator starts in acc_dtype; each multiply happens in the promotion of both sides.
static Epilogue make_epilogue(int qtype, const void* sa, int sa_dtype, const void* sb, int sb_dtype, int acc_dtype,
                              const void* zu, const int32_t* zv, int out_dtype, bool zu8 = false) {
  Epilogue ep{sa, sb, sa_dtype, sb_dtype, out_dtype, 0, 0, 0, zu8, zu, zv};
  int cur = (qtype == QWIX_INT8) ? QWIX_I32 : acc_dtype;
  if (cur == QWIX_BF16) ep.r0 = 1;
  auto step = [&](const void* s, int s_dtype, auto& r_after) {
    if (!s) return;
    const int t = (cur == QWIX_I32) ? s_dtype : ((cur == QWIX_F32 || s_dtype == QWIX_F32) ? QWIX_F32 : QWIX_BF16);
    if (cur == QWIX_I32 && t == QWIX_BF16) ep.r0 = 1;
    r_after = (t == QWIX_BF16);
    cur = t;
  };
  step(sa, sa_dtype, ep.r1);
  step(sb, sb_dtype, ep.r2);
  return ep;
}

// Argument checks shared by the dense and the ragged entry points.
static int check_gemm_args(const void* a, int64_t lda, const void* b, int64_t ldb, int qtype, int64_t M, int64_t N,
                           int64_t K, const void* sa, int sa_dtype, const void* sb, int sb_dtype, int acc_dtype,
                           const void* out, int out_dtype, int64_t ldo) {
  if (!a || !b || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null a/b/out");
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad GEMM shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
                (long long)K);
  if (qtype != QWIX_INT8 && qtype != QWIX_E4M3)
    return fail(QWIX_ERR_UNSUPPORTED, "qgemm supports int8 x int8 and e4m3 x e4m3 operands (got qtype %d)", qtype);
  if (K % 16 || lda % 16 || ldb % 16 || lda < K || ldb < K || !aligned16(a) || !aligned16(b))
    return fail(QWIX_ERR_UNSUPPORTED, "K, lda, ldb must be multiples of 16 bytes and a/b 16-byte aligned "
                "(K=%lld lda=%lld ldb=%lld)", (long long)K, (long long)lda, (long long)ldb);
  if (ldo < N || !aligned16(out) || (N % 4 == 0 && ldo % 4 != 0))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad output leading dimension %lld for N=%lld", (long long)ldo, (long long)N);
  auto ok_s = [](int d) { return d == QWIX_F32 || d == QWIX_BF16; };
  if ((sa && !ok_s(sa_dtype)) || (sb && !ok_s(sb_dtype)))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "scale dtypes must be f32 or bf16");
  if (out_dtype == QWIX_I32 && qtype != QWIX_INT8)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "raw int32 accumulators exist for int8 operands only");
  if (out_dtype != QWIX_I32 && !ok_s(out_dtype)) return fail(QWIX_ERR_INVALID_ARGUMENT, "bad out dtype %d", out_dtype);
  if (qtype == QWIX_E4M3 && !ok_s(acc_dtype)) return fail(QWIX_ERR_INVALID_ARGUMENT, "bad accumulator dtype %d", acc_dtype);
  return QWIX_OK;
}

// out[m, n] = epilogue(sum over splits of ws[s][m][n]); four consecutive elements of the flattened (m, n) per thread.
template <bool IS_INT>
__global__ void __launch_bounds__(256)
    splitk_reduce_kernel(const uint8_t* __restrict__ ws, int splits, int M, int N, Epilogue ep, uint8_t* __restrict__ out,
                         int64_t ldo) {
  const int64_t total = static_cast<int64_t>(M) * N;
  const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (i0 >= total) return;
  const bool vec = (N & 3) == 0;  // then the four share a row and the loads are 16-byte aligned
  float v[4];
  // Eight partials are requested before the first is added: one trip to memory per eight splits, not per split.
  // They are added in split order (int32 sums do not depend on it; the f32 sums of e4m3 partials do).
  constexpr int kBatch = 8;
  if constexpr (IS_INT) {
    int a[4] = {0, 0, 0, 0};
    for (int s0 = 0; s0 < splits; s0 += kBatch) {
      if (vec) {
        int4 w[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          w[j] = make_int4(0, 0, 0, 0);
          if (s0 + j < splits) w[j] = *reinterpret_cast<const int4*>(reinterpret_cast<const int*>(ws) + (s0 + j) * total + i0);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) { a[0] += w[j].x; a[1] += w[j].y; a[2] += w[j].z; a[3] += w[j].w; }
      } else {
        for (int s = s0; s < min(splits, s0 + kBatch); ++s) {
          const int* p = reinterpret_cast<const int*>(ws) + s * total + i0;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (i0 + e < total) a[e] += p[e];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = static_cast<float>(a[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = 0.f;
    for (int s0 = 0; s0 < splits; s0 += kBatch) {
      if (vec) {
        float4 w[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          w[j] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (s0 + j < splits) w[j] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(ws) + (s0 + j) * total + i0);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          if (s0 + j < splits) { v[0] += w[j].x; v[1] += w[j].y; v[2] += w[j].z; v[3] += w[j].w; }
        }
      } else {
        for (int s = s0; s < min(splits, s0 + kBatch); ++s) {
          const float* p = reinterpret_cast<const float*>(ws) + s * total + i0;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (i0 + e < total) v[e] += p[e];
        }
      }
    }
  }
  const bool r0 = ep.r0 != 0, r1 = ep.r1 != 0, r2 = ep.r2 != 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t i = i0 + e;
    if (i >= total) break;
    const int m = static_cast<int>(i / N), n = static_cast<int>(i % N);
    float t = v[e];
    if (r0) t = round_bf16(t);
    if (ep.sa != nullptr) t *= load_scale(ep.sa, ep.sa_dtype, m);
    if (r1) t = round_bf16(t);
    if (ep.sb != nullptr) t *= load_scale(ep.sb, ep.sb_dtype, n);
    if (r2) t = round_bf16(t);
    if (ep.out_dtype == QWIX_BF16)
      reinterpret_cast<uint16_t*>(out)[static_cast<int64_t>(m) * ldo + n] = f32_to_bf16_bits(t);
    else
      reinterpret_cast<float*>(out)[static_cast<int64_t>(m) * ldo + n] = t;
  }
}

}  // namespace
}  // namespace qwix
