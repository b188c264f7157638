// Batched quantized GEMM with a short contraction (K = 64 or 128: attention scores), int8 or e4m3.
//
//   out[z][m, n] = ((T(sum_k a[z][m, k] b[z][n, k]) * sa[z][m]) * sb[z][n])
//
// Bound by writing the result: 32 x 2048 x 2048 x 128 has 17 MB of operands and 268 MB of bf16 scores.  A tile of its own
// per workgroup is load, multiply, store, one after the other, with nothing of the same workgroup to put in between.  Here a
// workgroup keeps the fragments of a strip of rows in registers and walks along the columns: the next columns' fragments
// are requested before the current ones are multiplied, and the stores of one step drain under the following ones.
// The four wavefronts of a workgroup stand side by side, 64 columns each, or two by two; a wavefront reads its columns' rows of b straight
// into registers (16 rows x 64 bytes per instruction, b stays in L2), and turns its 16 RT x 64 results through a piece of
// LDS of its own into whole 128-byte row pieces: no barrier anywhere.
// Measured at the shape above: see launch_strips.
#include "common.h"
#include "qgemm_strips.h"

namespace qwix {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Sixteen KS bf16 values of a row in each of the four lanes lane % 16 + 16 {0, 1, 2, 3}, raw[k] the 64-value step's: the row's absmax
// scale and its codes, rounded as the quantization of rows rounds them (rows_kernel).
template <int QT, int KS>
__device__ __forceinline__ float quantize_row(const v4u (&raw)[KS][2], v4i (&code)[KS]) {
  // |x| as a key that orders as the value does and puts NaN below everything (15 bits of |x|; adding 0x7F turns exactly the NaNs negative)
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  s16x2 m = {0x7F, 0x7F};
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m = __builtin_elementwise_max(m, __builtin_bit_cast(s16x2, (raw[k][h][e] & 0x7FFF7FFFu) + 0x007F007Fu));
  float mx = bf16_bits_to_f32(static_cast<uint16_t>((m[0] > m[1] ? m[0] : m[1]) - 0x7F));
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  const float s = sym_scale<BF16, QT>(mx);
  const Divider<BF16, false, false> div(s);
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int w = 0; w < 4; ++w) {  // four codes from two words
      const uint32_t x0 = raw[k][w / 2][2 * (w % 2)], x1 = raw[k][w / 2][2 * (w % 2) + 1];
      float t[4] = {__uint_as_float(x0 << 16), __uint_as_float(x0 & 0xFFFF0000u), __uint_as_float(x1 << 16), __uint_as_float(x1 & 0xFFFF0000u)};
      div.pair_unsigned(t[0], t[1]);
      div.pair_unsigned(t[2], t[3]);
      if constexpr (QT == QWIX_INT8)
        code[k][w] = static_cast<int>(pack4_low_bytes(rne_bits_clamped(t[0], -128.f, 127.f), rne_bits_clamped(t[1], -128.f, 127.f),
                                                      rne_bits_clamped(t[2], -128.f, 127.f), rne_bits_clamped(t[3], -128.f, 127.f)));
      else  // (the sign of a zero quotient is its dividend's)
        code[k][w] = static_cast<int>((__builtin_amdgcn_perm(x1, x0, 0x07050301u) & 0x80808080u) |
                                      ((to_e4m3x2_bounded(t[0], t[1]) | (to_e4m3x2_bounded(t[2], t[3]) << 16)) & 0x7F7F7F7Fu));
    }
  return s;
}

// KS: K / 64.  RT: tiles of 16 rows per wavefront.  WR: wavefronts of the workgroup below each other.  BF: bf16 scales and results with every step of the chain rounded to bf16;
// otherwise f32 throughout.  ACT: a and b hold bf16 values, quantized per row
// right behind their loads; the rows of b once per strip, so this is for problems of one strip.
template <int QT, int KS, int RT, int WR, bool BF, bool ACT>
__global__ void __launch_bounds__(256, BF && !ACT ? 4 : 2)
    qgemm_strips_kernel(StripArgs p, int strips, int cols, bool nt) {
  constexpr bool IS_INT = QT == QWIX_INT8;
  constexpr int ES = BF ? 2 : 4, PITCH = 64 * ES + 16, ROWS = 16 * RT;
  using Acc = typename std::conditional<IS_INT, v4i, v4f>::type;
  __shared__ __attribute__((aligned(16))) uint8_t stage_all[4 * ROWS * PITCH];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* const stage = stage_all + wave * (ROWS * PITCH);
  const int z = blockIdx.y;
  const int wr = wave % WR, wc = wave / WR;
  constexpr int CSTEP = 64 * (4 / WR);
  const int m0 = (static_cast<int>(blockIdx.x % static_cast<unsigned>(strips)) * WR + wr) * ROWS;
  const int n_begin = static_cast<int>(blockIdx.x / static_cast<unsigned>(strips)) * cols;
  const int n_end = min(n_begin + cols, p.N);
  const int l16 = lane & 15, l4 = lane >> 4;
  const uint8_t* A = p.a + z * p.a_stride;
  const uint8_t* B = p.b + z * p.b_stride;
  const uint8_t* SB = static_cast<const uint8_t*>(p.sb) + z * p.sb_stride * ES;
  const auto rout = __builtin_amdgcn_make_buffer_rsrc(p.out + z * p.out_stride * ES, 0,
                                                      static_cast<int>(static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.ldo) * ES),
                                                      0x00020000);

  // Operand lane layout: row lane % 16, bytes 16 (lane / 16) .. of each 64-byte step; the same K order on both sides.
  v4i fa[RT][KS];
  float sa[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = min(m0 + i * 16 + l16, p.M - 1);
    if constexpr (ACT) {
      v4u raw[KS][2];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          raw[k][h] = *reinterpret_cast<const v4u*>(A + static_cast<int64_t>(m) * p.lda + k * 128 + l4 * 32 + h * 16);
      sa[i] = quantize_row<QT, KS>(raw, fa[i]);
    } else {
#pragma unroll
      for (int k = 0; k < KS; ++k) fa[i][k] = *reinterpret_cast<const v4i*>(A + static_cast<int64_t>(m) * p.lda + k * 64 + l4 * 16);
      sa[i] = load1<typename std::conditional<BF, BF16, F32>::type>(p.sa, z * p.sa_stride + m);
    }
  }

  // 32 columns: two tiles of 16, with the four scales of a lane's four consecutive columns in each
  struct Cols {
    v4i b[2][KS];
    uint32_t s[2][BF ? 2 : 4];
    v4u raw[ACT ? 2 : 1][KS][2];
  };
  auto load = [&](Cols& c, int n) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // 32-bit offsets from a uniform base (a problem's b is below 2 GiB)
      const uint32_t row = static_cast<uint32_t>(min(n + j * 16 + l16, p.N - 1)) * static_cast<uint32_t>(p.ldb) + l4 * (ACT ? 32 : 16);
      if constexpr (ACT) {
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
          for (int h = 0; h < 2; ++h) c.raw[j][k][h] = *reinterpret_cast<const v4u*>(B + k * 128 + h * 16 + row);
      } else {
#pragma unroll
        for (int k = 0; k < KS; ++k) c.b[j][k] = *reinterpret_cast<const v4i*>(B + k * 64 + row);
        const uint8_t* sp = SB + static_cast<uint32_t>(min(n + j * 16 + 4 * l4, p.N - 4)) * ES;
        if constexpr (BF) {
          const uint2 w = *reinterpret_cast<const uint2*>(sp);
          c.s[j][0] = w.x;
          c.s[j][1] = w.y;
        } else {
          const uint4 w = *reinterpret_cast<const uint4*>(sp);
          c.s[j][0] = w.x; c.s[j][1] = w.y; c.s[j][2] = w.z; c.s[j][3] = w.w;
        }
      }
    }
  };
  auto encode = [&](Cols& c) {
    if constexpr (ACT) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int s = static_cast<int>(__float_as_uint(quantize_row<QT, KS>(c.raw[j], c.b[j])) >> 16);  // a bf16: lane % 16 is its column
#pragma unroll
        for (int h = 0; h < 2; ++h)
          c.s[j][h] = static_cast<uint32_t>(__shfl(s, 4 * l4 + 2 * h, 64)) | static_cast<uint32_t>(__shfl(s, 4 * l4 + 2 * h + 1, 64)) << 16;
      }
    }
  };
  auto multiply = [&](const Cols& c, int half) {
    // v[r]: row 16 i + lane % 16, column 16 j + 4 (lane / 16) + r
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        Acc v = {0, 0, 0, 0};
        if constexpr (IS_INT) {
#pragma unroll
          for (int k = 0; k < KS; ++k) v = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.b[j][k], fa[i][k], v, 0, 0, 0);
        } else {
          v8i x = {0, 0, 0, 0, 0, 0, 0, 0}, y = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
          for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[4 * k + e] = c.b[j][k][e];
              y[4 * k + e] = fa[i][k][e];
            }
          v = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, v, 0, 0, 0, 0, 0, 0);
        }
        uint8_t* dst = stage + (i * 16 + l16) * PITCH + (half * 32 + j * 16 + 4 * l4) * ES;
        if constexpr (BF) {
          uint32_t w[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            uint32_t pk = pack_bf16x2(static_cast<float>(v[2 * h]), static_cast<float>(v[2 * h + 1]));
            pk = pack_bf16x2(__uint_as_float(pk << 16) * sa[i], __uint_as_float(pk & 0xFFFF0000u) * sa[i]);
            w[h] = pack_bf16x2(__uint_as_float(pk << 16) * __uint_as_float(c.s[j][h] << 16),
                               __uint_as_float(pk & 0xFFFF0000u) * __uint_as_float(c.s[j][h] & 0xFFFF0000u));
          }
          *reinterpret_cast<qwix_v2i*>(dst) = qwix_v2i{static_cast<int>(w[0]), static_cast<int>(w[1])};
        } else {
          v4i w;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            w[r] = static_cast<int>(__float_as_uint(static_cast<float>(v[r]) * sa[i] * __uint_as_float(c.s[j][r])));
          *reinterpret_cast<v4i*>(dst) = w;
        }
      }
  };

  constexpr int CPR = 64 * ES / 16;  // 16-byte chunks per staged row
  const uint32_t row_step = static_cast<uint32_t>(64 / CPR) * static_cast<uint32_t>(p.ldo) * ES;
  auto flush = [&](int n) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // The bounds are the buffer's: a row past M or a column past the range has an offset past its end (2^31 + less than 2^31:
    // the host has checked M + 128 rows), and is not written.
    // A branch around each store would cost a full wait at every join.
    constexpr int NST = ROWS * CPR / 64, STEP = NST < 4 ? NST : 4;  // four stores at a time: registers
    const int col = n + (lane % CPR) * (16 / ES);
    const uint32_t at = col < n_end ? (static_cast<uint32_t>(m0 + lane / CPR) * static_cast<uint32_t>(p.ldo) + col) * ES : 0x80000000u;
    const uint8_t* const src = stage + (lane / CPR) * PITCH + (lane % CPR) * 16;
#pragma unroll
    for (int t0 = 0; t0 < NST; t0 += STEP) {
      v4u v[STEP];
#pragma unroll
      for (int t = 0; t < STEP; ++t) v[t] = *reinterpret_cast<const v4u*>(src + (t0 + t) * (64 / CPR) * PITCH);
#pragma unroll
      for (int t = 0; t < STEP; ++t)
        if (nt) __builtin_amdgcn_raw_buffer_store_b128(v[t], rout, at + (t0 + t) * row_step, 0, 2);
        else __builtin_amdgcn_raw_buffer_store_b128(v[t], rout, at + (t0 + t) * row_step, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Both halves of the next step (behind the last one: of the last one again) are requested in front of the stores of this one: loads and stores share one in-order
  // counter, so a load behind them would be waited for together with the stores (90 us instead of 67 at the shape above).
  Cols c0, c1;
  int n = n_begin + wc * 64;
  load(c0, n);
  load(c1, n + 32);
  for (; n < n_end; n += CSTEP) {
    encode(c0);
    multiply(c0, 0);
    load(c0, n + CSTEP >= n_end ? n : n + CSTEP);
    encode(c1);
    multiply(c1, 1);
    load(c1, n + CSTEP >= n_end ? n : n + CSTEP + 32);
    __builtin_amdgcn_sched_barrier(0);
    flush(n);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// 32 problems of 2048 x 2048, int8 (the result alone, by a fill: 40 us), in us at K 128 / 64: tiles of 128 x 128 104 / 95;
// strips of 64 rows per workgroup 67 / 54, of 128 rows (two wavefronts below each other, b read half as often) 64.6 / 55.3,
// of 256 rows 66 / 58; strips cut into parts of 256 columns for 1024, 2048, 4096 workgroups 64.2 / 59.4, 64.6 / 55.3,
// 76.3 / 50.4.  64 problems of 500 x 1000: 128 rows 25.8, 64 rows 31.4.
template <int QT, int KS, bool BF, bool ACT = false>
int launch_strips(const StripArgs& p, int64_t batch, hipStream_t st) {
  const int rows = p.M <= 16 ? 16 : p.M <= 32 ? 32 : p.M <= 64 ? 64 : 128;
  const int strips = (p.M + rows - 1) / rows;
  const int64_t steps = (p.N + 255) / 256;
  int64_t parts = (2048 + strips * batch - 1) / (strips * batch);
  parts = parts < steps ? parts : steps;
  const int64_t per = (steps + parts - 1) / parts;
  parts = (steps + per - 1) / per;
  const dim3 grid(static_cast<unsigned>(strips * parts), static_cast<unsigned>(batch));
  const int cols = static_cast<int>(per * 256);
  // Nontemporal stores for whole 128-byte lines only: where rows start inside a line its halves come from different
  // wavefronts and have to meet in L2 (64 problems of 500 x 1000: 25.8 against 41.6 us; aligned 2048 x 2048: 84 against 65).
  const int64_t es = BF ? 2 : 4;
  const bool nt = reinterpret_cast<uintptr_t>(p.out) % 128 == 0 && p.ldo * es % 128 == 0 && p.out_stride * es % 128 == 0;
  if (rows == 16) qgemm_strips_kernel<QT, KS, 1, 1, BF, ACT><<<grid, 256, 0, st>>>(p, strips, cols, nt);
  else if (rows == 32) qgemm_strips_kernel<QT, KS, 2, 1, BF, ACT><<<grid, 256, 0, st>>>(p, strips, cols, nt);
  else if (rows == 64) qgemm_strips_kernel<QT, KS, 4, 1, BF, ACT><<<grid, 256, 0, st>>>(p, strips, cols, nt);
  else if constexpr (!ACT) qgemm_strips_kernel<QT, KS, 4, 2, BF, ACT><<<grid, 256, 0, st>>>(p, strips, cols, nt);
  return check_launch("batched qgemm (strips)");
}

}  // namespace

int qgemm_strips(int qtype, int64_t K, bool bf16, const StripArgs& p, int64_t batch, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (qtype == QWIX_INT8) {
    if (K == 64) return bf16 ? launch_strips<QWIX_INT8, 1, true>(p, batch, st) : launch_strips<QWIX_INT8, 1, false>(p, batch, st);
    return bf16 ? launch_strips<QWIX_INT8, 2, true>(p, batch, st) : launch_strips<QWIX_INT8, 2, false>(p, batch, st);
  }
  if (K == 64) return bf16 ? launch_strips<QWIX_E4M3, 1, true>(p, batch, st) : launch_strips<QWIX_E4M3, 1, false>(p, batch, st);
  return bf16 ? launch_strips<QWIX_E4M3, 2, true>(p, batch, st) : launch_strips<QWIX_E4M3, 2, false>(p, batch, st);
}

int qgemm_strips_act(int qtype, int64_t K, const StripArgs& p, int64_t batch, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (qtype == QWIX_INT8)
    return K == 64 ? launch_strips<QWIX_INT8, 1, true, true>(p, batch, st) : launch_strips<QWIX_INT8, 2, true, true>(p, batch, st);
  return K == 64 ? launch_strips<QWIX_E4M3, 1, true, true>(p, batch, st) : launch_strips<QWIX_E4M3, 2, true, true>(p, batch, st);
}

}  // namespace qwix
