// Sub-channel GEMM on tiles of 64 TM rows x 256 columns, groups of 128: int8 x int8 / int4 and e4m3 x e4m3 with one bf16 scale per
// column and group and, with OUTER, one per row and group.
//
//   out[m,n] = cast( sum_g (acc_g[m,n] * sa[m,g]) * sb[g,n] ),  acc_g = sum_{k in g} a[m,k] b[n,k]
//
// Bound by what goes on beside the MFMAs: a fold of every accumulator per group (one FMA; with OUTER convert and FMA), 192 KB of LDS
// fragment reads and 64 KB of direct-to-LDS loads per 256 x 256 x 128 slab (int4 weights: 160 and 48 KB), all issued by the same eight
// wavefronts.  Against the 128 x 256 tile of qgemm_grouped.hip (wavefronts of 128 x 32):
//   * wavefronts of 32 TM x 64: 1.5 instead of 2.5 KB of fragments per two MFMAs, half the loads per product at TM 4;
//   * a slab's fragments of a row tile are all in registers; its two column tiles' MFMAs alternate and are folded behind them, so only
//     two of the tiles' partials exist at a time and 128 sums fit a lane;
//   * one barrier per slab, in the middle: by then every wavefront has read all of the slab's b and the slab before it is done with, so
//     three stages of a and two of b hold a slab in use, one that has landed and one on its way, and the first fragments of the next
//     slab are requested under the last row tile of this one.
// Arithmetic, order and results are those of the 128 x 256 tile, bit for bit.  Measured on one card, that tile -> this one, us:
// 4096^3, one scale per row, int8 90 -> 74, e4m3 79 -> 65; scales on both sides, int8 105 -> 88, e4m3 94 -> 78; 2048 x 8192 over K
// 8192, int4 155 -> 134; 450 x 20480 over K 1536, int8 on both sides 43 -> 20 (TM 2); 1823 x 5056 over K 4096, int4 77 -> 50 (TM 3).
// Of 88 us (int8, both sides) 15 are the loads' and 19 the fold's, found by leaving them out; without both it is the 60 us that the
// plain int8 GEMM takes.  Not faster: the fold between the next tile's MFMAs, the upper and lower wavefronts half a row tile apart,
// raised priorities, loads spread one by one over the slab (all within 2 %).
#include <type_traits>

#include "common.h"
#include "qgemm_grouped.h"

namespace qwix {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ auto buffer_bytes(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

__device__ __forceinline__ float load_scale(const void* p, int dtype, int64_t i) {
  return dtype == QWIX_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]) : reinterpret_cast<const float*>(p)[i];
}

template <int BQT, int TM>
struct Wide {
  static constexpr int kBM = 64 * TM, kBN = 256, kBK = 128;
  static constexpr int kBRow = BQT == QWIX_INT4 ? 64 : 128;  // bytes of one weight row in a slab
  static constexpr int kABytes = kBM * kBK, kBBytes = kBN * kBRow;
  static constexpr int kLds = 3 * kABytes + 2 * kBBytes;
};

template <int BQT, bool OUTER, int TM, bool MAGIC>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
    qgemm_grouped_wide_kernel(GroupedArgs p) {
  using W = Wide<BQT, TM>;
  constexpr bool W4 = BQT == QWIX_INT4, F8 = BQT == QWIX_E4M3;
  constexpr int BM = W::kBM, BN = W::kBN, BK = W::kBK, B_ROWB = W::kBRow, A_BYTES = W::kABytes, B_BYTES = W::kBBytes;
  constexpr int NW = 8, WROWS = 32 * TM, B_BASE = 3 * A_BYTES;
  constexpr int A_LOADS = A_BYTES / 1024 / NW, B_LOADS = BN * B_ROWB / 1024 / NW;
  using AccV = typename std::conditional<F8, v16f, v16i>::type;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  int tile_m, tile_n;
  {  // every XCD gets a contiguous run of tiles; tiles walk down 8 tile-rows before moving along N
    const int nb = gridDim.x;
    int pid = blockIdx.x;
    if ((nb & 7) == 0) pid = (pid & 7) * (nb >> 3) + (pid >> 3);
    constexpr int GM = 8;
    const int per_group = GM * tiles_n, grp = pid / per_group, first_m = grp * GM;
    const int gsz = min(tiles_m - first_m, GM);
    tile_m = first_m + (pid % per_group) % gsz;
    tile_n = (pid % per_group) / gsz;
  }
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // ---- loader: one 32-bit offset per lane and operand, the slab as a scalar offset.  The buffers end with the last row: rows past
  // it are not read (they come as zeros, and their results are not stored).
  const uint8_t* const a_base = p.A + static_cast<int64_t>(m0) * p.lda;
  const uint8_t* const b_base = p.B + static_cast<int64_t>(n0) * p.ldb;
  const uint32_t a_bytes = static_cast<uint32_t>(min(BM, p.M - m0) - 1) * static_cast<uint32_t>(p.lda) + p.K;
  const uint32_t b_bytes = static_cast<uint32_t>(min(BN, p.N - n0) - 1) * static_cast<uint32_t>(p.ldb) + (W4 ? p.K / 2 : p.K);
  const int lrow = wave * (W4 ? 16 : 8) + (lane >> (W4 ? 2 : 3)), arow = wave * 8 + (lane >> 3);
  const uint32_t a_off = static_cast<uint32_t>(arow) * static_cast<uint32_t>(p.lda) + (((lane & 7) ^ swz128(arow)) << 4);
  const uint32_t b_off = static_cast<uint32_t>(lrow) * static_cast<uint32_t>(p.ldb) +
                         ((W4 ? ((lane & 3) ^ ((lane >> 4) & 3)) : ((lane & 7) ^ swz128(lrow))) << 4);
  const int a_step = 64 * static_cast<int>(p.lda), b_step = (W4 ? 128 : 64) * static_cast<int>(p.ldb);  // between a wavefront's pieces
  // piece j of slab kt (the rows of A first) into stage `to` of A; past the last slab the buffers are empty, and zeros are written
  const int KT = p.K / BK;
  auto issue_load = [&](int j, int kt, int to) __attribute__((always_inline)) {
    if (j < A_LOADS) {
      uint32_t ao = a_off;
      asm volatile("" : "+v"(ao));  // the pieces' offsets are added here, not kept in registers over the loop
      buffer_to_lds16(buffer_bytes(a_base, kt < KT ? a_bytes : 0), smem + to * A_BYTES + wave * 1024 + j * (NW * 1024),
                      ao + j * a_step, kt * BK);
    } else {
      const int jb = j - A_LOADS;
      uint32_t bo = b_off;
      asm volatile("" : "+v"(bo));
      buffer_to_lds16(buffer_bytes(b_base, kt < KT ? b_bytes : 0), smem + B_BASE + (kt & 1) * B_BYTES + wave * 1024 + jb * (NW * 1024),
                      bo + jb * b_step, kt * B_ROWB);
    }
  };
  constexpr int LOADS = A_LOADS + B_LOADS;

  // ---- scales: columns n0 + 64 wc + 32 j + frow; OUTER: rows m0 + WROWS wr + 32 i + frow
  const int frow = lane & 31, hx = lane >> 5;
  const auto rsb = buffer_bytes(p.sb, static_cast<uint32_t>(p.K / BK) * static_cast<uint32_t>(p.N) * 2);
  const auto rsa = buffer_bytes(p.sa, OUTER ? static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.ga) * 2 : 0);
  const uint32_t sb_off = static_cast<uint32_t>(n0 + wc * 64 + frow) * 2, sb_last = static_cast<uint32_t>(p.N - 1) * 2;
  const uint32_t sa_off = static_cast<uint32_t>(m0 + wr * WROWS + frow) * static_cast<uint32_t>(p.ga) * 2;
  struct Scales {
    unsigned b[2];
    unsigned a[OUTER ? TM : 1];
  };
  auto load_scales = [&](Scales& s, int g) __attribute__((always_inline)) {
    uint32_t bo = sb_off;
    asm volatile("" : "+v"(bo));
#pragma unroll
    for (int j = 0; j < 2; ++j) s.b[j] = __builtin_amdgcn_raw_buffer_load_b16(rsb, min(bo + j * 64, sb_last), g * p.N * 2, 0);
    if constexpr (OUTER) {
      uint32_t so = sa_off;
      asm volatile("" : "+v"(so));
#pragma unroll
      for (int i = 0; i < TM; ++i) s.a[i] = __builtin_amdgcn_raw_buffer_load_b16(rsa, so + static_cast<uint32_t>(i * 64) * static_cast<uint32_t>(p.ga), g * 2, 0);
    }
  };
  // ---- fragments: 16-byte chunk c of a row stands at chunk position c ^ key, so the addresses of a lane's chunks differ from the
  // first one's by an exclusive or (rows are whole multiples of the chunks it touches)
  const uint32_t a_lane = (wr * WROWS + frow) * BK + (((W4 ? 2 * hx : hx) ^ swz128(frow)) << 4);
  const uint32_t b_lane = B_BASE + (wc * 64 + frow) * B_ROWB + ((hx ^ (W4 ? ((frow >> 2) & 3) : swz128(frow))) << 4);

  float accf[TM][2][16];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) accf[i][j][r] = 0.f;
  constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23
  v16i magic;
  if constexpr (MAGIC) {
#pragma unroll
    for (int r = 0; r < 16; ++r) magic[r] = 0x4B400000;
    asm volatile("" : "+v"(magic));
  }
  float corr[2] = {0.f, 0.f};

  Scales raw_s;
  unsigned cur_b, cur_a[OUTER ? (TM + 1) / 2 : 1];  // two to a register
  auto take_scales = [&]() __attribute__((always_inline)) {
    cur_b = raw_s.b[0] | raw_s.b[1] << 16;
    if constexpr (OUTER) {
#pragma unroll
      for (int i = 0; i < TM; i += 2) cur_a[i / 2] = i + 1 < TM ? raw_s.a[i] | raw_s.a[i + 1 < TM ? i + 1 : i] << 16 : raw_s.a[i];
    }
  };
  v4i fa[4], fbr[2][W4 ? 2 : 4], fb[2][4];
  v8i fa8[2], fb8[2][2];  // e4m3: two 16-byte pieces of consecutive k-steps make one operand
  auto at = [&](uint32_t where) __attribute__((always_inline)) { return *reinterpret_cast<const v4i*>(smem + where); };
  auto joined = [&](const v4i& lo, const v4i& hi) __attribute__((always_inline)) {
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  // a quarter (k-step q; e4m3: half q / 2, with q odd) of a row tile's fragment, of both column tiles' fragments
  auto read_a = [&](uint32_t base, int q) __attribute__((always_inline)) {
    if constexpr (F8) {
      if (q % 2) fa8[q / 2] = joined(at(base ^ (q / 2 * 64)), at(base ^ (q / 2 * 64 + 32)));
    } else {
      fa[q] = at(base ^ (W4 ? (q >> 1) * 64 + (q & 1) * 16 : q * 32));
    }
  };
  auto read_b = [&](uint32_t base, int q) __attribute__((always_inline)) {
    if constexpr (F8) {
      if (q % 2) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          fb8[j][q / 2] = joined(at((base + j * 32 * B_ROWB) ^ (q / 2 * 64)), at((base + j * 32 * B_ROWB) ^ (q / 2 * 64 + 32)));
      }
    } else if constexpr (W4) {
      fbr[q % 2][q / 2] = at((base + (q % 2) * 32 * B_ROWB) ^ (q / 2 * 32));
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) fbr[j][q] = at((base + j * 32 * B_ROWB) ^ (q * 32));
    }
  };
  auto a_base_of = [&](int stage, int i) __attribute__((always_inline)) {
    uint32_t base = a_lane;
    asm volatile("" : "+v"(base));
    return base + stage * A_BYTES + i * 32 * BK;
  };
  auto b_base_of = [&](int stage) __attribute__((always_inline)) {
    uint32_t base = b_lane;
    asm volatile("" : "+v"(base));
    return base + stage * B_BYTES;
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- prologue: slab 0 has landed, slab 1 is on its way, the first fragments of slab 0 are requested
  load_scales(raw_s, 0);
#pragma unroll
  for (int j = 0; j < LOADS; ++j) issue_load(j, 0, 0);
  barrier();
  take_scales();
#pragma unroll
  for (int j = 0; j < LOADS; ++j) issue_load(j, 1, 1);
  {
    const uint32_t ab = a_base_of(0, 0), bb = b_base_of(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      read_a(ab, q);
      read_b(bb, q);
    }
  }
  int as = 0;  // stage of A that holds the current slab
#pragma clang loop unroll(disable)
  for (int kt = 0; kt < KT; ++kt) {
    const bool recentre = (kt & 3) == 3 || kt == KT - 1;
    const int as1 = as == 2 ? 0 : as + 1, as2 = as == 0 ? 2 : as - 1;  // of the next slab, of the one after it
    auto widen = [&](int j, int ks) __attribute__((always_inline)) {
      if constexpr (W4) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const unsigned w = static_cast<unsigned>(fbr[j][ks >> 1][2 * (ks & 1) + h]);
          const unsigned ev = (w << 4) & 0xF0F0F0F0u, od = w & 0xF0F0F0F0u;  // nibbles 0,2,4,6 and 1,3,5,7, x 16
          fb[j][ks][2 * h] = static_cast<int>(__builtin_amdgcn_perm(od, ev, 0x05010400));
          fb[j][ks][2 * h + 1] = static_cast<int>(__builtin_amdgcn_perm(od, ev, 0x07030602));
        }
      }
    };
    float sbg[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) sbg[j] = __uint_as_float(j == 0 ? cur_b << 16 : cur_b & 0xFFFF0000u) * (W4 ? 0.0625f : 1.0f);
    if constexpr (!F8 && !OUTER) {
#pragma unroll
      for (int j = 0; j < 2; ++j) corr[j] = __builtin_fmaf(kMagic, sbg[j], corr[j]);
    }
    AccV acc[2];
    v16f prod;
    auto outer = [&](int i, int j) __attribute__((always_inline)) {
      if constexpr (OUTER) {
        const unsigned keep = hx == 0 ? 0xFFFFu : 0u;  // k 0 sits in the lower half of the lanes
        const qwix_v2i va = {static_cast<int>((i % 2 ? cur_a[i / 2] >> 16 : cur_a[i / 2]) & keep), 0},
                       vb = {static_cast<int>((j ? cur_b >> 16 : cur_b) & keep), 0};
        const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        prod = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(v4s, va), __builtin_bit_cast(v4s, vb), zero, 0, 0, 0);
      }
    };
    // the slab's MFMAs of one row tile, the two column tiles in turn (one that waits for the sums of the one before it takes twice as long)
    auto multiply = [&](int i) __attribute__((always_inline)) {
      if constexpr (F8) {
        const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa8[kp], fb8[j][kp], kp == 0 ? zero : acc[j], 0, 0, 0, 0, 0, 0);
          }
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if (i == 0) widen(j, ks);
            const v4i& b = W4 ? fb[j][ks] : fbr[j][ks];
            if constexpr (MAGIC) {
              acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[ks], b, ks == 0 ? magic : acc[j], 0, 0, 0);
            } else {
              const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
              acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[ks], b, ks == 0 ? zero : acc[j], 0, 0, 0);
            }
          }
        }
      }
    };
    auto fold = [&](int i, int j) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float& s = accf[i][j][r];
        if constexpr (OUTER && F8) s = __builtin_fmaf(acc[j][r], prod[r], s);
        else if constexpr (OUTER && MAGIC) s = __builtin_fmaf(__int_as_float(acc[j][r]) - kMagic, prod[r], s);
        else if constexpr (OUTER) s = __builtin_fmaf(static_cast<float>(acc[j][r]), prod[r], s);
        else if constexpr (F8) s = __builtin_fmaf(acc[j][r], sbg[j], s);
        else s = __builtin_fmaf(__int_as_float(acc[j][r]), sbg[j], s);
      }
      if constexpr (!F8 && !OUTER) {
        if (recentre) {
#pragma unroll
          for (int r = 0; r < 16; ++r) accf[i][j][r] -= corr[j];
        }
      } else {
        // a use right behind the fold: without one the compiler moves it to where the sums are next read, and keeps the partials
        float* s = accf[i][j];
        asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]), "+v"(s[6]), "+v"(s[7]), "+v"(s[8]),
                     "+v"(s[9]), "+v"(s[10]), "+v"(s[11]), "+v"(s[12]), "+v"(s[13]), "+v"(s[14]), "+v"(s[15]));
      }
    };
    // every wavefront has read its fragments of this slab's b and all of the last slab's a; the next slab has landed
    auto slab_barrier = [&]() __attribute__((always_inline)) {
      barrier();
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i == 1) {
        slab_barrier();
        load_scales(raw_s, min(kt + 1, KT - 1));
      }
      outer(i, 0);
      // behind a k-step's MFMAs: its fragments of the next row tile (of the next slab's first one, and of its columns), and
      // the slab after next into the stages that the barrier has freed
      const uint32_t ab = a_base_of(i + 1 < TM ? as : as1, i + 1 < TM ? i + 1 : 0);
      const uint32_t bb = b_base_of((kt + 1) & 1);
      multiply(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) read_a(ab, q);
      if (i == TM - 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) read_b(bb, q);
      }
      __builtin_amdgcn_sched_barrier(0);
      fold(i, 0);
      if (i >= 1) {
        constexpr int PER = (LOADS + TM - 2) / (TM - 1);
#pragma unroll
        for (int l = (i - 1) * PER; l < i * PER && l < LOADS; ++l) issue_load(l, kt + 2, as2);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_sched_barrier(0);
      outer(i, 1);
      __builtin_amdgcn_sched_barrier(0);
      fold(i, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!F8 && !OUTER) {
      if (recentre) corr[0] = corr[1] = 0.f;
    }
    take_scales();
    as = as1;
  }
  barrier();  // LDS turns into staging space for the output

  // ---- epilogue: 32 rows x 64 columns of f32 per wavefront and pass through LDS
  constexpr int ROW_F = 68;
  float* stg = reinterpret_cast<float*>(smem) + wave * (32 * ROW_F);
  static_assert(NW * 32 * ROW_F * 4 <= W::kLds, "epilogue staging must fit");
  const bool t_bf16 = p.t_dtype == QWIX_BF16;
  const bool vec_ok = p.ldo % 8 == 0 && p.N % 8 == 0;
  const int n = n0 + wc * 64 + (lane & 7) * 8;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    float sav[4] = {1.f, 1.f, 1.f, 1.f};
    if (!OUTER && p.sa != nullptr) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = min(m0 + wr * WROWS + i * 32 + (lane >> 3) + 8 * q, p.M - 1);
        sav[q] = load_scale(p.sa, p.sa_dtype, m);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) stg[(8 * (r >> 2) + 4 * hx + (r & 3)) * ROW_F + j * 32 + frow] = accf[i][j][r];
    if (vec_ok) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = (lane >> 3) + 8 * q, m = m0 + wr * WROWS + i * 32 + row;
        const v4f lo = *reinterpret_cast<const v4f*>(stg + row * ROW_F + (lane & 7) * 8);
        const v4f hi = *reinterpret_cast<const v4f*>(stg + row * ROW_F + (lane & 7) * 8 + 4);
        float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] *= sav[q];
          if (t_bf16) v[e] = round_bf16(v[e]);
        }
        if (m >= p.M || n >= p.N) continue;
        if (p.out_dtype == QWIX_BF16) {
          uint32_t u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
          nt_store16(reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.out) + static_cast<int64_t>(m) * p.ldo + n),
                     make_uint4(u[0], u[1], u[2], u[3]));
        } else {
          uint4* o = reinterpret_cast<uint4*>(reinterpret_cast<float*>(p.out) + static_cast<int64_t>(m) * p.ldo + n);
          nt_store16(o, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
          nt_store16(o + 1, make_uint4(__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])));
        }
      }
    } else {
      // rows that do not start on 16 bytes: one column per lane, row by row
      const int nl = n0 + wc * 64 + lane;
#pragma clang loop unroll(disable)
      for (int row = 0; row < 32; ++row) {
        const int m = m0 + wr * WROWS + i * 32 + row;
        float v = stg[row * ROW_F + lane];
        if (!OUTER && p.sa != nullptr) v *= load_scale(p.sa, p.sa_dtype, min(m, p.M - 1));
        if (t_bf16) v = round_bf16(v);
        if (m >= p.M || nl >= p.N) continue;
        if (p.out_dtype == QWIX_BF16) reinterpret_cast<uint16_t*>(p.out)[static_cast<int64_t>(m) * p.ldo + nl] = f32_to_bf16_bits(v);
        else reinterpret_cast<float*>(p.out)[static_cast<int64_t>(m) * p.ldo + nl] = v;
      }
    }
  }
}

template <int BQT, bool OUTER, int TM, bool MAGIC>
int launch_wide(const GroupedArgs& p, hipStream_t st) {
  using W = Wide<BQT, TM>;
  constexpr size_t smem = W::kLds;
  auto kern = qgemm_grouped_wide_kernel<BQT, OUTER, TM, MAGIC>;
  static LdsGrant granted;
  if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted)) return e_;
  const int64_t tiles = static_cast<int64_t>((p.M + W::kBM - 1) / W::kBM) * ((p.N + W::kBN - 1) / W::kBN);
  kern<<<dim3(static_cast<unsigned>(tiles)), 512, smem, st>>>(p);
  return check_launch("qgemm_grouped (wide)");
}

template <int BQT, bool OUTER>
int launch_rows(int tm, const GroupedArgs& p, hipStream_t st) {
  constexpr bool kInt = BQT != QWIX_E4M3;
  // (128 rows per wavefront, scales on both sides: no registers for the sixteen constants)
  if (tm == 4) return launch_wide<BQT, OUTER, 4, kInt && !OUTER>(p, st);
  if (tm == 3) return launch_wide<BQT, OUTER, 3, kInt>(p, st);
  return launch_wide<BQT, OUTER, 2, kInt>(p, st);
}

}  // namespace

int qgemm_grouped_wide(const GroupedArgs& p, int b_qtype, bool outer, int tm, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (b_qtype == QWIX_INT4) return launch_rows<QWIX_INT4, false>(tm, p, st);
  if (b_qtype == QWIX_INT8) return outer ? launch_rows<QWIX_INT8, true>(tm, p, st) : launch_rows<QWIX_INT8, false>(tm, p, st);
  return outer ? launch_rows<QWIX_E4M3, true>(tm, p, st) : launch_rows<QWIX_E4M3, false>(tm, p, st);
}

}  // namespace qwix
