// Weight-only GEMM beyond the decode batch: bf16 activations x int4 / int8 / e4m3 weights dequantized inside the workgroup.
#include <algorithm>

#include "common.h"
#include "qgemm_tiles.h"

namespace qwix {
namespace {

// ------------------------------------------------------------------------------------------------
// bf16 activations x int4 weights with K-group scales, beyond the decode batch (prefill): the weights are dequantized
// inside the workgroup instead of in a pass of their own.  A 256 x 128 tile on 8 wavefronts (64 x 64 each),
// v_mfma_f32_32x32x16_bf16, K in slabs of 64 elements (128 bytes of a row of activations), 160 KB of LDS.
//   The packed weights come in whole 128-byte lines: one direct-to-LDS load per 8 rows fetches 256 elements of
// K per row, four slabs' worth (a superslab), into one of two raw buffers; the next superslab and its four scales
// (untracked loads) are requested in the first slab of this one.  While slab kt is multiplied, slab kt + 1 of the
// weight tile is converted: every thread takes 16 nibbles of one row out of the raw buffer, turns them into
// bf16(q * scale) -- the value the reference's dequantize gives (qarray.py:692-708, computed in f32 and rounded to
// bf16: exact for bf16 scales, one more rounding for f32 scales, as qwix_hip_dequantize_rm does) -- and writes them
// where the dense bf16 kernel expects the weight slab (same XOR swizzle), a quarter of the work in front of each of
// the slab's four k-steps.  The activations go through three LDS stages by direct-to-LDS loads requested two slabs
// ahead (four stages, three slabs in the 128-row tile).  One barrier per slab; the wait in front of it is counted
// (vmcnt), so that the requests of the slab that ends (in the 128-row tile: and of the one before) stay in flight: a
// full wait there costs a memory round trip per slab (87 us instead of 65 at 512 x 14336 x 4096).
//   LDS is read and written through ext_vector types only (v4i, qwix_v2i).  Through HIP's struct vectors (uint2,
// uint4) the compiler cannot tell the access from the destinations of the direct-to-LDS loads in flight and puts
// an s_waitcnt vmcnt(0) in front of it, which turns every counted wait into a full one.
// Results are bit-identical to qwix_hip_dequantize_rm + qwix_hip_gemm_bf16: the same bf16 weights, the same MFMA,
// K walked in the same order.
// BN = 64 (tiles of 256 x 64, wavefronts of 64 x 32, 128 KB of LDS) is for calls whose 128-column tiles would leave
// more than half of the CUs without a workgroup: a workgroup's time is mostly its MFMAs and the conversion, which
// both halve, while its activation traffic stays.
// BITS = 8: int8 weights.  A row's 128-byte line would hold only two slabs, too few to request a buffer ahead, so
// they come as 64-byte pieces, one slab per request (16 rows per load instruction), into a ring of four buffers:
// slab kt + 3 is requested in slab kt, behind the activations of slab kt + 2 (128-row tile: kt + 4 behind kt + 3, into
// the buffer that was read in slab kt - 1).  With 64-column tiles on eight requesting wavefronts the upper half of
// a load instruction's lanes repeats the lower half's rows (every wavefront issues one load per slab, so that all
// count their requests alike); the repeated rows land in padding.  A byte b holds q = (b ^ 0x80) - 128 and
// q * scale = fma(b ^ 0x80, scale, -128 scale), exact as for the nibbles.  BITS = 9 stands for e4m3 weights: the same
// bytes, converted by v_cvt_pk_f32_fp8 (two per instruction) and multiplied by the scale.
// ZP: asymmetric weights, (q - zero_point) * scale with one int8 zero point per scale.  It is requested with the scale
// and joins the offset of the storage format: bf16 scales fma(u, scale, -(offset + zp) scale), every term still exact
// in f32 (nine bits times eight); f32 scales float(u - offset - zp) * scale, the integer difference first, because
// (offset + zp) * scale would no longer be exact.
// BM = 128 (tiles of 128 x 64) is for calls of at most 128 rows: half the MFMAs and half the activation loads per
// workgroup of the 256-row tile, whose upper half would multiply padding.  Its eight wavefronts split the work: four
// multiply (64 x 32 each) and load nothing, four only request the operands, three slabs ahead, and wait for them; a
// wavefront issues in order, so one that requests and multiplies stands at a load instruction while the memory
// pipeline is full and its SIMD's matrix core idles (requests, conversion and MFMAs added up to the run time: 10 +
// 4 + 7 us on top of 9.4 us of skeleton at 128 x 4096 x 4096, int8; 34 -> 29 us at 128 x 14336 x 4096).  The
// requesting wavefronts also dequantize int4 weights (35.6 -> 29.3 us against 32.6 with the conversion between the
// MFMAs); bytes convert faster between the MFMAs (28.5 against 32.8 us).  The requesting wavefronts end after the last
// slab: a wavefront that has ended no longer counts at the workgroup's barriers.
//   In the 256-row tiles every wavefront requests and multiplies; there the four activation loads of a slab are issued
// one per k-step instead of together (512 x 4096 x 4096: int4 47 -> 42 us, int8 50 -> 45 us).
// BM = 192 (192 x 128, wavefronts of 96 x 32) is for rows that would leave a 256-row tile's end as padding: a quarter of
// the MFMAs and of the activation loads less per workgroup, the same fragment reads and conversion, 0.88 of its time.  256 / 192 rows
// per tile: int4 333 x 14336 over K 4096 64.9 -> 56.2 us, 181 x 28288 over K 1792 29.0 -> 26.7, 160 x 28672 over K 8192 122 -> 109,
// 700 x 14336 over K 4096 118 -> 107; int8 333 x 14336 62.3 -> 54.5; e4m3 380 x 10240 over K 2048 31.0 -> 27.3; where it takes
// another round, 512 x 14336 over K 4096, 61 against 104.
//   With int4 weights it splits the work as the 128-row tile does: four wavefronts of 96 x 64 multiply (80 KB of fragment reads per
// slab instead of 128), four request and dequantize, and the LDS (160 KB) holds a fourth stage of activations.  333 x 14336 over K 4096
// 59.5 -> 56.5 us, 700 x 14336 over K 4096 105 -> 101, 160 x 28672 over K 8192 102 -> 95.5, 181 x 28288 over K 1792 27.5 -> 27.3; no part
// of a slab bounds it alone (without MFMAs 43, without activation loads 46, without conversion 52).  A 256-row tile has no room for that
// stage and loses (512 x 14336 over K 4096 63.7 -> 66.9); a HALF one spills.
// RAGGED: rows in groups (mixture of experts), found on the device as in the ragged GEMM: the tile's rows end with its
// group, and weights and scales are the group's.
// HALF: K may be 128 mod 256, the last superslab half of one: another tail behind a branch, clamped loads of the last line of
// int4 weights and of its scales.  A template parameter because the branch costs registers that all K would pay for (bf16
// result, 128 x 64 int4 / int8, 256 x 128 int4: 124 / 151 / 248 per lane with it, 86 / 111 / 173 without).
// Whether a tile's wavefronts split the work (see above), and its stages of activations.
constexpr bool wq_spec(int bm, int bn, int bits, bool half) { return bm == 128 || (bits == 4 && bm == 192 && !half); }
constexpr int wq_stages(int bm, int bn, int bits, bool half) { return wq_spec(bm, bn, bits, half) ? 4 : 3; }
struct NoGroups {};  // (unused arguments would move the ones behind them into another line of the argument block)
template <int OUT, bool SBF, int BM, int BN, int BITS, bool ZP, bool HALF, bool RAGGED = false>
__global__ void __launch_bounds__(512)
    wgemm_wq_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ Q, int64_t ldq,
                    const void* __restrict__ S, const int8_t* __restrict__ Z, int M, int N, int K, int group,
                    uint8_t* __restrict__ out, int64_t ldo, int ksplit,
                    typename std::conditional<RAGGED, Ragged, NoGroups>::type rg) {
  static_assert((BM == 256 && (BN == 128 || BN == 64)) || (BM == 192 && BN == 128) || (BM == 128 && BN == 64),
                "tiles of 256 x 128, 192 x 128, 256 x 64, 128 x 64");
  if (ksplit > 0) {
    // K split over blockIdx.y: this workgroup contracts elements [y ksplit, (y + 1) ksplit), or what is left of them --
    // ksplit a multiple of 256, and a multiple or a divisor of the group, so that a range starts a group or lies inside
    // one; a last range is a multiple of 128 from 256 on -- and writes its tile
    // of the y-th M x N partial (the host passes OUT = f32 and ldo = N); every operand pointer moves to the range's
    // first element (the scales': to the group that holds it).
    const int k0 = static_cast<int>(blockIdx.y) * ksplit;
    A += static_cast<int64_t>(k0) * 2;
    Q += (BITS >= 8) ? k0 : k0 / 2;
    S = static_cast<const char*>(S) + static_cast<int64_t>(k0 / group) * N * (SBF ? 2 : 4);
    if constexpr (ZP) Z += static_cast<int64_t>(k0 / group) * N;
    out += static_cast<int64_t>(blockIdx.y) * M * N * 4;
    K = min(ksplit, K - k0);
  }
  // SPEC: as many wavefronts again that only request the operands (rows and weight rows of wavefront wave - NWAVES)
  constexpr bool SPEC = wq_spec(BM, BN, BITS, HALF);
  constexpr int NWAVES = SPEC ? 4 : 8, NTHREADS = NWAVES * 64, NA = BM / 8 / NWAVES;  // NA: activation loads per wavefront and slab
  constexpr int WGN = BM == 192 && !SPEC ? 4 : 2, WN = BN / WGN, WM = BM / (NWAVES / WGN), TM = WM / 32, TN = WN / 32;
  constexpr int BK = 128, NK = 4;  // bytes of an activation row per slab (64 elements); k-steps of 16 elements
  static_assert(BITS == 4 || BITS == 8 || BITS == 9, "int4, int8 or (9) e4m3 weights");
  constexpr bool W8 = BITS >= 8;   // one byte per weight
  constexpr bool F8 = BITS == 9;   // e4m3: the byte converts to f32 directly; no offset, no zero point
  static_assert(!(F8 && ZP), "float weights have no zero point");
  // raw weights: int4 two buffers of a superslab (BN x 128 bytes), int8 four of a slab (1 KB per wavefront)
  constexpr int A_STAGE = BM * BK, C_STAGE = BN * BK, R_STAGE = W8 ? NWAVES * 1024 : BN * 128;
  // slabs between the request of activations and their use; where the LDS holds it one more
  constexpr int AST = wq_stages(BM, BN, BITS, HALF), AL = AST - 1;
  static_assert(AL == 2 || AL == 3, "the last four slabs are the only special ones");
  constexpr int C_BASE = AST * A_STAGE, R_BASE = C_BASE + 2 * C_STAGE, LDS_BYTES = R_BASE + (W8 ? 4 : 2) * R_STAGE;  // <= 160 KB
  constexpr int RPW = BN / NWAVES;  // weight rows per wavefront: 16, 8 or 32
  constexpr int NQ = W8 ? 1 : RPW / 8;  // direct-to-LDS loads of weights per wavefront and request
  constexpr int TPR = NTHREADS / BN;    // converter threads per weight row: 4, 8 or 2
  constexpr int NPT = 64 / TPR;     // elements per thread and slab: 16, 8 or 32
  constexpr int NCQ = NPT / 4;      // conversion steps of four elements: 4, 2 or 8
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const bool loader = SPEC && wave >= NWAVES;
  // who dequantizes: the requesting wavefronts for int4 (measured 32.6 -> 30.2 us at 128 x 14336 x 4096), the multiplying
  // ones for bytes (30.4 against 32.8 us)
  constexpr bool LC = SPEC && !W8;
  const int ldw = SPEC ? (wave & (NWAVES - 1)) : wave;
  int m0, n0;
  if constexpr (RAGGED) {
    int g, m_lim;
    const int kind = ragged_tile<BM, BN>(rg, M, N, &g, &m0, &m_lim, &n0);
    if (kind == 0) return;
    if (kind == 2) {
      using OutT = typename std::conditional<OUT == QWIX_BF16, uint16_t, uint32_t>::type;
      zero_tile<BM, BN, OutT>(out, ldo, m0, m_lim, n0, N, 512);
      return;
    }
    M = m_lim;
    Q += g * rg.b_group_stride;
    S = static_cast<const char*>(S) + g * rg.sb_group_stride * (SBF ? 2 : 4);
  } else {
    int tile_m, tile_n;
    tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, &tile_m, &tile_n);
    m0 = tile_m * BM;
    n0 = tile_n * BN;
  }

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // ---- loaders: 8 rows x 128 bytes per instruction; the global 16-byte chunk that lands at position lane & 7
  const int lr = lane >> 3;
  uint32_t goffa[NA], goffq[NQ], back[HALF ? NQ : 1];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int row = (ldw * NA + j) * 8 + lr;
    goffa[j] = static_cast<uint32_t>(min(m0 + row, M - 1)) * static_cast<uint32_t>(lda) + (((lane & 7) ^ swz8(row)) << 4);
  }
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    if constexpr (W8) {  // 16 rows x 64 bytes per instruction (64-column tiles: 8 rows, twice)
      const int row = ldw * RPW + ((lane >> 2) & (RPW - 1));
      goffq[j] = static_cast<uint32_t>(min(n0 + row, N - 1)) * static_cast<uint32_t>(ldq) + ((lane & 3) << 4);
    } else {
      const int row = ldw * RPW + j * 8 + lr;
      const uint32_t chunk = (lane & 7) ^ swz8(row);
      goffq[j] = static_cast<uint32_t>(min(n0 + row, N - 1)) * static_cast<uint32_t>(ldq) + (chunk << 4);
      if constexpr (HALF) back[j] = chunk >= 4 ? 64 : 0;
    }
  }
  auto issue_a = [&](int kt, int stage) __attribute__((always_inline)) {  // NA loads
    const uint8_t* gk = A + kt * BK;
    uint8_t* dst = smem + stage * A_STAGE + ldw * NA * 1024;
#pragma unroll
    for (int j = 0; j < NA; ++j) QWIX_GLDS16(gk + goffa[j], dst + j * 1024);
  };
  auto issue_raw = [&](int ss) __attribute__((always_inline)) {  // int4: superslab ss (elements 256 ss ..), NQ loads; int8: slab ss, one load
    if constexpr (W8) {
      QWIX_GLDS16(Q + ss * 64 + goffq[0], smem + R_BASE + (ss & 3) * R_STAGE + ldw * 1024);
    } else {
      const uint8_t* gq = Q + ss * 128;
      uint8_t* dst = smem + R_BASE + (ss & 1) * R_STAGE + ldw * RPW * 128;
      // the last 128 elements of a K that is no multiple of 256: the line's upper half repeats the lower one
      const uint32_t half = HALF && ss * 256 + 256 > K ? ~0u : 0u;
#pragma unroll
      for (int j = 0; j < NQ; ++j) QWIX_GLDS16(gq + (goffq[j] - (HALF ? back[HALF ? j : 0] & half : 0)), dst + j * 1024);
    }
  };

  // ---- converter: thread -> (weight row, NPT of the slab's 64 elements)
  const int ctid = tid & (NTHREADS - 1);
  const int crow = ctid / TPR, cpart = ctid % TPR;
  const char* const sptr = static_cast<const char*>(S) + static_cast<int64_t>(min(n0 + crow, N - 1)) * (SBF ? 2 : 4);
  const int64_t s_group_pitch = static_cast<int64_t>(N) * (SBF ? 2 : 4);
  // The scales of four slabs are requested at once, a superslab ahead, by untracked loads (valid once a later
  // end-of-slab wait has covered them); the pointer walks the groups slab by slab.
  const int slabs_per_group = group >> 6;
  const char* sc_ptr = sptr;
  const int8_t* zp_ptr = ZP ? Z + min(n0 + crow, N - 1) : nullptr;
  int sc_left = slabs_per_group, sc_groups = K / group;  // (HALF: the two slabs past K read the last group's)
  auto request_scales = [&](uint32_t (&dst)[4], int (&dstz)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (SBF)
        asm volatile("global_load_ushort %0, %1, off" : "=&v"(dst[j]) : "v"(sc_ptr) : "memory");
      else
        asm volatile("global_load_dword %0, %1, off" : "=&v"(dst[j]) : "v"(sc_ptr) : "memory");
      if constexpr (ZP) asm volatile("global_load_sbyte %0, %1, off" : "=&v"(dstz[j]) : "v"(zp_ptr) : "memory");
      if (--sc_left == 0) {
        sc_left = slabs_per_group;
        if (!HALF || --sc_groups > 0) {
          sc_ptr += s_group_pitch;
          if constexpr (ZP) zp_ptr += N;
        }
      }
    }
  };
  auto pin_scales = [&](uint32_t (&v)[4], int (&vz)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      asm volatile("" : "+v"(v[j]));
      if constexpr (ZP) asm volatile("" : "+v"(vz[j]));
    }
  };
  constexpr int kSL = ZP ? 8 : 4;  // loads of one request_scales
  constexpr int NRAW = NPT * (W8 ? 8 : 4) / 32;  // dwords of raw weights per thread and slab
  int craw[NRAW];
  uint32_t cout[NPT / 2];
  auto convert_read = [&](int kt) __attribute__((always_inline)) {
    const uint8_t* src;
    if constexpr (W8) {  // the row's 64 bytes of this slab, NPT of them
      src = smem + R_BASE + (kt & 3) * R_STAGE + (crow / RPW) * 1024 + (crow % RPW) * 64 + cpart * NPT;
    } else {  // NPT / 2 bytes of the row's line: 32 bytes per slab, in two 16-byte chunks
      const int byte = cpart * (NPT / 2);  // of the slab's 32
      const int chunk = ((kt & 3) * 2 + (byte >> 4)) ^ swz8(crow);
      src = smem + R_BASE + ((kt >> 2) & 1) * R_STAGE + crow * 128 + (chunk << 4) + (byte & 15);
    }
    if constexpr (NRAW == 4) {
      const v4i v = *reinterpret_cast<const v4i*>(src);
#pragma unroll
      for (int e = 0; e < 4; ++e) craw[e] = v[e];
    } else if constexpr (NRAW == 2) {
      const qwix_v2i v = *reinterpret_cast<const qwix_v2i*>(src);
      craw[0] = v[0];
      craw[1] = v[1];
    } else {
      craw[0] = *reinterpret_cast<const int*>(src);
    }
  };
  // A nibble n holds q = (n ^ 8) - 8.  With the 8 folded into the multiply-add, q * scale = fma(n ^ 8, scale, -8 scale): every
  // term is exact in f32 (four bits times the eight of a bf16 scale), so the product is the one of float(q) * scale, and a
  // byte of the masked word converts in one instruction.
  auto convert_quarter = [&](int q4, float sc, int zp) __attribute__((always_inline)) {  // elements 4 q4 .. 4 q4 + 3 of this thread's NPT
    if (q4 >= NCQ) return;
    const int off = (W8 ? 128 : 8) + (ZP ? zp : 0);          // what the stored byte / nibble carries too much
    const float moff = -static_cast<float>(off) * sc;        // exact (see above)
    auto value = [&](uint32_t u) -> float {
      if constexpr (ZP && !SBF) return static_cast<float>(static_cast<int>(u) - off) * sc;
      return __builtin_fmaf(static_cast<float>(u), sc, moff);
    };
    float f0, f1, f2, f3;
    if constexpr (F8) {
      // two bytes per instruction: v_cvt_pk_f32_fp8 issues in 8 counter ticks, v_cvt_f32_fp8 in 12.5 for one byte
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(craw[q4], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(craw[q4], true);
      f0 = lo[0] * sc;
      f1 = lo[1] * sc;
      f2 = hi[0] * sc;
      f3 = hi[1] * sc;
    } else if constexpr (W8) {
      const uint32_t u = static_cast<uint32_t>(craw[q4]) ^ 0x80808080u;
      f0 = value(u & 0xFFu);
      f1 = value((u >> 8) & 0xFFu);
      f2 = value((u >> 16) & 0xFFu);
      f3 = value(u >> 24);
    } else {
      const uint32_t w = static_cast<uint32_t>(craw[q4 >> 1]) ^ 0x88888888u;
      uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
      // opaque to the optimizer: it would fold the masks into one bit-field extract per nibble in front of the byte
      // conversion (v_bfe_u32 + v_cvt_f32_ubyte0) instead of converting the masked words' bytes in place
      asm("" : "+v"(even));
      asm("" : "+v"(odd));
      const int b0 = (q4 & 1) * 16;
      f0 = value((even >> b0) & 0xFFu);
      f1 = value((odd >> b0) & 0xFFu);
      f2 = value((even >> (b0 + 8)) & 0xFFu);
      f3 = value((odd >> (b0 + 8)) & 0xFFu);
    }
    cout[2 * q4] = pack_bf16x2(f0, f1);
    cout[2 * q4 + 1] = pack_bf16x2(f2, f3);
  };
  auto convert_write = [&](int kt) __attribute__((always_inline)) {  // NPT bf16 values: one or two 16-byte chunks of the row's slab
    uint8_t* row = smem + C_BASE + (kt & 1) * C_STAGE + crow * 128;
#pragma unroll
    for (int c = 0; c < NPT / 8; ++c)
      *reinterpret_cast<v4i*>(row + (((cpart * (NPT / 8) + c) ^ swz8(crow)) << 4)) =
          v4i{(int)cout[4 * c], (int)cout[4 * c + 1], (int)cout[4 * c + 2], (int)cout[4 * c + 3]};
  };
  auto scale_value = [&](uint32_t bits) { return __uint_as_float(SBF ? bits << 16 : bits); };

  // ---- fragments
  const int a_row = (wm * WM + (lane & 31)) * BK;
  const int b_row = C_BASE + (wn * WN + (lane & 31)) * BK;
  const int hx = lane >> 5, x7 = swz8(lane & 31);
  v4i fa[2][TM], fb[2][TN];
  auto read_frags = [&](int sta, int stc, int ks, int buf) __attribute__((always_inline)) {
    const int off = ((ks * 2 + hx) ^ x7) << 4;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[buf][i] = *reinterpret_cast<const v4i*>(smem + sta * A_STAGE + a_row + i * 32 * BK + off);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[buf][j] = *reinterpret_cast<const v4i*>(smem + stc * C_STAGE + b_row + j * 32 * BK + off);
  };
  auto mfma_step = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb[buf][j]),
                                                            __builtin_bit_cast(bf16x8, fa[buf][i]), acc[i][j], 0, 0, 0);
  };
  // End of a slab: this wavefront's LDS writes are done and its loads have landed, except the NEWEST `newest` of
  // them (vmcnt counts in issue order): the requests of the slab that ends are for two slabs ahead and stay in
  // flight across the barrier.  Then everybody's.
  auto end_of_slab = [&](auto newest) {
    constexpr int n = decltype(newest)::value;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14));  // vmcnt(n), lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  using std::integral_constant;

  const int KT = K / 64;  // a multiple of 4 (HALF: of 2), at least 4
  uint32_t sc_cur[4], sc_next[4] = {0, 0, 0, 0};
  int zp_cur[4] = {0, 0, 0, 0}, zp_next[4] = {0, 0, 0, 0};
  int sta = 0;  // LDS stage of the activations of the slab being multiplied: kt % 3
  // One slab, J = kt % 4 with LEFT slabs behind it (4: four or more): requests activations two slabs ahead (and, at
  // J == 0, the packed weights and scales of the next superslab), converts the weights of slab kt + 1 between the
  // k-steps of slab kt.
  // role 0: a wavefront requests and multiplies; 1: multiplies only; 2: requests only
  constexpr auto requests_of = [](int j, int left, int role) constexpr {  // load instructions issued in such a slab
    const bool converts = role == 0 || (role == 2) == LC;
    const bool la = role != 1 && left >= AL, ls = converts && left >= 4 && j == 0;
    const bool lw = role != 1 && (W8 ? left >= AL + 1 : (left >= 4 && j == 0));
    return (la ? NA : 0) + (lw ? NQ : 0) + (ls ? kSL : 0);
  };
  auto slab = [&](int kt, auto J, auto LEFT, auto ROLE) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value, left = decltype(LEFT)::value, role = decltype(ROLE)::value;
    constexpr bool requests = role != 1, multiplies = role != 2, converts = role == 0 || (role == 2) == LC;
    constexpr bool more = left >= 1;
    constexpr bool loads_a = requests && left >= AL, loads_s = converts && left >= 4 && j == 0;
    // int8: slab kt + AL + 1; int4: the next superslab
    constexpr bool loads_w = requests && (W8 ? left >= AL + 1 : (left >= 4 && j == 0));
    constexpr bool SPREAD = multiplies;  // a wavefront that also multiplies issues one activation load per k-step
    __builtin_amdgcn_sched_barrier(0);
    const int sta_req = sta == 0 ? AST - 1 : sta - 1;
    if constexpr (loads_a && !SPREAD) issue_a(kt + AL, sta_req);
    if constexpr (loads_w) issue_raw(W8 ? kt + AL + 1 : (kt >> 2) + 1);
    if constexpr (loads_s) request_scales(sc_next, zp_next);
    __builtin_amdgcn_sched_barrier(0);
    float sc = 0.f;
    int zc = 0;
    if constexpr (converts && more) {
      // requested at j == 0 (when four slabs were left there), covered by the wait that ended j == AL - 1
      if constexpr (j == AL && left + j >= 4) pin_scales(sc_next, zp_next);
      sc = scale_value(j == 3 ? sc_next[0] : sc_cur[(j + 1) & 3]);
      zc = j == 3 ? zp_next[0] : zp_cur[(j + 1) & 3];
      convert_read(kt + 1);
    }
    if constexpr (role == 2 && converts && more) {  // the whole conversion while the requests are under way
#pragma unroll
      for (int q4 = 0; q4 < (NCQ > 4 ? NCQ : 4); ++q4) convert_quarter(q4, sc, zc);
    }
    if constexpr (multiplies) {
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
        if constexpr (loads_a && SPREAD) {  // one activation load per k-step
          if (ks < NA) QWIX_GLDS16(A + (kt + AL) * BK + goffa[ks < NA ? ks : 0], smem + sta_req * A_STAGE + (ldw * NA + ks) * 1024);
        }
        if (ks + 1 < NK) read_frags(sta, j & 1, ks + 1, (ks + 1) & 1);
        if constexpr (converts && more) convert_quarter(ks, sc, zc);
        mfma_step(ks & 1);
      }
    }
    if constexpr (converts && more) convert_write(kt + 1);
    // in flight across the barrier: the requests of this slab and of the AL - 2 before it
    constexpr int before = AL == 3 ? requests_of((j + 3) & 3, left < 4 ? left + 1 : 4, role) : 0;
    end_of_slab(integral_constant<int, requests_of(j, left, role) + before>{});
    sta = sta == AST - 1 ? 0 : sta + 1;
    if constexpr (multiplies && more) read_frags(sta, (j + 1) & 1, 0, 0);
  };
  using I0 = integral_constant<int, 0>;
  using I1 = integral_constant<int, 1>;
  using I2 = integral_constant<int, 2>;
  using I3 = integral_constant<int, 3>;
  using I4 = integral_constant<int, 4>;
  auto next_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sc_cur[e] = sc_next[e];
      zp_cur[e] = zp_next[e];
    }
  };
  auto slabs = [&](auto ROLE) __attribute__((always_inline)) {  // every role passes the same K / 64 barriers
    int kt = 0;
    // (written as 'kt + 8 <= KT' the same loop takes 102 / 135 / 200 registers in the three tiles named above)
    for (; kt + (HALF ? 6 : 4) < KT; kt += 4) {
      slab(kt, I0{}, I4{}, ROLE);
      slab(kt + 1, I1{}, I4{}, ROLE);
      slab(kt + 2, I2{}, I4{}, ROLE);
      slab(kt + 3, I3{}, I4{}, ROLE);
      next_scales();
    }
    if (HALF && (KT & 2)) {  // six left
      slab(kt, I0{}, I4{}, ROLE);
      slab(kt + 1, I1{}, I4{}, ROLE);
      slab(kt + 2, I2{}, I3{}, ROLE);
      slab(kt + 3, I3{}, I2{}, ROLE);
      next_scales();
      slab(kt + 4, I0{}, I1{}, ROLE);
      slab(kt + 5, I1{}, I0{}, ROLE);
    } else {
      slab(kt, I0{}, I3{}, ROLE);
      slab(kt + 1, I1{}, I2{}, ROLE);
      slab(kt + 2, I2{}, I1{}, ROLE);
      slab(kt + 3, I3{}, I0{}, ROLE);
    }
  };

  // ---- prologue: packed weights of slabs 0..3 (int8: 0..AL), activations of slabs 0..AL - 1, scales; slab 0 converted.
  // Two barriers for every role.
  const bool converter = !SPEC || loader == LC;  // wave-uniform
  if (!SPEC || loader) {
    issue_raw(0);
    if constexpr (W8) {
#pragma unroll
      for (int i = 1; i <= AL; ++i) issue_raw(i);
    }
#pragma unroll
    for (int i = 0; i < AL; ++i) issue_a(i, i);
  }
  // every wavefront requests them: registers of loads in flight must not pass the join of a branch
  request_scales(sc_cur, zp_cur);
  end_of_slab(integral_constant<int, 0>{});
  pin_scales(sc_cur, zp_cur);
  if (converter) {
    convert_read(0);
#pragma unroll
    for (int q4 = 0; q4 < (NCQ > 4 ? NCQ : 4); ++q4) convert_quarter(q4, scale_value(sc_cur[0]), zp_cur[0]);
    convert_write(0);
  }
  end_of_slab(integral_constant<int, 0>{});
  if constexpr (SPEC) {
    if (loader) {
      slabs(I2{});
      return;  // a wavefront that has ended no longer counts at the workgroup's barriers
    }
    read_frags(0, 0, 0, 0);
    slabs(I1{});
  } else {
    read_frags(0, 0, 0, 0);
    slabs(I0{});
  }

  float sav[TM];
  float sbv[TN][4][4];
#pragma unroll
  for (int i = 0; i < TM; ++i) sav[i] = 1.f;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd)
#pragma unroll
      for (int r = 0; r < 4; ++r) sbv[j][qd][r] = 1.f;
  const Epilogue ep{nullptr, nullptr, 0, 0, OUT, 0, 0, 0, 0, nullptr, nullptr};
  staged_epilogue<OUT, 0, TM, TN, NWAVES, LDS_BYTES, false>(acc, sav, sbv, ep, m0 + wm * WM, n0 + wn * WN, M, N, out, ldo,
                                                            smem, wave, lane);
}

}  // namespace
}  // namespace qwix

using namespace qwix;

// K in ranges for `tiles` workgroups (qwix_hip_gemm_bf16_wq_ws): elements per range, 0 = none.  The tile kernel walks K in
// slabs however few workgroups there are; while they cover at most half of the CUs, K is cut into ranges (whole 256-element
// superslabs; whole scale groups, or equal parts of one; at least 1024 elements, the last one what is left) for up to
// one workgroup per CU.
static int64_t wq_range(int64_t tiles, int64_t K, int64_t group) {
  if (tiles > 128) return 0;
  const int64_t most = std::min<int64_t>(256 / tiles, K / 1024);
  if (most < 2) return 0;
  // a range is whole superslabs, and whole scale groups or a whole part of one (never across a group's end)
  for (int64_t len = ((K + most - 1) / most + 255) / 256 * 256; len < K; len += 256) {
    const bool whole = len % group == 0 && (K % len == 0 || K % len >= 256);
    const bool part = group % len == 0 && K % len == 0;
    if (whole || part) return len;
  }
  return 0;
}

// Tile and K ranges of a call.  128 x 64 tiles up to 128 rows; 64-column tiles while 128-column ones would occupy at most half
// of the CUs, of 128 rows where twice the workgroups are one round of them and the model says so: 0.37 us per 64 of K for a
// 128 x 64 tile, 0.65 for 256 x 64, 3.5 us for the second kernel and its partials at 8 TB/s.  int4, 256 / 128 rows per tile:
// 188 x 1280 over K 2560 18.5 -> 14.7 us, 640 x 3072 over K 2048 23.1 -> 15.7, 256 x 8192 over K 4096 32.3 -> 27.6; where the taller
// tiles fill the chip with two ranges, 512 x 4096 over K 14336, 83.9 against 87.3, they stay.
struct WqPlan {
  bool low, narrow;
  int64_t range;
};
static WqPlan wq_plan(int64_t M, int64_t N, int64_t K, int64_t group) {
  WqPlan p{M <= 128, ((M + 255) / 256) * ((N + 127) / 128) <= 128, 0};
  if (M <= 0 || N <= 0 || K < 256 || group <= 0 || K % 128 || group % 64 || K % group) return p;
  const int64_t cols = (N + (p.low || p.narrow ? 63 : 127)) / (p.low || p.narrow ? 64 : 128);
  const int64_t low_tiles = (M + 127) / 128 * ((N + 63) / 64), tiles = p.low ? low_tiles : (M + 255) / 256 * cols;
  p.range = wq_range(tiles, K, group);
  if (p.low || low_tiles > 256) return p;
  auto model = [&](double per_slab, int64_t len) {
    return len == 0 ? static_cast<double>(K) / 64 * per_slab
                    : static_cast<double>(len) / 64 * per_slab + 3.5 + static_cast<double>((K + len - 1) / len * M * N) * 1e-6;
  };
  const int64_t range = wq_range(low_tiles, K, group);
  if (model(0.37, range) < 0.95 * model(0.65, p.range)) {
    p.low = true;
    p.range = range;
  }
  return p;
}
static int wq_splits(int64_t M, int64_t N, int64_t K, int64_t group) {
  const int64_t len = wq_plan(M, N, K, group).range;
  return len == 0 ? 0 : static_cast<int>((K + len - 1) / len);
}

// LDS of a workgroup: activations in three stages (where the wavefronts split the work: four), converted weights 2 x BN x 128, raw weights
// 2 x BN x 128 (bytes: 4 KB per 32 rows): at most 160 KB.
static constexpr size_t wq_lds_bytes(int bm, int bn, int bits, bool half) {
  return static_cast<size_t>(wq_stages(bm, bn, bits, half)) * bm * 128 + 2 * bn * 128 + (bits >= 8 ? 4 * (bm == 128 ? 4 : 8) * 1024 : 2 * bn * 128);
}

// Tiles whose HALF variant keeps its registers: that of 256 x 128 with int4 zero points and f32 scales spills.
static constexpr bool wq_half_fits(int bm, int bn, int bits, bool zp, bool sbf) { return !(bm == 256 && bn == 128 && bits == 4 && zp && !sbf); }

static int check_wq_args(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int q_qtype, int64_t M, int64_t N,
                         int64_t K, int64_t group, const void* s, int s_dtype, const int8_t* zp, const void* out,
                         int out_dtype, int64_t ldo) {
  if (!a || !q || !s || !out) return fail(QWIX_ERR_INVALID_ARGUMENT, "null a/q/s/out");
  if (q_qtype != QWIX_INT4 && q_qtype != QWIX_INT8 && q_qtype != QWIX_E4M3)
    return fail(QWIX_ERR_UNSUPPORTED, "weight qtype %d: int4, int8 or e4m3", q_qtype);
  if (q_qtype == QWIX_E4M3 && zp) return fail(QWIX_ERR_INVALID_ARGUMENT, "e4m3 weights have no zero point");
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || 2 * K > INT32_MAX)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad GEMM shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
                (long long)K);
  if ((out_dtype != QWIX_BF16 && out_dtype != QWIX_F32) || (s_dtype != QWIX_BF16 && s_dtype != QWIX_F32))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "scale and output dtypes must be f32 or bf16");
  // K in groups of four 64-element slabs (for int4 a 128-byte line of packed weights), the last one may
  // be half of one; a scale group covers whole slabs
  if (K < 256 || K % 128 || group <= 0 || group % 64 || K % group)
    return fail(QWIX_ERR_UNSUPPORTED, "K=%lld must be a multiple of 128 from 256 on and group=%lld a multiple of 64 that divides K",
                (long long)K, (long long)group);
  const int64_t row_bytes = q_qtype == QWIX_INT4 ? K / 2 : K;
  if (lda % 8 || lda < K || ldq_bytes % 16 || ldq_bytes < row_bytes || !aligned16(a) || !aligned16(q))
    return fail(QWIX_ERR_UNSUPPORTED, "activation and weight rows must be 16-byte aligned (lda=%lld ldq=%lld)",
                (long long)lda, (long long)ldq_bytes);
  if (ldo < N || !aligned16(out) || (N % 4 == 0 && ldo % 4 != 0))
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad output leading dimension %lld for N=%lld", (long long)ldo, (long long)N);
  if (M * lda * 2 >= (int64_t{1} << 31) || N * ldq_bytes >= (int64_t{1} << 31))
    return fail(QWIX_ERR_UNSUPPORTED, "operands beyond 2 GiB are not supported");
  return QWIX_OK;
}

static int gemm_bf16_wq_impl(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int q_qtype, int64_t M,
                             int64_t N, int64_t K, int64_t group, const void* s, int s_dtype, const int8_t* zp,
                             void* out, int out_dtype, int64_t ldo, void* stream, void* workspace,
                             size_t workspace_bytes) {
  if (const int rc = check_wq_args(a, lda, q, ldq_bytes, q_qtype, M, N, K, group, s, s_dtype, zp, out, out_dtype, ldo))
    return rc;
  const WqPlan plan = wq_plan(M, N, K, group);
  const bool low = plan.low, narrow = plan.narrow;
  // 192-row tiles where they need no more rounds of the CUs than the 256-row ones
  auto rounds = [&](int64_t rows) { return ((M + rows - 1) / rows * ((N + 127) / 128) + 255) / 256; };
  const bool half = K % 256 != 0;
  const bool mid = rounds(192) <= rounds(256) || (half && !wq_half_fits(256, 128, q_qtype == QWIX_INT4 ? 4 : 8, zp != nullptr, s_dtype == QWIX_BF16));
  hipStream_t st = static_cast<hipStream_t>(stream);
  // with a workspace that holds them: f32 partials of `splits` K ranges, added up (in range order) by a second kernel
  int splits = workspace && plan.range > 0 ? static_cast<int>((K + plan.range - 1) / plan.range) : 0;
  if (splits > 0 && (workspace_bytes < static_cast<size_t>(splits) * M * N * 4 || !aligned16(workspace))) splits = 0;
  const int ksplit = splits > 0 ? static_cast<int>(plan.range) : 0;
  const int kern_out = splits > 0 ? QWIX_F32 : out_dtype;
  uint8_t* const kern_dst = static_cast<uint8_t*>(splits > 0 ? workspace : out);
  const int64_t kern_ldo = splits > 0 ? N : ldo;
#define QWIX_WQ_LAUNCH(OUTT, SBFF, BMM, BNN, BITS) \
  do {                                             \
    if (zp) QWIX_WQ_LAUNCH_Z(OUTT, SBFF, BMM, BNN, BITS, (BITS != 9)); else QWIX_WQ_LAUNCH_Z(OUTT, SBFF, BMM, BNN, BITS, false); \
  } while (0)
#define QWIX_WQ_LAUNCH_Z(OUTT, SBFF, BMM, BNN, BITS, ZPP)                                                            \
  do {                                                                                                               \
    auto kern = half ? wgemm_wq_kernel<OUTT, SBFF, BMM, BNN, BITS, ZPP, wq_half_fits(BMM, BNN, BITS, ZPP, SBFF)>      \
                     : wgemm_wq_kernel<OUTT, SBFF, BMM, BNN, BITS, ZPP, false>;                                      \
    const size_t smem = wq_lds_bytes(BMM, BNN, BITS, half && wq_half_fits(BMM, BNN, BITS, ZPP, SBFF));                \
    const dim3 grid(static_cast<unsigned>(((M + BMM - 1) / BMM) * ((N + BNN - 1) / BNN)),                            \
                    static_cast<unsigned>(splits > 0 ? splits : 1));                                                 \
    static LdsGrant granted[2];                                                                                      \
    if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted[half])) return e_;                     \
    kern<<<grid, 512, smem, st>>>(static_cast<const uint8_t*>(a), 2 * lda, static_cast<const uint8_t*>(q), ldq_bytes, s, \
                                  zp, static_cast<int>(M), static_cast<int>(N), static_cast<int>(K),                 \
                                  static_cast<int>(group), kern_dst, kern_ldo, ksplit, NoGroups{});                            \
  } while (0)
#define QWIX_WQ_TILE(OUTT, SBFF, BITS)                                                                               \
  do {                                                                                                               \
    if (low) QWIX_WQ_LAUNCH(OUTT, SBFF, 128, 64, BITS);                                                              \
    else if (narrow) QWIX_WQ_LAUNCH(OUTT, SBFF, 256, 64, BITS);                                                      \
    else if (mid) QWIX_WQ_LAUNCH(OUTT, SBFF, 192, 128, BITS);                                                        \
    else QWIX_WQ_LAUNCH(OUTT, SBFF, 256, 128, BITS);                                                                 \
  } while (0)
#define QWIX_WQ_BITS(OUTT, SBFF)                                                                                     \
  do {                                                                                                               \
    if (q_qtype == QWIX_INT4) QWIX_WQ_TILE(OUTT, SBFF, 4);                                                           \
    else if (q_qtype == QWIX_INT8) QWIX_WQ_TILE(OUTT, SBFF, 8);                                                      \
    else QWIX_WQ_TILE(OUTT, SBFF, 9); /* e4m3 */                                                                     \
  } while (0)
  if (kern_out == QWIX_BF16) {
    if (s_dtype == QWIX_BF16) QWIX_WQ_BITS(QWIX_BF16, true); else QWIX_WQ_BITS(QWIX_BF16, false);
  } else {
    if (s_dtype == QWIX_BF16) QWIX_WQ_BITS(QWIX_F32, true); else QWIX_WQ_BITS(QWIX_F32, false);
  }
#undef QWIX_WQ_BITS
#undef QWIX_WQ_TILE
#undef QWIX_WQ_LAUNCH
#undef QWIX_WQ_LAUNCH_Z
  if (int e = check_launch("gemm_bf16_wq")) return e;
  if (splits > 0) {
    const Epilogue ep{nullptr, nullptr, 0, 0, out_dtype, 0, 0, 0, 0, nullptr, nullptr};
    const int64_t threads = (M * N + 3) / 4;
    splitk_reduce_kernel<false><<<dim3(static_cast<unsigned>((threads + 255) / 256)), 256, 0, st>>>(
        static_cast<const uint8_t*>(workspace), splits, static_cast<int>(M), static_cast<int>(N), ep,
        static_cast<uint8_t*>(out), ldo);
    return check_launch("gemm_bf16_wq (split K)");
  }
  return 0;
}

extern "C" int qwix_hip_gemm_bf16_wq(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int q_qtype, int64_t M,
                                     int64_t N, int64_t K, int64_t group, const void* s, int s_dtype, const int8_t* zp,
                                     void* out, int out_dtype, int64_t ldo, void* stream) {
  if (K % 256) return fail(QWIX_ERR_UNSUPPORTED, "K=%lld must be a multiple of 256", (long long)K);
  return gemm_bf16_wq_impl(a, lda, q, ldq_bytes, q_qtype, M, N, K, group, s, s_dtype, zp, out, out_dtype, ldo, stream,
                           nullptr, 0);
}

extern "C" size_t qwix_hip_gemm_bf16_wq_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t group) {
  return static_cast<size_t>(wq_splits(M, N, K, group)) * static_cast<size_t>(M > 0 ? M : 0) * static_cast<size_t>(N > 0 ? N : 0) * 4;
}

extern "C" int qwix_hip_gemm_bf16_wq_ws(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int q_qtype,
                                        int64_t M, int64_t N, int64_t K, int64_t group, const void* s, int s_dtype,
                                        const int8_t* zp, void* out, int out_dtype, int64_t ldo, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  return gemm_bf16_wq_impl(a, lda, q, ldq_bytes, q_qtype, M, N, K, group, s, s_dtype, zp, out, out_dtype, ldo, stream,
                           workspace, workspace_bytes);
}

static int wq_ragged(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int64_t q_group_stride, int q_qtype,
                     int64_t M, int64_t N, int64_t K, int64_t group, const void* s, int s_dtype, int64_t s_group_stride,
                     const int32_t* group_sizes, int64_t G, int64_t stream_rows, void* out, int out_dtype, int64_t ldo,
                     void* stream) {
  if (const int rc = check_wq_args(a, lda, q, ldq_bytes, q_qtype, M, N, K, group, s, s_dtype, nullptr, out, out_dtype, ldo))
    return rc;
  if (!group_sizes || G <= 0 || G > 65536)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "1..65536 group sizes are needed (G=%lld)", (long long)G);
  if (q_group_stride % 16 || q_group_stride < 0 || s_group_stride < 0)
    return fail(QWIX_ERR_INVALID_ARGUMENT, "bad group strides (weights: %lld bytes, scales: %lld elements)",
                (long long)q_group_stride, (long long)s_group_stride);
  if ((M / 128 + G + 1) * ((N + 63) / 64) >= (int64_t{1} << 30))
    return fail(QWIX_ERR_UNSUPPORTED, "too many tiles (M=%lld N=%lld G=%lld)", (long long)M, (long long)N, (long long)G);
  if (stream_rows > 0) {
    if (const int rc = gemv_wq_groups(a, lda, q, ldq_bytes, q_group_stride, q_qtype, M, N, K, group, s, s_dtype, s_group_stride,
                                      group_sizes, G, stream_rows, out, out_dtype, ldo, stream))
      return rc;
    if (stream_rows >= M) return QWIX_OK;
  }
  const Ragged rg{group_sizes, static_cast<int>(G), static_cast<int>(stream_rows), q_group_stride, s_group_stride};
  hipStream_t st = static_cast<hipStream_t>(stream);
  // Up to 80 rows per group on average most groups fit 128 rows; 64-column tiles while 128-column ones would occupy at most
  // half of the CUs.  Tiles of 128 x 64 / 256 x 128, 64 and 96 rows per group on average, some groups up to half as many
  // again: 64 groups, K 2048, N 1024, int8 72 / 71 and 88 / 75 us; 8 groups, K 2176, N 5312 56 / 71 and 73 / 72 us; 8 groups,
  // K 4096, N 14336, int4 193 / 230 and 217 / 233 us; 128 rows 312 / 236 us.  A group with nearly all rows has its weight converted
  // once per row tile; sizes are not known here.  Such calls group by group / here, 640 rows in 8 groups, all but 28 in one, K 4096,
  // N 14336: int4 324 / 177 us, int8 334 / 215; 1280 rows int4 353 / 229, int8 398 / 280; 140 rows in 2 groups int8 119 / 74.
  const bool half = K % 256 != 0;  // (groups of more than 256 rows, where dot_general's rule says what is streamed)
  const int tile = M <= 80 * G && !half ? 0 : (M / 256 + G) * ((N + 127) / 128) <= 128 ? 1 : 2;
#define QWIX_WQR(OUTT, SBFF, BMM, BNN, BITS)                                                                         \
  do {                                                                                                               \
    auto kern = half ? wgemm_wq_kernel<OUTT, SBFF, BMM, BNN, BITS, false, (BMM > 128), true>                         \
                     : wgemm_wq_kernel<OUTT, SBFF, BMM, BNN, BITS, false, false, true>;                              \
    const size_t smem = wq_lds_bytes(BMM, BNN, BITS, half && (BMM > 128));                                            \
    static LdsGrant granted[2];                                                                                      \
    if (int e_ = grant_lds(reinterpret_cast<const void*>(kern), smem, granted[half])) return e_;                     \
    kern<<<dim3(ragged_grid(M, N, G, BMM, BNN)), 512, smem, st>>>(                                                   \
        static_cast<const uint8_t*>(a), 2 * lda, static_cast<const uint8_t*>(q), ldq_bytes, s, nullptr,              \
        static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), static_cast<int>(group),                      \
        static_cast<uint8_t*>(out), ldo, 0, rg);                                                                     \
  } while (0)
#define QWIX_WQR_TILE(OUTT, SBFF, BITS)                       \
  do {                                                        \
    if (tile == 0) QWIX_WQR(OUTT, SBFF, 128, 64, BITS);       \
    else if (tile == 1) QWIX_WQR(OUTT, SBFF, 256, 64, BITS);  \
    else QWIX_WQR(OUTT, SBFF, 256, 128, BITS);                \
  } while (0)
#define QWIX_WQR_BITS(OUTT, SBFF)                               \
  do {                                                          \
    if (q_qtype == QWIX_INT4) QWIX_WQR_TILE(OUTT, SBFF, 4);     \
    else if (q_qtype == QWIX_INT8) QWIX_WQR_TILE(OUTT, SBFF, 8); \
    else QWIX_WQR_TILE(OUTT, SBFF, 9);                          \
  } while (0)
  if (out_dtype == QWIX_BF16) {
    if (s_dtype == QWIX_BF16) QWIX_WQR_BITS(QWIX_BF16, true); else QWIX_WQR_BITS(QWIX_BF16, false);
  } else {
    if (s_dtype == QWIX_BF16) QWIX_WQR_BITS(QWIX_F32, true); else QWIX_WQR_BITS(QWIX_F32, false);
  }
#undef QWIX_WQR_BITS
#undef QWIX_WQR_TILE
#undef QWIX_WQR
  return check_launch("gemm_bf16_wq (ragged)");
}

extern "C" int qwix_hip_gemm_bf16_wq_ragged(const void* a, int64_t lda, const void* q, int64_t ldq_bytes,
                                            int64_t q_group_stride, int q_qtype, int64_t M, int64_t N, int64_t K,
                                            int64_t group, const void* s, int s_dtype, int64_t s_group_stride,
                                            const int32_t* group_sizes, int64_t G, void* out, int out_dtype, int64_t ldo,
                                            void* stream) {
  return wq_ragged(a, lda, q, ldq_bytes, q_group_stride, q_qtype, M, N, K, group, s, s_dtype, s_group_stride, group_sizes, G, 0,
                   out, out_dtype, ldo, stream);
}

// Two launches over the same group sizes, each with the groups of its kind.
extern "C" int qwix_hip_gemm_wq_groups(const void* a, int64_t lda, const void* q, int64_t ldq_bytes, int64_t q_group_stride,
                                       int q_qtype, int64_t M, int64_t N, int64_t K, int64_t group, const void* s, int s_dtype,
                                       int64_t s_group_stride, const int32_t* group_sizes, int64_t G, int64_t stream_rows,
                                       void* out, int out_dtype, int64_t ldo, void* stream) {
  if (stream_rows < 0) return fail(QWIX_ERR_INVALID_ARGUMENT, "stream_rows=%lld is negative", (long long)stream_rows);
  return wq_ragged(a, lda, q, ldq_bytes, q_group_stride, q_qtype, M, N, K, group, s, s_dtype, s_group_stride, group_sizes, G,
                   std::min(stream_rows, M), out, out_dtype, ldo, stream);
}
