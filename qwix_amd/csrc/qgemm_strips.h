// Batched GEMM with a short contraction along strips of rows (qgemm_strips.hip) and with a long one by wavefronts that split it
// (qgemm_long.hip), called by qwix_hip_qgemm_batched.
#pragma once
#include <stdint.h>

namespace qwix {

struct StripArgs {
  const uint8_t* a;
  int64_t lda, a_stride;  // bytes; strides between consecutive problems
  const uint8_t* b;
  int64_t ldb, b_stride;
  const void* sa;
  int64_t sa_stride;      // elements
  const void* sb;
  int64_t sb_stride;
  uint8_t* out;
  int64_t ldo, out_stride;  // elements
  int M, N;
};

// K is 64 or 128; bf16: scales and results in bf16 with every step rounded, else f32 throughout.  The caller has checked the
// operands: 16-byte aligned rows of a and b, N and the strides of sb multiples of 4, whole aligned 16-byte pieces of
// out, and 32-bit byte offsets over b and over M + 128 rows of out.
int qgemm_strips(int qtype, int64_t K, bool bf16, const StripArgs& p, int64_t batch, void* stream);

// The same from bf16 rows of both, quantized in the kernel, for up to 64 rows of a (strides in bytes of them, sa and sb unused).
int qgemm_strips_act(int qtype, int64_t K, const StripArgs& p, int64_t batch, void* stream);

struct LongArgs {
  const uint8_t* a;
  int64_t lda, a_stride;  // bytes; strides between consecutive problems
  const uint8_t* b;
  int64_t ldb, b_stride;
  const void* sa;         // per row, or null
  int sa_dtype;
  int64_t sa_stride;      // elements
  const void* sb;         // per column, or null
  int sb_dtype;
  int64_t sb_stride;
  int r0, r1, r2;         // which steps of ((T(acc) * sa) * sb) round to bf16
  uint8_t* out;
  int out_dtype;
  int64_t ldo, out_stride;  // elements
  int M, N, K;
};

// f32 or bf16 results.  The caller has checked the operands: K a multiple of 16, 16-byte aligned rows of a and b, 32-bit byte
// offsets over one problem of each, N, ldo and out_stride multiples of 4.
bool qgemm_long_takes(int64_t M, int64_t N, int64_t K, int64_t batch);
int qgemm_long(int qtype, const LongArgs& p, int64_t batch, void* stream);

}  // namespace qwix
