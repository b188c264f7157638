// Batched GEMM with a short contraction along strips of rows (qgemm_strips.hip), called by qwix_hip_qgemm_batched.
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

}  // namespace qwix
