// Arguments of the sub-channel GEMM kernels (qgemm_grouped.hip), and the entry of the ones that stand in a file of their own
// (qgemm_grouped_wide.hip).
#pragma once
#include <stdint.h>

namespace qwix {

struct GroupedArgs {
  const uint8_t* A; int64_t lda;
  const uint8_t* B; int64_t ldb;
  int M, N, K, group;
  const void* sa; int sa_dtype; int ga;
  const void* sb; int sb_dtype;
  int t_dtype;      // dtype of the scaled partials (promotion of the scale dtypes, and of acc_dtype for e4m3)
  int acc_dtype;    // e4m3 operands: the dtype each group's f32 dot is rounded to before it is scaled
  uint8_t* out; int out_dtype; int64_t ldo;
  int32_t* acc_out;
  // Zero-point correction of an asymmetric operand, per group: acc_g[m,n] -= zu[m,g] * zv[g,n].  One array
  // holds zero points, the other the per-group K-sums of the opposite operand; element strides, 0 along the
  // group axis for an array that is the same for all groups.  Both null: symmetric operands.
  const int32_t* zu; int64_t zu_sm, zu_sg;
  const int32_t* zv; int64_t zv_sn, zv_sg;
  // One group spans all of K (int4 weights with per-channel scales): the fast kernel then scales like the untiled
  // contraction, ((T(acc) * sx) * sy) with a rounding per step (dot_general.py:255-261), not like a sum of partials.
  int single;
  // K in ranges (0: none): workgroups with blockIdx.y = y contract elements [y ksplit, (y + 1) ksplit) -- whole groups --
  // and write the f32 sums of their scaled partials, without the activation scale and the final rounding, as the y-th
  // M x N array at `out` (the host passes f32, ldo = N, sa = null); grouped_reduce_kernel finishes.
  int ksplit;
};

// 256-column tiles of 64 by 64 to 128 by 64 per wavefront, groups of 128, bf16 scales: per column and group, with `outer` per
// row and group as well.  The caller has checked the operands as for the 128 x 256 tiles.
int qgemm_grouped_wide(const GroupedArgs& p, int b_qtype, bool outer, int tm, void* stream);

}  // namespace qwix
