// Regions of the B^T Z + Z^T B work items and their wanted blocks, shared by
// the FP64 and the mixed kernel (gemm_fp64.hip, gemm_mixed.hip).
#pragma once
#include "internal.hpp"

namespace xcq {

// Region of an item: blocks of 16 functions, rows [r0, r1) and columns [c0,
// c1), without the rows above and the columns right of its part on or below
// the diagonal, so c0 <= r0 and c1 <= r1.
struct SyrRegion {
  int r0, r1, c0, c1;
};
template <bool MX>
__device__ __forceinline__ SyrRegion syr_region(const DevTask& t, int a, int b) {
  const int nb = (t.nbe + 15) / 16;
  const int ni = syr_row_groups<MX>(nb), nj = syr_col_groups<MX>(nb);
  const int r1 = (a + 1) * nb / ni, c0 = b * nb / nj;
  return SyrRegion{max(a * nb / ni, c0), r1, c0, min((b + 1) * nb / nj, r1)};
}

// The region's wanted blocks, bit (row - r0) * (c1 - c0) + column - c0: on or
// below the diagonal, and not negligible by the bound table, |sum_p B_pi
// Z_pj| <= npts max|B_i| max|Z_j| (1.01 covers the rounding of the stored
// maxima and of the products).  Lane l of a wave decides bit l (a region has
// at most 64 blocks).
__device__ __forceinline__ uint64_t syr_mask(const DevTask& t, const SyrRegion& s, int lane,
                                             const unsigned* tmax, double drop) {
  const int nc = s.c1 - s.c0;
  const int rb = s.r0 + lane / nc, cb = s.c0 + lane % nc;
  bool want = rb < s.r1 && rb >= cb;
  if (want && tmax) {
    const unsigned* tm = tmax + 2 * t.tmax_off;
    const int gi = 16 * rb / kGran, gj = 16 * cb / kGran;
    const double bound =
        1.01 * (double)t.npts *
        ((double)__uint_as_float(tm[2 * gi]) * (double)__uint_as_float(tm[2 * gj + 1]) +
         (double)__uint_as_float(tm[2 * gi + 1]) * (double)__uint_as_float(tm[2 * gj]));
    want = !(bound < drop);
  }
  return __builtin_amdgcn_ballot_w64(want);
}

}  // namespace xcq
