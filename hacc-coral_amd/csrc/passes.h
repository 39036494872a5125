// passes.h -- how the targets of a leaf are split into the passes of the
// leaf and adjoint kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Target slots (a power of two, at least 4 R) of the next pass over a leaf
// with `rem` targets left, R targets per lane, at most pmax a pass.  A pass
// works for all its slots, used or not, and stages the whole list once.  With
// the chip full of waves the staging costs a pass about what 4 slots do;
// where few waves share a SIMD (thin) its loads are not hidden and it costs
// about 16.  So the remainder above a power of two c goes into one pass of
// 2 c slots when splitting it into c and smaller powers would cost more.
// Against powers of two down to 8 and then the rest: leaf kernel 0.40 ->
// 0.35 ms at 61^3 (quadrupole, leaves of 100), 0.033 -> 0.020 ms at 16^3
// (leaves of 32), 8.77 -> 8.53 ms for 24 boxes of 20^3..64^3 (leaves of 256).
// The fused adjoint takes the same passes, though its pairs cost three times
// as much beside the staging.  Powers of two and this rule there: 0.21 and 0.19
// ms at 16^3 (leaves of 32), 0.26 and 0.25 at 32^3 (50), 12.12 and 11.84 at
// 64^3 (64), 10.82 and 10.79 (100), 61.5 and 62.2 at 128^3 (100), 453.4 and
// 455.5 at 256^3 (384), each with its hot loop at its best place (loop_offset).
template <int R>
__host__ __device__ inline int pass_slots(int64_t rem, int pmax, bool thin) {
  if (rem >= pmax) return pmax;
  int c = 4 * R;
  while (2 * c <= rem) c *= 2;
  if (rem <= c) return c;  // also fewer than 4 R targets
  const int over = (int)rem - c;
  const int split = thin ? (c <= 16 ? 0 : (c <= 32 ? 8 : c / 2))   // the largest part
                         : (c <= 8 ? 0 : (c <= 16 ? 8 : 3 * c / 4));  // worth its own pass
  return over > split && 2 * c <= pmax ? 2 * c : c;
}
