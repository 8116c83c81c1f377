// What the attention kernels' softmaxes have in common.
#ifndef ILT_SOFTMAX_H
#define ILT_SOFTMAX_H
#include "ilt_device.h"

namespace {

// What one lane of a wave stored in LDS, for the other lanes of that wave: the hardware keeps a wave's LDS
// accesses in program order; this keeps the compiler from moving them across.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The softmax's 1/sum as the CPU rounds it to a single, from a sum of n exps added in another order than the CPU's: one
// division, then whether every sum that the CPU's could be has the same single for its reciprocal.  No term is negative, so
// the CPU's n - 1 adds one after another leave a double within (n - 1) 2^-53 of the exact sum, relatively, and a sum whose
// terms go through at most ADDS adds each one within ADDS 2^-53; each of the two divisions and the bounds' own subtraction
// and addition round once more, and what is of second order is under 2^-53 in all for fewer than 2^26 terms.  That is
// n + ADDS + 3 of the n + 128 taken, and rounding to single keeps the reciprocals' order.  False: the caller adds the exps
// again in the CPU's order.
template <int ADDS>
__device__ __forceinline__ bool recip_settled(double sum, int n, float* inv) {
  static_assert(ADDS + 3 <= 128, "more adds than the bound counts");
  const double r = 1.0 / sum, d = (double)(n + 128) * 0x1p-53;
  *inv = (float)r;
  return (float)(r - r * d) == (float)(r + r * d);
}
// The adds that a term goes through in a sum by threads: a thread's own TERMS one after another (the first to nothing), a
// wave's six (wave_sum_double), and what the waves' sums take.
constexpr int sum_adds(int terms, int waves) { return terms - 1 + 6 + waves; }

}  // namespace

#endif  // ILT_SOFTMAX_H
