// How many K slices each tile of a ragged-M launch of few tiles is cut in.
#pragma once

namespace fm {

// One tile alone takes 1.1 to 1.9 us a step (its loads, a step or two in flight,
// wait for memory: weights of experts with few tokens are read once), and the
// idle CUs take the other slices.  The time of s slices in steps (a step as
// 1.4 us for BF16, 1.15 us for FP8): nk / s, a launch (5 for BF16, 6.5 for FP8), and the
// partials' way out and back, 0.1 us a slice and tile (1/14, 1/11).  At least 8 steps
// a slice; `by_cu` slices at most fit the CUs.
// In integers, as fractions over s: the slicing kernel and the one that sums the
// slices each work it out and must agree, also where two counts cost the same
// (16 BF16 tiles of 64 steps in 7 or in 8; more slices, whose steps divide more
// evenly, then).  As floats the choice there was the compiler's, by whether it fused
// a multiply and an add.
constexpr int kSliceSteps = 8, kMaxSlices = 8;
__device__ __forceinline__ int slice_count(int tiles, int by_cu, int nk, bool bf16) {
  const int by_k = nk / kSliceSteps, part = bf16 ? 14 : 11, launch2 = bf16 ? 10 : 13;
  int best = 1;
  long long cost = 2ll * part * nk;   // x 2 part s: 2 part nk + part (2 launch) s + 2 tiles s^2
  for (int s = 2; s <= kMaxSlices && s <= by_cu && s <= by_k; ++s) {
    const long long c = 2ll * part * nk + part * launch2 * s + 2ll * tiles * s * s;
    const long long a = c * best, b = cost * s;
    if (a < b || (a == b && best > 1)) {
      cost = c;
      best = s;
    }
  }
  return best;
}

}  // namespace fm
