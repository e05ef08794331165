// The step of the SSF partition (Stratmann, Scuseria and Frisch), shared by the
// weights and their derivatives.
#pragma once
#include "internal.hpp"

namespace xcq {

constexpr double kSsfA = 0.64;

// s(mu) at v = mu / a: 1 below -1, 0 above 1, (1 - g(v)) / 2 with the Frisch
// polynomial g between; its values at the clamped ends are exact.  A NaN (two
// atoms at one place) gives 0.
__device__ __forceinline__ double ssf_s(double v) {
  v = fmax(fmin(v, 1.), -1.);
  const double v2 = v * v;
  const double g = v * (35. + v2 * (-35. + v2 * (21. - 5. * v2))) * 0.0625;
  return 0.5 * (1. - g);
}

}  // namespace xcq
