// The FP64 weight chain of the mixed-precision kernels (one-ulp square root
// and reciprocal in the reference's order), shared by the mixed Generate,
// AverageOn and regenerating scatter (genbod_mixed.hip) and the mixed
// Unweight's flags (generate_unweight.hip).  Every function turns
// contraction off itself, so the bits do not depend on the translation
// unit's flags.
#pragma once

#include <type_traits>

#include "hpsp_launch.h"

namespace hpsp {

// FP64 weight chain of DecayMother::process (DecayMother.h:170-212):
// sorted uniforms, invMas, pdk and the weight product in the reference's
// order (so the a - b - c cancellation near threshold is the FP64 one), pdk
// with a one-ulp square root and reciprocal instead of correctly rounded ones.
// The momenta pd and invMas[1 .. N-2], which the boosts take, are handed on in
// FP32.
template <int N, int ENGINE, typename WordFn>
__device__ __forceinline__ double weight_chain(const DecayK& d, const WordFn& word,
                                               float (&pd)[N - 1], float (&mas)[N - 1]) {
#pragma clang fp contract(off)
  double rno[N];
  rno[0] = 0.0;
  rno[N - 1] = 1.0;
  if constexpr (N > 2) {
    using WT = std::conditional_t<is_squares<ENGINE>(), uint32_t, uint64_t>;
    WT v[N - 2];
#pragma unroll
    for (int k = 0; k < N - 2; ++k) v[k] = (WT)word(k);
    sort_net(v);
#pragma unroll
    for (int k = 0; k < N - 2; ++k) rno[k + 1] = to_unit<ENGINE>(v[k]);
  }
  double wt = d.maxw;
  double c = d.mas0;
#pragma unroll
  for (int n = 0; n < N - 1; ++n) {
    const double a = n < N - 2 ? rno[n + 1] * d.ecm + d.msum[n + 1] : d.masN;
    const double r = n < N - 2 ? rcp_fast(a) : d.rmasN;
    const double q = sqrt_fast(pdk_radicand(a, c, d.m[n + 1])) * (0.5 * r);
    wt *= q;
    pd[n] = (float)q;
    if (n + 1 < N - 1) mas[n + 1] = (float)a;
    c = a;
  }
  return wt;
}

}  // namespace hpsp
