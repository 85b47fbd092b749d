// Kernel entries for the kernels that evaluate them by the billion: the value
// of kernel_eval to an ulp or two, without its correctly rounded square root and
// division and the general exponential's range checks (about 35 vector
// instructions an entry for Yukawa, 70 with kernel_eval).
#pragma once

#include <cfloat>

#include "common.hpp"

namespace mxg {

// 2^f for |f| <= 1/2: interpolation at 12 Chebyshev nodes (error 2e-17)
__device__ inline double exp2_poly(double f) {
  double p = 4.4558179083360645e-10;
  p = fma(p, f, 7.074194297288521e-09);
  p = fma(p, f, 1.0178057087733941e-07);
  p = fma(p, f, 1.3215432535912375e-06);
  p = fma(p, f, 1.5252733841556773e-05);
  p = fma(p, f, 0.00015403530463724353);
  p = fma(p, f, 0.001333355814640647);
  p = fma(p, f, 0.009618129107587256);
  p = fma(p, f, 0.055504108664821625);
  p = fma(p, f, 0.24022650695910158);
  p = fma(p, f, 0.6931471805599453);
  return fma(p, f, 1.0);
}

// What the evaluation needs of a kernel: K(0), -alpha log2(e) as the unevaluated
// sum of two doubles, the largest squared distance that kernel_scaled is for, and
// the largest coordinate whose distances all are that small.
struct EvalArgs {
  double diag, ch, cl, far2, reach;
};

inline EvalArgs eval_args(mxg_kernel_t k) {
  // the product's rounding error and log2(e)'s own tail make the second part
  const double L2E = 1.4426950408889634, L2E_TAIL = 2.0355273740931033e-17, ch = -k.alpha * L2E;
  double far2 = DBL_MAX;
  if (k.id == MXG_KERNEL_YUKAWA || k.id == MXG_KERNEL_GAUSSIAN) {
    // an exponent of at most 2^30 in magnitude
    const double d = 1073741824.0 / std::fabs(ch), d2 = k.id == MXG_KERNEL_YUKAWA ? d * d : d;
    far2 = d2 >= DBL_MIN ? std::min(d2, far2) : 0.;
  }
  // 12 reach^2 < far2
  return EvalArgs{k.id == MXG_KERNEL_GAUSSIAN ? 1.0001 : k.diag, ch, std::fma(-k.alpha, L2E, -ch) - k.alpha * L2E_TAIL, far2,
                  std::sqrt(far2) * 0.288};
}

// 1 / sqrt(x) from the hardware's estimate y and the first terms of the binomial
// series of (1 - e)^(-1/2), e = 1 - x y^2.
__device__ inline double rsqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// K(d) 2^shift from a squared distance above zero and up to far2.
template <int KID>
__device__ inline double kernel_scaled(double d2, const EvalArgs& k, int shift) {
  if constexpr (KID == MXG_KERNEL_LAPLACE) {
    return ldexp(rsqrt_refined(d2), shift);
  } else {
    const double v = KID == MXG_KERNEL_YUKAWA ? rsqrt_refined(d2) : 1.0;
    const double d = KID == MXG_KERNEL_YUKAWA ? d2 * v : d2;
    const double y = d * k.ch, r = rint(y);
    double p = exp2_poly(fma(d, k.cl, fma(d, k.ch, -r)));
    if constexpr (KID == MXG_KERNEL_YUKAWA) p *= v;
    return ldexp(p, (int)r + shift);
  }
}

// K(d) from any squared distance, as kernel_eval gives it: infinite ones, whose
// entries are zero where the steps of rsqrt_refined give NaN, exponents beyond an
// int, and NaN.
template <int KID>
__device__ inline double kernel_any(double d2, const EvalArgs& k) {
  const double d = KID == MXG_KERNEL_GAUSSIAN ? d2 : sqrt(d2);
  double v = 1.0;
  if constexpr (KID != MXG_KERNEL_LAPLACE) {
    const double y = d * k.ch, r = rint(y);
    v = ldexp(exp2_poly(fma(d, k.cl, fma(d, k.ch, -r))), (int)r);
    if (!(fabs(y) <= 1073741824.0)) v = y < 0. ? 0. : y * __builtin_inf();
  }
  if constexpr (KID != MXG_KERNEL_GAUSSIAN) v /= d;
  return d2 == 0. ? k.diag : v;
}

}  // namespace mxg
