// tanh in double precision for kernels that the FP64 pipe bounds: 1 - 2 /
// (e^2x + 1) with e^2x = 2^(n/32) p(r), 2^(j/32) from a table that the
// workgroup keeps in LDS.
#pragma once

#include "dpk_common.h"

namespace dpk {
namespace {

// 2^(j/32), correctly rounded
__constant__ double kExp2Tab[32] = {
    0x1.0000000000000p+0, 0x1.059b0d3158574p+0, 0x1.0b5586cf9890fp+0, 0x1.11301d0125b51p+0,
    0x1.172b83c7d517bp+0, 0x1.1d4873168b9aap+0, 0x1.2387a6e756238p+0, 0x1.29e9df51fdee1p+0,
    0x1.306fe0a31b715p+0, 0x1.371a7373aa9cbp+0, 0x1.3dea64c123422p+0, 0x1.44e086061892dp+0,
    0x1.4bfdad5362a27p+0, 0x1.5342b569d4f82p+0, 0x1.5ab07dd485429p+0, 0x1.6247eb03a5585p+0,
    0x1.6a09e667f3bcdp+0, 0x1.71f75e8ec5f74p+0, 0x1.7a11473eb0187p+0, 0x1.82589994cce13p+0,
    0x1.8ace5422aa0dbp+0, 0x1.93737b0cdc5e5p+0, 0x1.9c49182a3f090p+0, 0x1.a5503b23e255dp+0,
    0x1.ae89f995ad3adp+0, 0x1.b7f76f2fb5e47p+0, 0x1.c199bdd85529cp+0, 0x1.cb720dcef9069p+0,
    0x1.d5818dcfba487p+0, 0x1.dfc97337b9b5fp+0, 0x1.ea4afa2a490dap+0, 0x1.f50765b6e4540p+0};

// tanh(x), absolute error about an ulp of 1.  |x| is clamped near 20 (tanh is
// +-1 there in FP64) in its high word; a NaN passes through.
__device__ __forceinline__ double tanh64(double x, const double* tab) {
  constexpr double K = 0x1.71547652b82fep+6;   // 2 * 32 / ln 2
  constexpr double kMagic = 0x1.8p+52;
  const unsigned hi = (unsigned)__double2hiint(x), a = hi & 0x7fffffffu;
  const unsigned lim = a > 0x7ff00000u ? a : (a < 0x40340000u ? a : 0x40340000u);
  const double xc = __hiloint2double((int)(lim | (hi & 0x80000000u)), __double2loint(x));
  const double ym = __fma_rn(xc, K, kMagic);
  const int n = __double2loint(ym);
  const double r = __fma_rn(xc, K, -(ym - kMagic));
  const double t0 = tab[n & 31];
  const double t = __hiloint2double(__double2hiint(t0) + (int)((unsigned)(n & ~31) << 15), __double2loint(t0));
  // (e^(r ln2/32) - 1) / r on |r| <= 1/2, interpolated at the Chebyshev nodes
  double p = __fma_rn(r, 0x1.5d884e708e6aap-35, 0x1.3b2b1bee88b09p-27);
  p = __fma_rn(r, p, 0x1.c6b08d70400d0p-20);
  p = __fma_rn(r, p, 0x1.ebfbdff8131c3p-13);
  p = __fma_rn(r, p, 0x1.62e42fefa39efp-6);
  p = __fma_rn(r, p, 1.0);
  const double d = __fma_rn(t, p, 1.0);        // e^2x + 1
  const double q0 = __builtin_amdgcn_rcp(d);
  const double e = __fma_rn(-d, q0, 1.0);
  const double q = __fma_rn(q0, __fma_rn(e, e, e), q0);
  return __fma_rn(-2.0, q, 1.0);
}

}  // namespace
}  // namespace dpk
