// exprel.h -- relative exponentials of the Taylor-Duffy integrands.
#pragma once

#include "devmath.h"

namespace scuffx {

// complex products by fused multiply-adds: a b + c and a b
__device__ inline cplx cfma(cplx a, cplx b, cplx c)
{
  return mk(fma(a.r, b.r, fma(-a.i, b.i, c.r)), fma(a.r, b.i, fma(a.i, b.r, c.i)));
}
__device__ inline cplx cmulf(cplx a, cplx b) { return mk(fma(a.r, b.r, -(a.i * b.i)), fma(a.r, b.i, a.i * b.r)); }

#define TD_NER 8                         // orders 0 .. 7
struct InvTable {
  double v[112];                         // 1 / n; v[0] infinite
};
constexpr InvTable inv_table()
{
  InvTable t{};
  t.v[0] = __builtin_inf();
  for (int n = 1; n < 112; n++) t.v[n] = 1.0 / n;
  return t;
}
static __constant__ const InvTable c_inv = inv_table();

// relative exponentials ExpRelV3P0 (TaylorDuffy.cc:840-893) of orders
// 0 .. nTop of Z, ez = exp(Z): n! / Z^n (e^Z - the first n terms of its
// series), or the series past those terms (to 1e-8) where |Z| < 0.1.  The
// first form for all orders from one exponential and one reciprocal
__device__ inline void exprels(int nTop, cplx Z, cplx ez, cplx *ER)
{
  const double z2 = norm2(Z);
  if (z2 >= 0.1 * 0.1) {
    const double d = 1.0 / z2;
    const cplx iz = mk(Z.r * d, -Z.i * d);
    cplx Sum = ez, Term = mk(1, 0), iT = mk(1, 0);
    ER[0] = Sum;
#pragma unroll
    for (int n = 1; n < TD_NER; n++) {
      if (n > nTop) break;
      Sum = Sum - Term;
      Term = cmulf(Term, (1.0 / n) * Z);
      iT = cmulf(iT, (double)n * iz);
      ER[n] = cmulf(Sum, iT);
    }
    return;
  }
  const bool real = Z.i == 0.0;
#pragma unroll
  for (int n = 0; n < TD_NER; n++) {
    if (n > nTop) break;
    cplx Term = mk(1, 0), Sum = mk(1, 0);
    for (int m = 1; m < 100; m++) {
      Term = cmulf(Term, c_inv.v[m + n] * Z);
      Sum += Term;
      if (real ? fabs(Term.r) < 1.0e-8 * fabs(Sum.r) : norm2(Term) < 1.0e-16 * norm2(Sum)) break;
    }
    ER[n] = Sum;
  }
}

}  // namespace scuffx
