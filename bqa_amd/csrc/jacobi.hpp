// The rotation of a one-sided Jacobi step, shared by the canonicalisers.
#pragma once

#include <hip/hip_runtime.h>

namespace bqa {

// 1 / sqrt(x) for normal x > 0: the hardware estimate (relative error below 2^-22) and one third-order step, whose
// error is its cube (below 2^-66).  Six instructions where the library's form handles every argument.
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// 1 / x for normal x > 0 in the same way.
__device__ __forceinline__ double rcp_pos(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

// Columns with squared norms a, b and product g = (gr, gi): tangent t, cosine c, sine s, phase e = conj(g) / |g|
// and |g| t, so that (c p - s e q, s p + c e q) are orthogonal, all to rounding: the canonicalisers skip the sweep that
// would find what a rougher tangent leaves of a pair's cosine, and with the hardware's 22 bits the bases were 5 to 20%
// further from 64-bit ones (n = 4 to 32) at the same time.  The scalar chain of a round is what its waves wait for: with
// the library's square roots and divisions it is 94 instructions and the n = 16 canonicaliser of 150,000 edges took
// 6.5 ms, with these under half of that and 5.1 ms.
struct JacobiStep {
  double t, c, s, er, ei, tg;
};
__device__ __forceinline__ JacobiStep jacobi_step(double a, double b, double gr, double gi, double g2) {
  JacobiStep r;
  const double rga = rsqrt_pos(g2);
  const double zeta = 0.5 * (b - a) * rga;
  const double h = fma(zeta, zeta, 1.0);
  r.t = copysign(rcp_pos(fma(h, rsqrt_pos(h), fabs(zeta))), zeta);
  r.c = rsqrt_pos(fma(r.t, r.t, 1.0));
  r.s = r.c * r.t;
  r.er = gr * rga;
  r.ei = -gi * rga;
  r.tg = r.t * (g2 * rga);
  return r;
}

}  // namespace bqa
