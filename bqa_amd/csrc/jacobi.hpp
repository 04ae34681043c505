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

// Columns with squared norms a, b and product g = (gr, gi): tangent t, cosine c, sine s, phase e = conj(g) / |g|
// and |g| t, so that (c p - s e q, s p + c e q) are orthogonal.  c, s and e are exact to rounding (the step stays
// unitary); the tangent comes from hardware estimates, accurate to 2^-21, which leaves that fraction of the pair's
// cosine for the next sweep to find below the test's threshold.  The scalar chain of a round is what its waves
// wait for: 35 instructions instead of 94 took the n = 16 canonicaliser of 150,000 edges from 6.5 to 5.1 ms.
struct JacobiStep {
  double t, c, s, er, ei, tg;
};
__device__ __forceinline__ JacobiStep jacobi_step(double a, double b, double gr, double gi, double g2) {
  JacobiStep r;
  const double rga = rsqrt_pos(g2);
  const double zeta = 0.5 * (b - a) * rga;
  const double h = fma(zeta, zeta, 1.0);
  const double w = fma(h, __builtin_amdgcn_rsq(h), fabs(zeta));
  r.t = copysign(__builtin_amdgcn_rcp(w), zeta);
  r.c = rsqrt_pos(fma(r.t, r.t, 1.0));
  r.s = r.c * r.t;
  r.er = gr * rga;
  r.ei = -gi * rga;
  r.tg = r.t * (g2 * rga);
  return r;
}

}  // namespace bqa
