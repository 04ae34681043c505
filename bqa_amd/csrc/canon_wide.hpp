// Canonicalisers for bond dimensions 17..32 (n = 2 chi = 34..64): host interface of canon_wide.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace bqa {

inline bool canon_wide_shape(int chi) { return chi >= 17 && chi <= 32; }

// Edges per round of launches, each with one workspace slot (the bases and root weights of both sides).
constexpr int kCanonWideEdges = 512;
inline size_t canon_wide_slot(int n) { return 2 * sizeof(cplx<double>) * n * n + 4 * sizeof(double) * n; }
inline size_t canon_wide_ws_bytes(int E, int chi) {
  const size_t edges = E < kCanonWideEdges ? E : kCanonWideEdges;
  return edges * canon_wide_slot(2 * chi);
}

void canon_wide(const cplx<double>* ext, int E, int chi, int ccols, double pinv_eps, double dtype_eps,
                cplx<double>* canon, double* lambdas, void* ws, hipStream_t s);

}  // namespace bqa
