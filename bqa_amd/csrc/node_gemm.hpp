// Node contractions as batched matrix products for the shapes without a kernel of their own
// (chi up to 32, degrees 2..6): host interface of node_gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels_node.hpp"

namespace bqa {

constexpr int kGemmMaxDegree = 6;
constexpr int kGemmMaxChi = 32;
constexpr int kGemmMaxProducts = 16;

// The products of one degree: product q multiplies bond bond[q] of product src[q] (-1: the node
// tensor) by that bond's incoming message, level by level; output k is the Gram of the products
// bra[k] and ket[k] over every index but bond k.  The messages are Hermitian, so a message moves
// from the ket to the bra unchanged, and each output needs only two partial products: 3 products
// at degree 3, 6 at degree 4 and 9 at degree 5, instead of d (d - 1).
struct GemmPlan {
  int d, products, levels;
  int first[8];                              // products of level l: first[l] .. first[l + 1] - 1
  int8_t src[kGemmMaxProducts], bond[kGemmMaxProducts];
  int8_t bra[kGemmMaxDegree], ket[kGemmMaxDegree];
};

GemmPlan gemm_plan(int d);

// Shapes served: a node tensor's elements are counted in 32 bits, and without a product to make (degree 1) or
// to sum (chi = 1) the kernels of kernels_node.hpp take fewer launches (300 degree-1 nodes at chi = 12: 16 against
// 19 us a sweep; 1,000 degree-3 nodes at chi = 1: 66 against 79 us).
inline bool gemm_shape(int d, int chi) {
  if (d < 2 || chi < 2 || d > kGemmMaxDegree || chi > kGemmMaxChi) return false;
  long s = 2;
  for (int k = 0; k < d; ++k) s *= chi;
  return s < (1L << 30);
}

// Products a node of degree d keeps in the workspace.
inline int gemm_products(int d) { return d <= 3 ? d : d == 4 ? 6 : d == 5 ? 9 : 12; }

// Nodes per round of launches: their products take at most kGemmBudget bytes (half of the Infinity Cache,
// so the Grams read them from there), and one node at least.
constexpr size_t kGemmBudget = 128u << 20;
inline size_t gemm_node_bytes(int d, int chi, size_t csize) {
  size_t s = 2 * csize * gemm_products(d);
  for (int k = 0; k < d; ++k) s *= chi;
  return s;
}
inline int gemm_chunk(int n, int d, int chi, size_t csize) {
  const size_t node = gemm_node_bytes(d, chi, csize);
  if (node == 0) return n;
  const size_t c = kGemmBudget / node;
  if (c >= (size_t)n) return n;
  return c >= 8 ? (int)(c / 8 * 8) : c > 0 ? (int)c : 1;
}

// One BP sweep of a class (R: float or double): product launches level by level, then one launch of
// Grams, for `chunk` nodes at a time; ws holds chunk * gemm_products(d) tensors.
template <typename R>
void gemm_bp(ClassView cv, int chi, const cplx<R>* T, cplx<R>* mA, cplx<R>* mB, BpStatus* st, void* ws, int chunk,
             hipStream_t s);

// Extended messages in FP64 arithmetic from R storage; cv.zz holds the step's ZZ-split gates.
template <typename R>
void gemm_ext(ClassView cv, int chi, const cplx<R>* T, const cplx<R>* msgs, cplx<double>* ext, void* ws, int chunk,
              hipStream_t s);

// Density matrices and Bloch vectors (FP64 sums): half of the messages on the ket and half on the bra, d products
// level by level and one block of sums per node, in chunk * gemm_products(d) tensors of workspace.  The generic
// kernel, one block per node with VALU loops, took 6.0 ms for the 9,604 degree-4 nodes of a 100x100 grid at chi = 8
// (FP64), 3.5 ms for 100 degree-3 nodes at chi = 32 and 2.0 ms for 120 degree-5 nodes at chi = 8 (FP32).
template <typename R>
void gemm_density(ClassView cv, int chi, const cplx<R>* T, const cplx<R>* msgs, double* rho, double* bloch, void* ws,
                  int chunk, hipStream_t s);

// Absorb (every bond k: T <- sum_c T[.., c, ..] W_p[c][.], W_p = g0 C_k[c] + (-1)^p g1 C_k[chi_in + c]) in FP64,
// one launch per bond, then one launch with the gates and the symmetric gauge (the flags of k_node_local).  It
// serves node tensors of which k_node_local cannot keep two FP64 copies in 64 KB of LDS (with them, one block
// does a node in one launch).
inline bool gemm_local_shape(int d, int chi_in, int chi_out) {
  const int most = chi_in > chi_out ? chi_in : chi_out;
  if (!gemm_shape(d, most) || chi_in < 2 || chi_out < 1) return false;
  long s = 2;
  for (int k = 0; k < d; ++k) s *= most;
  return 2 * s * (long)sizeof(cplx<double>) > 64 * 1024;
}
// Nodes per round: two FP64 tensors each, within kGemmBudget and within what 1,024 blocks of the generic kernel take.
inline size_t gemm_local_node_bytes(int d, int chi) {
  size_t s = 4 * sizeof(cplx<double>);
  for (int k = 0; k < d; ++k) s *= chi;
  return s;
}
inline int gemm_local_chunk(int n, int d, int chi) {
  size_t c = kGemmBudget / gemm_local_node_bytes(d, chi);
  if (c > 1024) c = 1024;
  if (c >= (size_t)n) return n;
  return c >= 8 ? (int)(c / 8 * 8) : c > 0 ? (int)c : 1;
}
template <typename R>
void gemm_local(ClassView cv, int chi_in, int chi_out, const cplx<R>* Tin, cplx<R>* Tout, const cplx<double>* canon,
                int canon_cols, double zz_time, int flags, double z_time, double x_time, const double* lmbd,
                int lstride, cplx<R>* msgs_init, void* ws, int chunk, hipStream_t s);

}  // namespace bqa
