// Node contractions as batched matrix products for the shapes without a kernel of their own
// (chi up to 32, degrees 2..6): host interface of node_gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels_node.hpp"
#include "node_gemm_shape.hpp"

namespace bqa {

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
// one launch per bond, then one launch with the gates and the symmetric gauge (the flags of k_node_local).
template <typename R>
void gemm_local(ClassView cv, int chi_in, int chi_out, const cplx<R>* Tin, cplx<R>* Tout, const cplx<double>* canon,
                int canon_cols, double zz_time, int flags, double z_time, double x_time, const double* lmbd,
                int lstride, cplx<R>* msgs_init, void* ws, int chunk, hipStream_t s);

}  // namespace bqa
