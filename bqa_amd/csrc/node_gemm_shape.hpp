// Which shapes the matrix-product kernels (node_gemm.hpp) serve and how many nodes at a time.  Host code without HIP,
// so its rules are tested on the CPU.
#pragma once

#include <cstddef>

namespace bqa {

constexpr int kGemmMaxDegree = 6;
constexpr int kGemmMaxChi = 32;
constexpr size_t kGemmElement = 16;   // bytes of a complex double

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

// Node tensors of a few hundred elements are a block's work in LDS, where the products' launches and workspace cost more
// than they save once the generic kernel's blocks, one a node, fill the chip.  Microseconds, products and generic kernel:
//   BP sweep, FP64: degree 2, 600 nodes chi = 9 29 and 16, 11 30 and 20, 12 32 and 26, 13 35 and 29, 14 36 and 32, 15 37 and
//   36; 10,000 nodes chi = 9 223 and 108, 12 241 and 228, 13 256 and 258; degree 5, chi = 2 400 nodes 38 and 34, 3,000 116
//   and 83, chi = 3 400 nodes 52 and 44, 10,000 703 and 502; but 260 nodes 38 and 43, and chi = 4 144 and 306 for 600.
//   Simple update: degree 5, 3,000 nodes chi = 2 164 and 128, 3 321 and 288; 600 nodes 69 and 69, 110 and 112; degree 2,
//   3,000 nodes chi = 9 716 and 692, 12 1,287 and 1,292.
//   Readout call: degree 5, 20 nodes chi = 2 48 and 39, chi = 4 47 and 63; 1,200 nodes chi = 2 60 and 43, 3 74 and 53, 4 172
//   and 157; degree 4, chi = 5 600 nodes 73 and 84, 3,000 195 and 187; degree 3, 3,000 nodes chi = 9 182 and 242; degree 2,
//   3,000 nodes chi = 9 78 and 61, 12 83 and 86.
// FP32 sweeps and readouts stay with the products, whose Grams are summed in FP64 (readouts within 0.7 times the generic
// kernel's distance from 64 bits), though degree 2 with 600 nodes at chi = 9 takes 23 us a sweep for 15; extended messages
// are FP64 arithmetic in both.
enum GemmUse { kGemmBp, kGemmExt, kGemmDensity };
inline bool gemm_too_small(GemmUse use, int n, int d, int chi, size_t element) {
  if (element != kGemmElement) return false;
  long s = 2;
  for (int k = 0; k < d && s <= 4096; ++k) s *= chi;
  switch (use) {
    case kGemmBp:
      if (d == 2 && s > 288) return s <= 400 && n >= 384 && n * s <= 500000;
      return s <= 512 && n >= (d == 2 ? 256 : 384);
    case kGemmExt:
      return s <= (d == 2 ? 256 : 512) && n >= 1024;
    default:
      if (d <= 3) return d == 2 && s <= 256;
      return s <= 512 || (s <= 2048 && n >= (d == 4 ? 1024 : 512));
  }
}

// Classes whose workspace fits.  A single node's products may be many times its tensor (twelve at degree 6), where the generic kernel
// keeps three node tensors a block: beyond kGemmNodeMost (a seventieth of the card) they may take no more than that, so
// that a job of one or two large hubs that fits with the generic kernels fits with these.
constexpr size_t kGemmNodeMost = (size_t)4 << 30;
inline bool gemm_fits(int n, int d, int chi) {
  return gemm_shape(d, chi) &&
         (gemm_node_bytes(d, chi, kGemmElement) <= kGemmNodeMost || gemm_products(d) <= 3 * (n < 1024 ? n : 1024));
}
// ... for a use with products of `element` bytes an element.
inline bool gemm_serves(GemmUse use, int n, int d, int chi, size_t element) {
  return gemm_fits(n, d, chi) && !gemm_too_small(use, n, d, chi, element);
}

// The absorb serves node tensors of which k_node_local cannot keep two FP64 copies in 64 KB of LDS (with them, one
// block does a node in one launch).
inline bool gemm_local_shape(int d, int chi_in, int chi_out) {
  const int most = chi_in > chi_out ? chi_in : chi_out;
  if (!gemm_shape(d, most) || chi_in < 2 || chi_out < 1) return false;
  long s = 2;
  for (int k = 0; k < d; ++k) s *= most;
  return 2 * s * (long)kGemmElement > 64 * 1024;
}
// Nodes per round: two FP64 tensors each, within kGemmBudget and within what 1,024 blocks of the generic kernel take.
inline size_t gemm_local_node_bytes(int d, int chi) {
  size_t s = 4 * kGemmElement;
  for (int k = 0; k < d; ++k) s *= chi;
  return s;
}
inline int gemm_local_chunk(int n, int d, int chi) {
  size_t c = kGemmBudget / gemm_local_node_bytes(d, chi);
  if (c > 1024) c = 1024;
  if (c >= (size_t)n) return n;
  return c >= 8 ? (int)(c / 8 * 8) : c > 0 ? (int)c : 1;
}

}  // namespace bqa
