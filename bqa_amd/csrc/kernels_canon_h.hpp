// Canonicalisers with split columns for bond dimensions chi <= 16 (n = 2 chi <= 32).
//
// Same results as k_canonicalize, organised for occupancy and
// fewer Jacobi sweeps:
//   * 2 * P2 lanes per edge (P2 = n/2 rounded up to a power of two): lane
//     (k, h) = k + P2 h holds rows [h n/2, (h+1) n/2) of the two columns of
//     pair k, so a column dot product is a lane-local sum plus one DPP
//     exchange with the other half (lane ^ P2);
//   * the Jacobi sweep pairs columns in a recursive xor order (all top x bot
//     pairs with only the bot columns moving by one lane-xor per round, then
//     each half split in two by one re-layout, and so on: 2 P2 - 1 rounds), so
//     a round moves one column per lane, through the LDS crossbar
//     (ds_bpermute) rather than VALU moves and selects.  It wants a power of
//     two of column pairs; padding with zero columns, which never rotate, makes
//     one, and each column then carries its number.  Where that is a third more
//     rounds than the n - 1 of a round-robin (n = 6, 10, 12, 18..24), columns go
//     round by DPP row shifts instead;
//   * the Hermitian PSD extended messages are factored M = L L^H by pivoted
//     Cholesky first; one-sided Jacobi on the columns of L then converges in
//     about half the sweeps of Jacobi on M and yields V_M Sigma_L directly,
//     with sigma_L^2 the eigenvalues (= singular values) of M;
//   * the bond matrix K runs Jacobi without accumulating V: with K = S_f X S_b,
//     X = conj(U_f^T U_b), the right singular vectors are
//     Vs = S_b U_b^T U_f S_f Us / Lambda for the kept columns.
#pragma once

#include "common.hpp"
#include "jacobi.hpp"

namespace bqa {

// Column pairs of n = 2 chi, padded to a power of two.
__host__ __device__ constexpr int canon_pairs(int n) {
  const int p = n / 2;
  return p <= 1 ? 1 : p <= 2 ? 2 : p <= 4 ? 4 : p <= 8 ? 8 : 16;
}
// The order of the Jacobi's rounds: xor (2 P2 - 1 rounds, P2 padded pairs) where that is at most 4/3 of a round-robin's
// n - 1.  Milliseconds for 8,192 (n <= 14: 16,384) edges, xor and round-robin: n = 10 0.58 and 0.48, 12 0.75 and
// 0.69, 14 0.94 and 1.02, 18 2.04 and 1.58, 20 2.34 and 1.94, 22 2.63 and 2.35, 24 3.01 and 2.95, 26 3.22 and 3.39, 28
// 3.63 and 4.08, 30 4.11 and 4.60.
__host__ __device__ constexpr bool canon_xor(int n) {
  return 3 * (2 * canon_pairs(n) - 1) <= 4 * (n - 1) || canon_pairs(n) == n / 2;
}
// Waves of all edges up to which the split form is taken.  With one a SIMD (1,024) it takes 0.7 to 0.8 of the time of
// one side after the other at every n.  With two, split over the other form's single wave at 1,100, 1,536 and 2,048: n = 2
// 0.91, 0.93, 0.92, 4 0.91, 0.92, 0.91, 8 0.93, 0.91, 0.93, 14 0.98, 1.01, 1.00 and 16 1.00, 1.06, 1.01 (kept, so that a
// batch's jobs fall into one launch), but 6 1.04, 1.06, 1.06, 10 1.10, 1.13, 1.11, 12 1.06, 1.11, 1.12, 18 1.11, 1.11,
// 1.09, 24 1.12, 1.10, 1.05, 26 1.03, 1.06, 1.05 and 32 1.03, 0.99, 1.02.
__host__ __device__ constexpr int canon_split_waves(int n) { return canon_xor(n) && n <= 16 ? 2048 : 1024; }

template <int N>
struct HCanon {
  static constexpr int P = N / 2;                                   // column pairs
  static constexpr int P2 = canon_pairs(N);
  static constexpr int G = 2 * P2;                                  // lanes per edge
  static constexpr int EPW = 64 / G;                                // edges per wave
  static constexpr int NH = N / 2;                                  // rows per lane
  static constexpr bool kXor = canon_xor(N);                        // order of the Jacobi's rounds
  // Split form (both sides of an edge at once): lanes and edges per wave, and the edges up to which it is taken.
  // A wave's serial chain of two factorisations and three Jacobi runs is then two thirds as long, but half of its
  // lanes idle in the third, and there are twice the waves.
  static constexpr int GS = 2 * G;
  static constexpr int EPWS = 64 / GS;
  static constexpr int kSplitEdges = canon_split_waves(N) * EPWS;
  // workspace doubles per edge: U_f, U_b, Q (N x N complex each), sorted Us and Z columns
  // (N x N complex each), sq/ip of both sides, 1/Lambda of the sorted columns
  static constexpr int WS = 10 * N * N + 5 * N;
};

template <int NH>
struct HCol {
  double re[NH], im[NH];
};

// 32-bit DPP move within 16-lane rows (every source lane valid for the
// patterns used here).
template <int CTRL>
__device__ __forceinline__ int dpp32(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}

// Value of lane ^ M (M = 1, 2, 4, 8) within 16-lane rows: quad permutations
// for 1 and 2, half-row mirror (lane ^ 7) then lane ^ 3 for 4, rotation by 8.
template <int M>
__device__ __forceinline__ int xor_lane32(int v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "lane xor within a row");
  if constexpr (M == 1) return dpp32<0xB1>(v);
  else if constexpr (M == 2) return dpp32<0x4E>(v);
  else if constexpr (M == 4) return dpp32<0x1B>(dpp32<0x141>(v));
  else return dpp32<0x128>(v);
}

template <int M>
__device__ __forceinline__ double xor_lane(double x) {
  const int lo = xor_lane32<M>(__double2loint(x)), hi = xor_lane32<M>(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

// Sum over both halves of a column.  Every lane of the edge's group must be switched on, padding lanes (k >= n / 2)
// included: at n = 6 the exchange is two chained moves that pass through padding lanes for pair 0.  With the sums for
// the Jacobi's scale under a branch on `active`, chi = 3 quenches had Bloch vectors off by up to 0.1 (FP64); with
// the same sums outside it, by 1e-13.
template <int N>
__device__ __forceinline__ double half_sum(double v) {
  if constexpr (HCanon<N>::P2 == 16)
    return v + __shfl_xor(v, 16, 64);     // the partner half is in the other 16-lane row
  else
    return v + xor_lane<HCanon<N>::P2>(v);
}

// Value of the next and of the previous lane of the row.
__device__ __forceinline__ double dpp_from_next(double x) {  // row_shl:1
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x101, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x101, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double dpp_from_prev(double x) {  // row_shr:1
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x111, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x111, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// One step of the round-robin; after N - 1 of them every column is back in its place.  Padding lanes take copies.
template <int N>
__device__ __forceinline__ void hrotate_owners(HCol<N / 2>& top, HCol<N / 2>& bot, int k) {
  constexpr int P = N / 2, NH = N / 2;
#pragma unroll
  for (int r = 0; r < NH; ++r) {
    const double xr = dpp_from_next(top.re[r]), xi = dpp_from_next(top.im[r]);
    const double yr = dpp_from_prev(bot.re[r]), yi = dpp_from_prev(bot.im[r]);
    const double tr = k == 0 ? top.re[r] : (k < P - 1 ? xr : bot.re[r]);
    const double ti = k == 0 ? top.im[r] : (k < P - 1 ? xi : bot.im[r]);
    bot.re[r] = k == 0 ? xr : yr;
    bot.im[r] = k == 0 ? xi : yi;
    top.re[r] = tr;
    top.im[r] = ti;
  }
}

template <int NH>
__device__ __forceinline__ double hnorm2(const HCol<NH>& c) {
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < NH; ++r) s = fma(c.re[r], c.re[r], fma(c.im[r], c.im[r], s));
  return s;
}

// One Jacobi round: rotate the pair of split columns held by this lane pair
// (top, bot) so that they become orthogonal; `rotated` / `unsettled` collect
// whether the round rotated at all and whether a rotation was still large.
// The xor order carries the squared column norms a, b (exact at each sweep's
// start, updated by the rotation's a - t|g|, b + t|g|, moved with their columns).
template <int N>
__device__ __forceinline__ void hjacobi_round(HCol<N / 2>& top, HCol<N / 2>& bot, double& a, double& b,
                                              double small2, double tol, int& rotated, int& unsettled) {
  constexpr int NH = N / 2;
  // A sweep whose rotations all had column cosine |g| / sqrt(a b) < 1e-8 and
  // sine |s| < 1e-6 leaves every cosine below ~1e-14 (each later rotation of
  // the sweep changes a settled pair by at most the product of the two), so
  // the sweep that would only confirm convergence is skipped; near-degenerate
  // pairs, where tiny cosines give large rotations, keep the full test.
  constexpr double kSettledCos2 = 1e-16, kSettledSin2 = 1e-12;
  double gr = 0.0, gi = 0.0, hr = 0.0, hi = 0.0;   // two chains each
#pragma unroll
  for (int r = 0; r < NH; ++r) {
    gr = fma(top.re[r], bot.re[r], gr);
    hr = fma(top.im[r], bot.im[r], hr);
    gi = fma(top.re[r], bot.im[r], gi);
    hi = fma(-top.im[r], bot.re[r], hi);
  }
  gr = half_sum<N>(gr + hr);
  gi = half_sum<N>(gi + hi);
  const double g2 = gr * gr + gi * gi;
  const double ab = a * b;
  if (fmin(a, b) >= small2 && g2 > tol * tol * ab) {
    rotated = 1;
    const JacobiStep j = jacobi_step(a, b, gr, gi, g2);
    unsettled |= (g2 > kSettledCos2 * ab || j.s * j.s > kSettledSin2) ? 1 : 0;
    a -= j.tg;
    b += j.tg;
#pragma unroll
    for (int r = 0; r < NH; ++r) {
      const double xr = j.er * bot.re[r] - j.ei * bot.im[r];
      const double xi = j.er * bot.im[r] + j.ei * bot.re[r];
      const double pr = top.re[r], pi = top.im[r];
      bot.re[r] = j.s * pr + j.c * xr;
      bot.im[r] = j.s * pi + j.c * xi;
      top.re[r] = j.c * pr - j.s * xr;
      top.im[r] = j.c * pi - j.s * xi;
    }
  }
}

// Value of lane `src` (a wave lane, passed as 4 * src) through the LDS
// crossbar: no VALU work beyond the address, for the column moves.
__device__ __forceinline__ double bperm(double x, int addr4) {
  const int lo = __builtin_amdgcn_ds_bpermute(addr4, __double2loint(x));
  const int hi = __builtin_amdgcn_ds_bpermute(addr4, __double2hiint(x));
  return __hiloint2double(hi, lo);
}

// One-sided Jacobi on the columns held by the lane pairs of an edge.  it, ib: the columns'
// numbers (-1: padding), which move with them in the padded xor order.
template <int N>
__device__ void hjacobi(HCol<N / 2>& top, HCol<N / 2>& bot, int& it, int& ib, int k) {
  constexpr int NH = N / 2, P = N / 2, P2 = HCanon<N>::P2;
  constexpr bool kIds = HCanon<N>::kXor && P != P2;
  double sc = fmax(half_sum<N>(hnorm2(top)), half_sum<N>(hnorm2(bot)));
#pragma unroll
  for (int o = 1; o < P2; o <<= 1) sc = fmax(sc, __shfl_xor(sc, o, 64));
  const double small2 = 1e-26 * sc;
  const double tol = 2.2204460492503131e-16 * N;
  const int lane = threadIdx.x & 63;
  for (int sweep = 0; sweep < 30; ++sweep) {
    int rotated = 0, unsettled = 0;
    if constexpr (!HCanon<N>::kXor) {
#pragma unroll 1
      for (int round = 0; round < N - 1; ++round) {
        double a = half_sum<N>(hnorm2(top)), b = half_sum<N>(hnorm2(bot));
        a = k < P ? a : 0.0;   // padding lanes hold copies and do not rotate
        hjacobi_round<N>(top, bot, a, b, small2, tol, rotated, unsettled);
        hrotate_owners<N>(top, bot, k);
      }
      if (!__any(rotated) || !__any(unsettled)) break;
      continue;
    }
    // recursive xor order: in the phase of group size L the tops and the
    // bots of each group of L lanes meet all pairs (bot at lane k holds the
    // bot that started at lane k ^ gray(t) in round t, so round t moves it by
    // the lowest set bit of t); the re-layout at bit L / 2 then leaves the
    // pairs within each half for size L / 2: lanes with the bit clear take
    // (own top, partner's top), lanes with it set (own bot, partner's bot)
    double a = half_sum<N>(hnorm2(top)), b = half_sum<N>(hnorm2(bot));
#pragma unroll 1
    for (int L = P2; L >= 1; L >>= 1) {
#pragma unroll 1
      for (int t = 0; t < L; ++t) {
        if (t > 0) {
          const int addr = 4 * (lane ^ (t & -t));
#pragma unroll
          for (int r = 0; r < NH; ++r) {
            bot.re[r] = bperm(bot.re[r], addr);
            bot.im[r] = bperm(bot.im[r], addr);
          }
          b = bperm(b, addr);
          if constexpr (kIds) ib = __builtin_amdgcn_ds_bpermute(addr, ib);
        }
        hjacobi_round<N>(top, bot, a, b, small2, tol, rotated, unsettled);
      }
      if (L > 1) {
        const int m = L >> 1, addr = 4 * (lane ^ m);
        const bool hi = (k & m) != 0;
#pragma unroll
        for (int r = 0; r < NH; ++r) {
          const double fr = bperm(hi ? top.re[r] : bot.re[r], addr);
          const double fi = bperm(hi ? top.im[r] : bot.im[r], addr);
          top.re[r] = hi ? bot.re[r] : top.re[r];
          top.im[r] = hi ? bot.im[r] : top.im[r];
          bot.re[r] = fr;
          bot.im[r] = fi;
        }
        const double fn = bperm(hi ? a : b, addr);
        a = hi ? b : a;
        b = fn;
        if constexpr (kIds) {
          const int fid = __builtin_amdgcn_ds_bpermute(addr, hi ? it : ib);
          it = hi ? ib : it;
          ib = fid;
        }
      }
    }
    if (!__any(rotated) || !__any(unsettled)) break;
  }
}

// Orders this wave's LDS accesses around a cross-lane exchange (the block is
// one wave, whose LDS operations complete in issue order).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One butterfly step of the pivot search: the larger diagonal of this lane and lane ^ M, ties to
// the lower column (-1: none).
template <int M>
__device__ __forceinline__ void pivot_step(double& bv, int& bc) {
  const double ov = xor_lane<M>(bv);
  const int oc = xor_lane32<M>(bc);
  if (ov > bv || (ov == bv && oc >= 0 && (bc < 0 || oc < bc))) {
    bv = ov;
    bc = oc;
  }
}

// Pivoted Cholesky M = L L^H in place: each column ends up holding one column of
// L (in pivot order) or zero beyond the numerical rank.  The scaled pivot
// column goes through the edge's LDS slot `lcol` (N complex).  dgt / dgb are the
// residual diagonals of the lane's columns ct = k and cb = N - 1 - k, updated
// with the arithmetic the column update applies to its diagonal element.
template <int N>
__device__ void hcholesky(HCol<N / 2>& top, HCol<N / 2>& bot, int k, int h, bool active, double dgt, double dgb,
                          double2* lcol) {
  constexpr int NH = N / 2, P2 = HCanon<N>::P2;
  const int ct = k, cb = N - 1 - k, r0 = h * NH;
  bool dt = !active, db = !active;  // done flags
  double d0 = 0.0;
  for (int step = 0; step < N; ++step) {
    // best undone diagonal over the group: value and the matrix column holding it
    double bv = -1.0;
    int bc = -1;
    if (!dt && dgt > bv) { bv = dgt; bc = ct; }
    if (!db && dgb > bv) { bv = dgb; bc = cb; }
    // butterfly over the column pairs by DPP lane xors (a step's latency is a few cycles, where a
    // shuffle through the LDS crossbar waits for its round trip); the same order as a shuffle loop
    if constexpr (P2 > 1) pivot_step<1>(bv, bc);
    if constexpr (P2 > 2) pivot_step<2>(bv, bc);
    if constexpr (P2 > 4) pivot_step<4>(bv, bc);
    if constexpr (P2 > 8) pivot_step<8>(bv, bc);
    if (step == 0) d0 = bv;
    if (!(bv > 1e-20 * d0) || bc < 0) {  // numerical rank reached: zero the rest
      if (!dt) {
#pragma unroll
        for (int r = 0; r < NH; ++r) { top.re[r] = 0.0; top.im[r] = 0.0; }
      }
      if (!db) {
#pragma unroll
        for (int r = 0; r < NH; ++r) { bot.re[r] = 0.0; bot.im[r] = 0.0; }
      }
      break;
    }
    // pivot column, scaled: l = R[:, bc] / sqrt(R[bc][bc]), written by the lane
    // pair holding column bc
    const int owner_k = bc < N / 2 ? bc : N - 1 - bc;
    const bool own_top = bc == owner_k;
    const double inv = rsqrt_pos(bv);
    if (k == owner_k) {
#pragma unroll
      for (int r = 0; r < NH; ++r)
        lcol[r0 + r] = make_double2((own_top ? top.re[r] : bot.re[r]) * inv, (own_top ? top.im[r] : bot.im[r]) * inv);
    }
    wave_lds_sync();
    HCol<NH> l;
#pragma unroll
    for (int r = 0; r < NH; ++r) {
      const double2 v = lcol[r0 + r];
      l.re[r] = v.x;
      l.im[r] = v.y;
    }
    // conj(l[j]) for this lane's two columns j
    const double2 lt = lcol[ct], lb = lcol[cb];
    wave_lds_sync();
    // one in-place form for every column: R[:, j] <- R[:, j] - l conj(x), with x = l[j] to update,
    // sqrt(R[bc][bc]) - 1 for the pivot column (sqrt(R[bc][bc]) l, which so becomes l) and 0 once done
    const bool pt = active && bc == ct, pb = active && bc == cb;
    const double less1 = fma(bv, inv, -1.0);
    const double ut = dt ? 0.0 : 1.0, ub = db ? 0.0 : 1.0;
    const double ltr = pt ? less1 : ut * lt.x, lti = pt ? 0.0 : ut * lt.y;
    const double lbr = pb ? less1 : ub * lb.x, lbi = pb ? 0.0 : ub * lb.y;
#pragma unroll
    for (int r = 0; r < NH; ++r) {
      top.re[r] = fma(-l.re[r], ltr, fma(-l.im[r], lti, top.re[r]));
      top.im[r] = fma(-l.im[r], ltr, fma(l.re[r], lti, top.im[r]));
      bot.re[r] = fma(-l.re[r], lbr, fma(-l.im[r], lbi, bot.re[r]));
      bot.im[r] = fma(-l.im[r], lbr, fma(l.re[r], lbi, bot.im[r]));
    }
    // the diagonal element's update (l[j] conj(l[j]) in the form above)
    dgt = fma(-ltr, ltr, fma(-lti, lti, dgt));
    dgb = fma(-lbr, lbr, fma(-lbi, lbi, dgb));
    dt = dt || pt;
    db = db || pb;
  }
}

// The edges of block `blk` of one job's launch: blk * EPW .. blk * EPW + EPW - 1.  SPLIT: the edge's two extended
// messages are factored by two lane groups at once, and the first group goes on with the bond matrix.
template <int N, bool SPLIT>
__device__ __forceinline__ void canon_h_run(const cplx<double>* __restrict__ ext, int E, int ccols, double pinv_eps,
                                            double deps, zd* __restrict__ canon, double* __restrict__ lfull,
                                            double* __restrict__ ws, int blk) {
  using S = HCanon<N>;
  constexpr int P = S::P, P2 = S::P2, G = S::G, NH = S::NH;
  constexpr int GL = SPLIT ? S::GS : G;        // lanes per edge
  const int lane = threadIdx.x;
  const int w = lane % GL;
  const int base = lane - lane % G;
  const int h = lane % G / P2, k = lane % P2;
  const int edge = blk * (64 / GL) + lane / GL;
  const bool valid = edge < E;
  const bool active = valid && k < P;
  const bool lead = w < G;                     // the lane group of the bond matrix
  double* wsE = ws + (size_t)(valid ? edge : 0) * S::WS;
  double* Uf = wsE;
  double* Ub = wsE + 2 * N * N;
  double* sqf = wsE + 4 * N * N;
  double* ipf = sqf + N;
  double* sqb = ipf + N;
  double* ipb = sqb + N;
  const int r0 = h * NH;

  // pivot columns, one slot an edge; the slots' stride puts the edges' and halves' rows on different banks
  constexpr int kSlot = N + 2;
  __shared__ double2 lslots[S::EPW * kSlot];   // one per lane group
  double2* lcol = lslots + (lane / G) * kSlot;
  HCol<NH> top, bot;
  for (int pass = 0; pass < (SPLIT ? 1 : 2); ++pass) {
    const int side = SPLIT ? w / G : pass;
    const int ct = k, cb = N - 1 - k;
    double dgt = 0.0, dgb = 0.0;
#pragma unroll
    for (int r = 0; r < NH; ++r) {
      top.re[r] = top.im[r] = bot.re[r] = bot.im[r] = 0.0;
    }
    if (active) {
      // Hermitian part (M + M^H) / 2: the extended message is Hermitian by
      // construction, and its anti-Hermitian rounding part (from FP32 messages)
      // is dropped rather than folded into the factorisation.
      // (columns and rows from four base pointers with constant offsets, one
      // column at a time, so few loads and no per-row addresses stay live)
      const cplx<double>* M = ext + (size_t)(side ? E + edge : edge) * N * N;
      const cplx<double>* Mt = M + r0 * N + ct;  // column ct from row r0
      const cplx<double>* Rt = M + ct * N + r0;  // row ct from column r0
      const cplx<double>* Mb = M + r0 * N + cb;
      const cplx<double>* Rb = M + cb * N + r0;
#pragma unroll
      for (int r = 0; r < NH; ++r) {
        const cplx<double> x = Mt[r * N], xt = Rt[r];
        top.re[r] = 0.5 * (x.x + xt.x);
        top.im[r] = 0.5 * (x.y - xt.y);
      }
      dgt = M[ct * N + ct].x;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < NH; ++r) {
        const cplx<double> y = Mb[r * N], yt = Rb[r];
        bot.re[r] = 0.5 * (y.x + yt.x);
        bot.im[r] = 0.5 * (y.y - yt.y);
      }
      dgb = M[cb * N + cb].x;
    }
    hcholesky<N>(top, bot, k, h, active, dgt, dgb, lcol);
    int it = k < P ? 2 * k : -1, ib = k < P ? 2 * k + 1 : -1;
    hjacobi<N>(top, bot, it, ib, k);
    // columns are V_M sigma: eigenvalue s = sigma^2, U = column / sigma
    double* U = side ? Ub : Uf;
    double* sq = side ? sqb : sqf;
    double* ip = side ? ipb : ipf;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const HCol<NH>& c = hh ? bot : top;
      const double sig = sqrt(half_sum<N>(hnorm2(c)));
      const int slot = hh ? ib : it;
      if (valid && slot >= 0) {
        const double s = sig * sig;
        const bool keep = s > pinv_eps;
        const double sqv = keep ? sig : 0.0;
        if (h == 0) {
          sq[slot] = sqv;
          ip[slot] = sqv > deps ? 1.0 / sqv : 0.0;
        }
        const double inv = sig > 0.0 ? 1.0 / sig : 0.0;
        double* uc = U + slot * 2 * N + 2 * r0;
#pragma unroll
        for (int r = 0; r < NH; ++r) {
          uc[2 * r] = c.re[r] * inv;
          uc[2 * r + 1] = c.im[r] * inv;
        }
      }
    }
  }
  __syncthreads();

  // K[i][j] = sq_f[i] sq_b[j] conj(sum_t U_f[t, i] U_b[t, j]); this lane: columns 2k, 2k+1, rows of half h
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    HCol<NH>& kc = hh ? bot : top;
    const int j = 2 * k + hh;
#pragma unroll
    for (int r = 0; r < NH; ++r) {
      kc.re[r] = 0.0;
      kc.im[r] = 0.0;
    }
    if (active && lead) {
      // t outermost with the NH row accumulators inside: each sum keeps its
      // order while the workspace loads stream through a small register window
      const double* ub = Ub + j * 2 * N;
      double ar[NH], ai[NH];
#pragma unroll
      for (int r = 0; r < NH; ++r) ar[r] = ai[r] = 0.0;
#pragma unroll 2
      for (int t = 0; t < N; ++t) {
        const double br = ub[2 * t], bi = ub[2 * t + 1];
#pragma unroll
        for (int r = 0; r < NH; ++r) {
          const double fr = Uf[(r0 + r) * 2 * N + 2 * t], fi = Uf[(r0 + r) * 2 * N + 2 * t + 1];
          ar[r] = fma(fr, br, fma(-fi, bi, ar[r]));
          ai[r] = fma(fr, bi, fma(fi, br, ai[r]));
        }
      }
      const double sj = sqb[j];
#pragma unroll
      for (int r = 0; r < NH; ++r) {
        const double wgt = sqf[r0 + r] * sj;
        kc.re[r] = wgt * ar[r];
        kc.im[r] = -wgt * ai[r];
      }
    }
  }
  int it = lead && k < P ? 2 * k : -1, ib = lead && k < P ? 2 * k + 1 : -1;
  hjacobi<N>(top, bot, it, ib, k);
  const bool realt = valid && it >= 0, realb = valid && ib >= 0;

  // singular values, descending ranks (padding below every column), masks, normalised lambdas
  const double nt = sqrt(half_sum<N>(hnorm2(top))), nb = sqrt(half_sum<N>(hnorm2(bot)));
  const double lt = it >= 0 ? nt : -1.0, lb = ib >= 0 ? nb : -1.0;
  int rt = 0, rb = 0;
#pragma unroll 1
  for (int q = 0; q < P2; ++q) {
    const double ot = __shfl(lt, base + q, 64), ob = __shfl(lb, base + q, 64);
    const int st = 2 * q, sb = 2 * q + 1;
    rt += (ot > lt || (ot == lt && st < 2 * k)) ? 1 : 0;
    rt += (ob > lt || (ob == lt && sb < 2 * k)) ? 1 : 0;
    rb += (ot > lb || (ot == lb && st < 2 * k + 1)) ? 1 : 0;
    rb += (ob > lb || (ob == lb && sb < 2 * k + 1)) ? 1 : 0;
  }
  const bool keept = lt > pinv_eps, keepb = lb > pinv_eps;
  const double mt = keept ? lt : 0.0, mb = keepb ? lb : 0.0;
  double nn = h == 0 ? mt * mt + mb * mb : 0.0;
#pragma unroll
  for (int o = 1; o < G; o <<= 1) nn += __shfl_xor(nn, o, 64);
  const double nrm = sqrt(nn);
  if (realt && h == 0) lfull[(size_t)edge * N + rt] = mt / nrm;
  if (realb && h == 0) lfull[(size_t)edge * N + rb] = mb / nrm;
  // Stage the sorted, masked Us columns (Us[:, c] = K column / Lambda) and 1/Lambda.
  double* Q = wsE + 4 * N * N + 4 * N;         // Q[t][i] = sum_u U_b[u][t] U_f[u][i] sq_f[i]
  double* Us = Q + 2 * N * N;                  // Us[c][row], c = rank
  double* Zc = Us + 2 * N * N;                 // Z[c][j] = keep_b[j] conj(sum_i Q[j][i] Us[c][i]) / Lambda_c
  double* il = Zc + 2 * N * N;                 // 1 / Lambda_c (0 when masked)
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    if (hh ? realb : realt) {
      const HCol<NH>& c = hh ? bot : top;
      const int rank = hh ? rb : rt;
      const double inv = (hh ? keepb : keept) ? 1.0 / (hh ? lb : lt) : 0.0;
      if (h == 0) il[rank] = inv;
      double* uc = Us + rank * 2 * N + 2 * r0;
#pragma unroll
      for (int r = 0; r < NH; ++r) {
        uc[2 * r] = c.re[r] * inv;
        uc[2 * r + 1] = c.im[r] * inv;
      }
    }
  }
  if constexpr (N == 16) {
    if (ccols <= 8) {
      // chi = 8: the same products regrouped without the 16 x 16 Q,
      //   V = U_f diag(sq_f) Us and C_f = U_f diag(ip_f) Us in one pass,
      //   Z[c][j] = keep_b[j] conj((U_b^T V)[j][c]) / Lambda_c,  C_b = U_b Z,
      // each lane taking a block of 4 (SPLIT: 2) rows x 2 columns so every row and column
      // it loads serves several outputs (about a quarter of the workspace
      // reads of the entry-per-lane form below).
      __syncthreads();
      constexpr int RB = 64 / GL;
      const int a0 = RB * (w >> 2), c0 = 2 * (w & 3);
      double* V = Q;  // V[c][a], 16 x ccols
      double xr[RB][2] = {}, xi[RB][2] = {}, yr[RB][2] = {}, yi[RB][2] = {};
      if (valid) {
#pragma unroll 2
        for (int t = 0; t < N; ++t) {
          double sr[2], si[2], pr[2], pi[2];
#pragma unroll
          for (int cc = 0; cc < 2; ++cc) {
            const int c = c0 + cc;
            const double ur = c < ccols ? Us[c * 2 * N + 2 * t] : 0.0, ui = c < ccols ? Us[c * 2 * N + 2 * t + 1] : 0.0;
            sr[cc] = sqf[t] * ur;
            si[cc] = sqf[t] * ui;
            pr[cc] = ipf[t] * ur;
            pi[cc] = ipf[t] * ui;
          }
#pragma unroll
          for (int r = 0; r < RB; ++r) {
            const double fr = Uf[t * 2 * N + 2 * (a0 + r)], fi = Uf[t * 2 * N + 2 * (a0 + r) + 1];
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
              xr[r][cc] = fma(fr, sr[cc], fma(-fi, si[cc], xr[r][cc]));
              xi[r][cc] = fma(fr, si[cc], fma(fi, sr[cc], xi[r][cc]));
              yr[r][cc] = fma(fr, pr[cc], fma(-fi, pi[cc], yr[r][cc]));
              yi[r][cc] = fma(fr, pi[cc], fma(fi, pr[cc], yi[r][cc]));
            }
          }
        }
        zd* Cf = canon + (size_t)(E + edge) * N * ccols;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          const int c = c0 + cc;
          if (c < ccols) {
#pragma unroll
            for (int r = 0; r < RB; ++r) {
              V[c * 2 * N + 2 * (a0 + r)] = xr[r][cc];
              V[c * 2 * N + 2 * (a0 + r) + 1] = xi[r][cc];
              Cf[(a0 + r) * ccols + c] = mk(yr[r][cc], yi[r][cc]);
            }
          }
        }
      }
      __syncthreads();
      // Z rows j = a0..a0+3, columns c0, c0+1
      double wr[RB][2] = {}, wi[RB][2] = {};
      if (valid) {
#pragma unroll 2
        for (int u = 0; u < N; ++u) {
          double vr[2], vi[2];
#pragma unroll
          for (int cc = 0; cc < 2; ++cc) {
            const int c = c0 + cc;
            vr[cc] = c < ccols ? V[c * 2 * N + 2 * u] : 0.0;
            vi[cc] = c < ccols ? V[c * 2 * N + 2 * u + 1] : 0.0;
          }
#pragma unroll
          for (int r = 0; r < RB; ++r) {
            const double br = Ub[(a0 + r) * 2 * N + 2 * u], bi = Ub[(a0 + r) * 2 * N + 2 * u + 1];
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
              wr[r][cc] = fma(br, vr[cc], fma(-bi, vi[cc], wr[r][cc]));
              wi[r][cc] = fma(br, vi[cc], fma(bi, vr[cc], wi[r][cc]));
            }
          }
        }
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          const int c = c0 + cc;
          if (c < ccols) {
#pragma unroll
            for (int r = 0; r < RB; ++r) {
              const int j = a0 + r;
              const double g = ipb[j] > 0.0 ? il[c] : 0.0;
              Zc[(c * N + j) * 2] = wr[r][cc] * g;
              Zc[(c * N + j) * 2 + 1] = -wi[r][cc] * g;
            }
          }
        }
      }
      __syncthreads();
      // C_b rows a0..a0+3, columns c0, c0+1
      if (valid) {
        double br_[RB][2] = {}, bi_[RB][2] = {};
#pragma unroll 2
        for (int t = 0; t < N; ++t) {
          double zr[2], zi[2];
#pragma unroll
          for (int cc = 0; cc < 2; ++cc) {
            const int c = c0 + cc;
            zr[cc] = c < ccols ? Zc[(c * N + t) * 2] : 0.0;
            zi[cc] = c < ccols ? Zc[(c * N + t) * 2 + 1] : 0.0;
          }
#pragma unroll
          for (int r = 0; r < RB; ++r) {
            const double vr = Ub[t * 2 * N + 2 * (a0 + r)], vi = Ub[t * 2 * N + 2 * (a0 + r) + 1];
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
              br_[r][cc] = fma(vr, zr[cc], fma(-vi, zi[cc], br_[r][cc]));
              bi_[r][cc] = fma(vr, zi[cc], fma(vi, zr[cc], bi_[r][cc]));
            }
          }
        }
        zd* Cb = canon + (size_t)edge * N * ccols;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          const int c = c0 + cc;
          if (c < ccols) {
#pragma unroll
            for (int r = 0; r < RB; ++r) Cb[(a0 + r) * ccols + c] = mk(br_[r][cc], bi_[r][cc]);
          }
        }
      }
      return;
    }
  }
  // Q, one entry per lane per step over the group
  if (valid) {
    for (int x = w; x < N * N; x += GL) {
      const int t = x / N, i = x % N;
      double ar = 0.0, ai = 0.0;
      for (int u = 0; u < N; ++u) {
        const double br = Ub[t * 2 * N + 2 * u], bi = Ub[t * 2 * N + 2 * u + 1];
        const double fr = Uf[i * 2 * N + 2 * u], fi = Uf[i * 2 * N + 2 * u + 1];
        ar = fma(br, fr, fma(-bi, fi, ar));
        ai = fma(br, fi, fma(bi, fr, ai));
      }
      Q[2 * x] = ar * sqf[i];
      Q[2 * x + 1] = ai * sqf[i];
    }
  }
  __syncthreads();
  if (valid) {
    for (int x = w; x < ccols * N; x += GL) {
      const int c = x / N, jj = x % N;
      double ar = 0.0, ai = 0.0;
      if (ipb[jj] > 0.0) {
        for (int i = 0; i < N; ++i) {
          const double qr = Q[(jj * N + i) * 2], qi = Q[(jj * N + i) * 2 + 1];
          const double ur = Us[c * 2 * N + 2 * i], ui = Us[c * 2 * N + 2 * i + 1];
          ar = fma(qr, ur, fma(-qi, ui, ar));
          ai = fma(qr, ui, fma(qi, ur, ai));
        }
      }
      Zc[2 * x] = ar * il[c];
      Zc[2 * x + 1] = -ai * il[c];
    }
  }
  __syncthreads();
  // C_f[a][c] = sum_t U_f[a][t] ip_f[t] Us[c][t];  C_b[a][c] = sum_j U_b[a][j] Z[c][j]
  if (valid) {
    zd* Cb = canon + (size_t)edge * N * ccols;
    zd* Cf = canon + (size_t)(E + edge) * N * ccols;
    for (int x = w; x < N * ccols; x += GL) {
      const int a = x / ccols, c = x % ccols;
      double fr_ = 0.0, fi_ = 0.0, br_ = 0.0, bi_ = 0.0;
      for (int t = 0; t < N; ++t) {
        const double ur = Uf[t * 2 * N + 2 * a], ui = Uf[t * 2 * N + 2 * a + 1];
        const double wr = ipf[t] * Us[c * 2 * N + 2 * t], wi = ipf[t] * Us[c * 2 * N + 2 * t + 1];
        fr_ = fma(ur, wr, fma(-ui, wi, fr_));
        fi_ = fma(ur, wi, fma(ui, wr, fi_));
        const double vr = Ub[t * 2 * N + 2 * a], vi = Ub[t * 2 * N + 2 * a + 1];
        const double zr = Zc[(c * N + t) * 2], zi = Zc[(c * N + t) * 2 + 1];
        br_ = fma(vr, zr, fma(-vi, zi, br_));
        bi_ = fma(vr, zi, fma(vi, zr, bi_));
      }
      Cf[x] = mk(fr_, fi_);
      Cb[x] = mk(br_, bi_);
    }
  }
}

template <int N, bool SPLIT>
__global__ __launch_bounds__(64, N <= 16 ? 3 : 2) void k_canon_h(const cplx<double>* __restrict__ ext, int E, int ccols,
                                                double pinv_eps, double deps, zd* __restrict__ canon,
                                                double* __restrict__ lfull, double* __restrict__ ws) {
  canon_h_run<N, SPLIT>(ext, E, ccols, pinv_eps, deps, canon, lfull, ws, blockIdx.x);
}

// One job's edges in a launch that covers several jobs' canonicalisers (the serving batch):
// its buffers and parameters, and its first block in the launch.
struct CanonEntry {
  const cplx<double>* ext;
  zd* canon;
  double* lfull;
  double* ws;
  int E, ccols;
  double pinv_eps, deps;
  int block0;
};

// The canonicalisers of several jobs (same n) in one launch: entry e takes blocks
// block0_e .. block0_{e+1} - 1 (found by binary search; block0 ascending, block0_0 = 0).
template <int N, bool SPLIT>
__global__ __launch_bounds__(64, N <= 16 ? 3 : 2) void k_canon_h_multi(const CanonEntry* __restrict__ tab,
                                                                      int entries) {
  int lo = 0, hi = entries - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (tab[mid].block0 <= (int)blockIdx.x)
      lo = mid;
    else
      hi = mid - 1;
  }
  const CanonEntry& e = tab[lo];
  canon_h_run<N, SPLIT>(e.ext, e.E, e.ccols, e.pinv_eps, e.deps, e.canon, e.lfull, e.ws, (int)blockIdx.x - e.block0);
}

}  // namespace bqa
