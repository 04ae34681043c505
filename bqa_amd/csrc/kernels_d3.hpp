// BP sweep and extended messages for degree-3 nodes at chi = 8 (the 100,000-qubit regular graphs) on MFMA, for both
// precisions: the register-chained products of kernels_d4.hpp on a whole node tensor (2 x 8^3 elements).
//
// With Y_j = T x_j m_j and the Hermitian messages moved to the bra side (backends.py:381-404 applies both to the ket):
//   out_0 = conj(Y_1) . Y_2,  out_1 = conj(Y_0) . Y_2,  out_2 = conj(Y_0) . Y_1,
// three mode products and three Grams a node.  Y_2 comes straight from the registers of the tensor's global loads,
// which also fill its LDS copy; Y_1 and Y_0 go from their product's registers into their first Gram's MFMAs, and
// through LDS (Y_0 in T's place) only for out_2.  The messages are loaded from memory as MFMA operands.  Everything
// a node reads from memory is loaded while the node before computes, its positions one node earlier.
// What bounds it: 192 MFMAs a node (0.50 ms FP64, 0.25 ms FP32 a sweep of 100,000 nodes at the matrix rate), with four
// short phases a node between barriers; three (FP64) and five (FP32) nodes share a CU.  Measured at 100,000 nodes:
// FP64 0.85 ms a sweep, FP32 0.52 ms; FP64 extended messages 1.19 ms.  The kernels that ran products and Grams
// through LDS took 1.05 ms (six contractions), 0.67 ms (nine) and 1.68 ms.
#pragma once

#include "common.hpp"
#include "kernels_d4.hpp"
#include "kernels_mfma.hpp"
#include "launch_grid.hpp"

namespace bqa {

// LDS position of element (p, b0, b1, b2): as d4_sw, a linear permutation within rows of 16 elements that spreads
// every (column bond, low bit of the row bond) used here over a row's slots.
__device__ __forceinline__ constexpr int d3_sw(int idx) {
  const int b1 = idx >> 3, b0 = idx >> 6;
  return idx ^ (b1 & 6) ^ (b0 & 6) ^ ((b0 & 1) * 9);
}
constexpr int d3_shift(int bond) { return 3 * (2 - bond); }

// An index that the compiler takes for a lane's own, so that the loads it addresses are counted with the other vector
// memory loads: a scalar load in flight would hold up the next wait for LDS until it arrives.
__device__ __forceinline__ int d3_lane_index(int x) { return x + opaque(0); }

// GT: the precision of the Grams.
template <typename R, typename GT>
struct D3 {
  static constexpr int NW = 4, S = 1024, TILES = 8 / NW, UNITS = 16 / NW;
  static constexpr int ES = 2 * sizeof(R), BUF = S * ES;
  static constexpr int RED = NW * 128 * (int)sizeof(double);         // the waves' Gram parts of one output
  static constexpr int FIT = BUF / RED < 3 ? BUF / RED : 3;          // outputs whose parts fit Y_2's buffer
  static constexpr int BYTES = 3 * BUF + (3 - FIT) * RED;
  using Acc = typename D4Acc<R>::type;
  using GAcc = typename D4Acc<GT>::type;

  // What a node reads from memory, as this lane holds it.
  struct Node {
    cplx<R> t[TILES][2];       // tile rows (lowest bit of b0, b1), b2 = kq and kq + 4
    R am[2][2];                // m_0 and m_1 as row operands
    cplx<R> c2[2];             // m_2[cb][kq], m_2[cb][kq + 4]
  };

  unsigned char *T, *Y1, *Y2, *extra;
  int lane, w, i16, kq, row, comp, cb;
  R sg;

  __device__ __forceinline__ D3(unsigned char* lds) : T(lds), Y1(lds + BUF), Y2(lds + 2 * BUF), extra(lds + 3 * BUF) {
    lane = threadIdx.x & 63;
    w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    i16 = lane & 15;
    kq = lane >> 4;
    row = d4_logical<R>(i16);
    const int col = d4_logical<GT>(i16);
    comp = col >> 3;
    cb = col & 7;
    sg = comp ? (R)1 : (R)-1;
  }
  static __device__ __forceinline__ int at(int idx) { return d3_sw(idx) * ES; }

  __device__ __forceinline__ void load(Node& nd, const cplx<R>* __restrict__ T_, const cplx<R>* min, const int (&pin)[3]) const {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const cplx<R>* p = T_ + (w * TILES + t) * 128 + row * 8 + kq;
      nd.t[t][0] = p[0];
      nd.t[t][1] = p[4];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const R* m = reinterpret_cast<const R*>(min + (size_t)pin[j] * 64 + (row & 7) * 8 + kq) + (row >> 3);
      nd.am[j][0] = m[0];
      nd.am[j][1] = m[8];
    }
    const cplx<R>* m = min + (size_t)pin[2] * 64 + cb * 8 + kq;
    nd.c2[0] = m[0];
    nd.c2[1] = m[4];
  }

  // T and Y_2 into LDS.
  __device__ __forceinline__ void front(const Node& nd) const {
    R bm[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) bm[s] = (s >> 1) == comp ? nd.c2[s & 1].x : (s >> 1) ? -nd.c2[s & 1].y : nd.c2[s & 1].y;
    const int ti = opaque(at(row * 8 + kq)), yi = opaque(at(kq * 8 + cb) + comp * (int)sizeof(R));
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int u = at((w * TILES + t) * 128);
      const cplx<R>(&x)[2] = nd.t[t];
      *reinterpret_cast<cplx<R>*>(T + (ti ^ u)) = x[0];
      *reinterpret_cast<cplx<R>*>(T + (ti ^ u ^ at(4))) = x[1];
      Acc d = {0, 0, 0, 0};
      d = d4_mm(x[0].x, bm[0], d);
      d = d4_mm(x[1].x, bm[1], d);
      d = d4_mm(x[0].y, bm[2], d);
      d = d4_mm(x[1].y, bm[3], d);
#pragma unroll
      for (int v = 0; v < 4; ++v) *reinterpret_cast<R*>(Y2 + (yi ^ u ^ at(64 * (v >> 1)) ^ at(32 * (v & 1)))) = d[v];
    }
  }

  __device__ __forceinline__ void add_entries(const GAcc& g0, const GAcc& g1, double (&ge)[2]) const {
    const double s = comp ? -1.0 : 1.0;
#pragma unroll
    for (int v = 0; v < 2; ++v)
      ge[v] = fma(s, d4_other<GT>((double)g0[v + 2] + (double)g1[v + 2]), (double)g0[v] + (double)g1[v]);
  }

  // Y = T x_J m of this wave's (p, other bond) pairs, columns bond K and rows bond J, to `out`, and this wave's part of
  // the Gram along K of conj(Y) and Y_2.
  template <int K, int J>
  __device__ __forceinline__ void product_gram(const R (&am)[2], unsigned char* out, double (&ge)[2]) const {
    const int li = opaque(at(cb << d3_shift(K) | kq << d3_shift(J)) + comp * (int)sizeof(R));
    GAcc g0 = {0, 0, 0, 0}, g1 = {0, 0, 0, 0};
    int pos[UNITS];
    R x0[UNITS], x1[UNITS];   // all reads of T before the first write, which may replace it
#pragma unroll
    for (int q = 0; q < UNITS; ++q) {
      const int e = w * UNITS + q;
      pos[q] = li ^ at((e >> 3) << 9 | (e & 7) << d3_shift(3 - K - J));
      x0[q] = *reinterpret_cast<const R*>(T + pos[q]);
      x1[q] = *reinterpret_cast<const R*>(T + (pos[q] ^ at(4 << d3_shift(J))));
    }
#pragma unroll
    for (int q = 0; q < UNITS; ++q) {
      const int p0 = pos[q], p1 = p0 ^ at(4 << d3_shift(J));
      Acc d = {0, 0, 0, 0};
      d = d4_mm(am[0], x0[q], d);
      d = d4_mm(am[1], x1[q], d);
      const R y0 = fma(sg, d4_other<GT>(d[2]), d[0]), y1 = fma(sg, d4_other<GT>(d[3]), d[1]);
      *reinterpret_cast<R*>(out + p0) = y0;
      *reinterpret_cast<R*>(out + p1) = y1;
      g0 = d4_mm((GT)y0, (GT)*reinterpret_cast<const R*>(Y2 + p0), g0);
      g1 = d4_mm((GT)y1, (GT)*reinterpret_cast<const R*>(Y2 + p1), g1);
    }
    add_entries(g0, g1, ge);
  }

  // This wave's part of the Gram along bond 2 of conj(Y_0) (in T's place) and Y_1: rows bond 0, pairs (p, b1).
  __device__ __forceinline__ void last_gram(double (&ge)[2]) const {
    const int li = opaque(at(cb | kq << 6) + comp * (int)sizeof(R));
    GAcc g0 = {0, 0, 0, 0}, g1 = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < UNITS; ++q) {
      const int e = w * UNITS + q;
      const int p0 = li ^ at((e >> 3) << 9 | (e & 7) << 3), p1 = p0 ^ at(4 << 6);
      g0 = d4_mm((GT)*reinterpret_cast<const R*>(T + p0), (GT)*reinterpret_cast<const R*>(Y1 + p0), g0);
      g1 = d4_mm((GT)*reinterpret_cast<const R*>(T + p1), (GT)*reinterpret_cast<const R*>(Y1 + p1), g1);
    }
    add_entries(g0, g1, ge);
  }

  // The waves' parts of output k's Gram, entries (c, (part, e)) of wave w at [w 128], in Y_2's buffer (dead by then)
  // and beyond it.
  __device__ __forceinline__ double* parts(int k) const {
    return reinterpret_cast<double*>(k < FIT ? Y2 + k * RED : extra + (k - FIT) * RED);
  }
  // The next node's Y_1 and Y_2 change places: its front may then write T and Y_2 while waves still read the parts.
  __device__ __forceinline__ void turn() {
    unsigned char* y = Y1;
    Y1 = Y2;
    Y2 = y;
  }

  // The node's three Grams; pairs of physical half p are those of waves 2 p and 2 p + 1.  Ends with a barrier.
  // `after` runs once the node's registers are read.
  template <typename After>
  __device__ __forceinline__ void run(Node& nd, After after) const {
    front(nd);
    const R a0[2] = {nd.am[0][0], nd.am[0][1]}, a1[2] = {nd.am[1][0], nd.am[1][1]};
    after();
    double ge[3][2];
    __syncthreads();
    product_gram<0, 1>(a1, Y1, ge[0]);
    __syncthreads();
    product_gram<1, 0>(a0, T, ge[1]);
    __syncthreads();
    last_gram(ge[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double* r = parts(k) + w * 128 + comp * 8 + cb;
      r[kq * 16] = ge[k][0];
      r[(kq + 4) * 16] = ge[k][1];
    }
    __syncthreads();
  }
};

// The class's nodes start, start + gridDim.x, ..: one sweep.
template <typename R>
__device__ void bp_d3c8_run(unsigned char* lds, ClassView cv, const cplx<R>* __restrict__ T, cplx<R>* msgA, cplx<R>* msgB,
                            BpStatus* st, int start) {
  using N = D3<R, R>;
  const int cur = bp_begin(st, cv.sweep);
  if (cur < 0) return;
  const cplx<R>* min = cur ? msgB : msgA;
  cplx<R>* mout = cur ? msgA : msgB;
  N s(lds);
  const int n = cv.n, G = gridDim.x, o = threadIdx.x & 63;
  const bool io = s.w < 3;   // waves 0..2 finish bond w's message
  const int kb = io ? s.w : 0;
  int i = start;
  if (i >= n) return;
  double dnum = 0.0, dden = 0.0;
  typename N::Node nd;
  int pin[3], pos = cv.out_pos[kb * n + i], pout = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[k * n + i];
  s.load(nd, T + (size_t)i * N::S, min, pin);
  cplx<R> old = min[(size_t)pos * 64 + o];
  if (i + G < n) {
#pragma unroll
    for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[d3_lane_index(k * n + i + G)];
    pout = cv.out_pos[d3_lane_index(kb * n + i + G)];
  }
  for (; i < n; i += G) {
    const int at = pos;
    const cplx<double> od = cast<double>(old);
    s.run(nd, [&] {
      if (i + G >= n) return;
      s.load(nd, T + (size_t)(i + G) * N::S, min, pin);
      pos = pout;
      old = min[(size_t)pos * 64 + o];
      if (i + 2 * G < n) {
#pragma unroll
        for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[d3_lane_index(k * n + i + 2 * G)];
        pout = cv.out_pos[d3_lane_index(kb * n + i + 2 * G)];
      }
    });
    if (io) {
      const int c = o >> 3, e = o & 7;
      double re = 0.0, im = 0.0;
#pragma unroll
      for (int q = 0; q < N::NW; ++q) {
        const double* r = s.parts(kb) + q * 128 + c * 16 + e;
        re += r[0];
        im += r[8];
      }
      double tr = 0.0;
#pragma unroll
      for (int d = 0; d < 8; ++d) tr += __shfl(re, d * 9, 64);
      const double inv = 1.0 / tr;
      const double rt = __shfl(re, e * 8 + c, 64), it = __shfl(im, e * 8 + c, 64);
      const cplx<R> v = cast<R>(mk(0.5 * (re + rt) * inv, 0.5 * (im - it) * inv));
      const cplx<double> vd = cast<double>(v);
      dnum = fmax(dnum, abs2(vd - od));
      dden = fmax(dden, abs2(vd + od));
      mout[(size_t)at * 64 + o] = v;
    }
    s.turn();
  }
  bp_end_waves<3>(st, cv.sweep, dnum, dden, reinterpret_cast<double*>(lds));
}

// Waves a SIMD: three (FP64) or five (FP32) blocks of four waves share a CU's LDS.
template <typename R>
constexpr int kD3Waves = sizeof(R) == sizeof(double) ? 3 : 5;

template <typename R>
__global__ __launch_bounds__(256, kD3Waves<R>) void k_bp_d3c8(ClassView cv, const cplx<R>* __restrict__ T, cplx<R>* msgA,
                                                              cplx<R>* msgB, BpStatus* st) {
  __shared__ __align__(16) unsigned char lds[D3<R, R>::BYTES];
  bp_d3c8_run<R>(lds, cv, T, msgA, msgB, st, blockIdx.x);
}

// One sweep of the classes of several jobs in one launch, nodes shared over the blocks as in k_small_multi.
template <typename R>
__global__ __launch_bounds__(256, kD3Waves<R>) void k_bp_d3c8_multi(const BpEntry* __restrict__ tab, int entries, int sweep) {
  __shared__ __align__(16) unsigned char lds[D3<R, R>::BYTES];
  for (int e = 0; e < entries; ++e) {
    ClassView cv = tab[e].cv;
    cv.sweep = sweep;
    const long g = gridDim.x;
    const int start = (int)((((long)blockIdx.x - tab[e].prefix) % g + g) % g);
    if (start >= cv.n) continue;  // none of this entry's nodes falls to this block
    bp_d3c8_run<R>(lds, cv, reinterpret_cast<const cplx<R>*>(tab[e].T), reinterpret_cast<cplx<R>*>(tab[e].mA),
                   reinterpret_cast<cplx<R>*>(tab[e].mB), tab[e].st, start);
    __syncthreads();   // the next entry's loads overwrite the LDS this one's last readers use
  }
}

// Extended messages (state.py:127-139, backends.py:393-404,519-526): the same products with the Grams kept per
// physical half, each 16 x 16 message assembled with its bond's ZZ-split gates as in k_ext_d4c8.
// FP64 jobs only: FP32 ones keep k_mfma8_ext32, whose Grams take the tensor itself on one side (1.14 ms; 1.17 here).
__global__ __launch_bounds__(256, 3) void k_ext_d3c8(ClassView cv, const cplx<double>* __restrict__ T,
                                                     const cplx<double>* __restrict__ msgs, cplx<double>* ext_out) {
  using R = double;
  using N = D3<R, R>;
  __shared__ __align__(16) unsigned char lds[N::BYTES];
  const N s(lds);
  cplx<double>* gm = reinterpret_cast<cplx<double>*>(s.T);   // [k][p][64] of the finished Grams (6 KB)
  const int n = cv.n, G = gridDim.x, t = threadIdx.x;
  int i = blockIdx.x;
  if (i >= n) return;
  typename N::Node nd;
  int pin[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[k * n + i];
  s.load(nd, T + (size_t)i * N::S, msgs, pin);
  if (i + G < n) {
#pragma unroll
    for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[d3_lane_index(k * n + i + G)];
  }
  for (; i < n; i += G) {
    s.run(nd, [&] {
      if (i + G >= n) return;
      s.load(nd, T + (size_t)(i + G) * N::S, msgs, pin);
      if (i + 2 * G < n) {
#pragma unroll
        for (int k = 0; k < 3; ++k) pin[k] = cv.in_pos[d3_lane_index(k * n + i + 2 * G)];
      }
    });
    for (int x = t; x < 3 * 128; x += 256) {
      const int kp = x >> 6;   // 2 k + p
      const double* r = s.parts(kp >> 1) + (kp & 1) * 2 * 128 + ((x >> 3) & 7) * 16 + (x & 7);
      gm[x] = mk(r[0] + r[128], r[8] + r[128 + 8]);
    }
    __syncthreads();
    const int row = t >> 4, col = t & 15, s1 = row >> 3, c = row & 7, s2 = col >> 3, e = col & 7;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      cplx<double> tr = mk(0.0, 0.0);
#pragma unroll
      for (int d = 0; d < 8; ++d) tr = tr + gm[(2 * k) * 64 + d * 9] + gm[(2 * k + 1) * 64 + d * 9];
      const cplx<double>* zg = cv.zz + 2 * (size_t)cv.lmbd_pos[k * n + i];
      const cplx<double> g0 = zg[0], g1 = zg[1];
      const cplx<double> inv = cinv(tr * mk(abs2(g0) + abs2(g1), 0.0));
      const cplx<double> a0 = gm[(2 * k) * 64 + c * 8 + e], a1 = gm[(2 * k + 1) * 64 + c * 8 + e];
      const cplx<double> ga = s1 ? g1 : g0, gb = s2 ? g1 : g0;
      ext_out[(size_t)cv.out_pos[k * n + i] * 256 + t] = conj(ga) * gb * (((s1 + s2) & 1) ? a0 - a1 : a0 + a1) * inv;
    }
    __syncthreads();   // the Grams are read
  }
}

template <typename R>
inline void launch_bp_d3c8(ClassView cv, const cplx<R>* T, cplx<R>* mA, cplx<R>* mB, BpStatus* st, hipStream_t s, int policy) {
  int grid = policy_grid<k_bp_d3c8<R>, 256>(cv.n, policy < kGridPolicies ? policy : 0);
  if (policy >= kGridPolicies) {   // as many blocks as give each the same number of nodes, but for one
    const int rounds = (cv.n + grid - 1) / grid;
    grid = (cv.n + rounds - 1) / rounds;
  }
  hipLaunchKernelGGL((k_bp_d3c8<R>), dim3(grid), dim3(256), 0, s, cv, T, mA, mB, st);
}

inline void launch_ext_d3c8(ClassView cv, const cplx<double>* T, const cplx<double>* msgs, cplx<double>* ext, hipStream_t s) {
  hipLaunchKernelGGL(k_ext_d3c8, dim3(node_grid<k_ext_d3c8, 256>(cv.n)), dim3(256), 0, s, cv, T, msgs, ext);
}

}  // namespace bqa
