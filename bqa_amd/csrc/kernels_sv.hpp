// Exact state-vector simulation of the Trotterised anneal (src/bqa/exact_sim.py:14-88),
// FP64, up to 32 qubits on one GPU (2^n complex128 amplitudes + 2^n doubles of
// diagonal energies: 24 GB at 30 qubits, 96 GB at 32).
//
// Qubit q is bit q of the basis index; Z_q = +1 on bit 0.  One Trotter layer is
//   psi <- prod_q exp(-i xtime X_q) exp(-i ztime Ez) psi,
//   Ez(x) = sum_q h_q z_q(x) + sum_(ab) J_ab z_a(x) z_b(x),
// which is the reference's order (every Z gate, every ZZ gate, then every X
// gate, exact_sim.py:51-63); the Z and ZZ gates are diagonal and the X gates on
// different qubits commute.
//
// The X layer runs in passes over groups of qubits, and the readout in the same passes.  A pass takes tiles of 4,096
// amplitudes, sixteen in a thread's registers at a time: the four tile bits that index a thread's registers are
// rotated (or summed over pairs) there, and an exchange through LDS brings the next four into the registers.  The
// first pass takes contiguous tiles (qubits 0..11, with the diagonal phase on the way in); later passes take 2^cb
// contiguous amplitudes (cb >= 4: 256-byte rows and more) times the 2^t values of t = 12 - cb <= 8 higher qubits.
// Bounded by memory: a rotation pass reads and writes the state once, a readout pass reads it.  At 26 qubits (1 GB)
// a layer is three passes and the readout three reads (0.70 + 2 x 0.41 and 0.72 ms); with tiles of 1,024 amplitudes and every rotation through
// LDS they were four passes (2.0 ms a layer) and the readout took 9.6 ms, most of it in lane reductions of every
// qubit of every tile and in a serial sum over the blocks.
// Few amplitudes run on tiles of 1,024 in LDS instead (k_sv_lds): up to 2^17 the register tiles are at most 32 blocks,
// each with the latency of its loads, sixteen sincos a thread and four exchanges.  Microseconds of a layer's call, LDS
// and register tiles: 4 qubits 12.9 and 18.0, 10 16.6 and 19.5, 12 20.0 and 21.1, 13 20.4 and 24.5, 16 23.2 and 26.0, 18
// 29.8 and 29.9, 20 47.6 and 38.4; of a readout's, 4 qubits 41.7 and 51.5, 10 48.7 and 51.8, 11 69.7 and 51.5.
#pragma once

#include "common.hpp"
#include "kernels_mfma.hpp"

namespace bqa {

constexpr int kSvTileBits = 12;            // amplitudes per tile: 4,096, sixteen per thread
constexpr int kSvRowBits = 4;              // least contiguous amplitudes per row in the high-qubit passes
constexpr int kSvThreads = 256;
constexpr int kSvMaxEdges = 2048;          // edges kept in LDS by the energy kernel
constexpr int kSvLdsBits = 10;             // amplitudes per LDS tile: 1,024
constexpr int kSvLdsLayer = 17;            // most qubits whose layers run on LDS tiles
constexpr int kSvLdsRead = kSvLdsBits;     // and whose readout does: one tile

// Ez(x) for every basis state; fields and edges staged in LDS.
__global__ __launch_bounds__(kSvThreads) void k_sv_energy(double* __restrict__ ez, int n, const double* __restrict__ h,
                                                          int E, const int32_t* __restrict__ lhs,
                                                          const int32_t* __restrict__ rhs,
                                                          const double* __restrict__ J) {
  __shared__ double sh[32];
  __shared__ int sa[kSvMaxEdges], sb[kSvMaxEdges];
  __shared__ double sj[kSvMaxEdges];
  for (int q = threadIdx.x; q < n; q += blockDim.x) sh[q] = h[q];
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    sa[e] = lhs[e];
    sb[e] = rhs[e];
    sj[e] = J[e];
  }
  __syncthreads();
  const unsigned long long dim = 1ULL << n;
  for (unsigned long long x = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; x < dim;
       x += (unsigned long long)gridDim.x * blockDim.x) {
    double e = 0.0;
    for (int q = 0; q < n; ++q) e += ((x >> q) & 1ULL) ? -sh[q] : sh[q];
    for (int k = 0; k < E; ++k) e += (((x >> sa[k]) ^ (x >> sb[k])) & 1ULL) ? -sj[k] : sj[k];
    ez[x] = e;
  }
}

// |->^n: psi[x] = (-1)^popcount(x) 2^(-n/2).
__global__ void k_sv_init(cplx<double>* __restrict__ psi, int n) {
  const unsigned long long dim = 1ULL << n;
  const double a = exp2(-0.5 * n);
  for (unsigned long long x = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; x < dim;
       x += (unsigned long long)gridDim.x * blockDim.x)
    psi[x] = mk(__popcll(x) & 1 ? -a : a, 0.0);
}

// One pass over qubits b0 .. b0 + t - 1 on LDS tiles of 2^row contiguous amplitudes times the 2^t values of the qubits
// (row <= b0, row + t <= 10).  MODE 0: the diagonal phase exp(-i ztime Ez) (when ez != nullptr), then the qubits' X
// rotations, each by all threads between two barriers.  MODE 1: the sums of the qubits' readout to part, where a wave
// adds its lanes' pairs by shuffles.
template <int MODE>
__global__ __launch_bounds__(kSvThreads) void k_sv_lds(cplx<double>* __restrict__ psi, int n, int b0, int t, int row,
                                                       const double* __restrict__ ez, double ztime, double c, double sn,
                                                       double* part) {
  __shared__ cplx<double> s[1 << kSvLdsBits];
  __shared__ double sums[4 * kSvLdsBits][kSvThreads / 64];
  const int size = 1 << (row + t), half = size >> 1, mid = b0 - row;
  const unsigned long long tiles = 1ULL << (n - row - t);
  for (unsigned long long T = blockIdx.x; T < tiles; T += gridDim.x) {
    const unsigned long long base = (T & ((1ULL << mid) - 1ULL)) << row | (T >> mid) << (b0 + t);
    auto at = [&](int k) { return base | (unsigned long long)(k & ((1 << row) - 1)) | (unsigned long long)(k >> row) << b0; };
    for (int k = threadIdx.x; k < size; k += kSvThreads) {
      cplx<double> a = psi[at(k)];
      if (MODE == 0 && ez) {
        double sp, cp;
        sincos(-ztime * ez[at(k)], &sp, &cp);
        a = a * mk(cp, sp);
      }
      s[k] = a;
    }
    __syncthreads();
    for (int b = row; b < row + t; ++b) {
      const int m = 1 << b;
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      for (int p = threadIdx.x; p < half; p += kSvThreads) {
        const int k0 = (p >> b) << (b + 1) | (p & (m - 1)), k1 = k0 | m;   // the p-th pair of bit b
        const cplx<double> a0 = s[k0], a1 = s[k1];
        if (MODE == 0) {
          // (cos t) a - i (sin t) X a
          s[k0] = mk(c * a0.x + sn * a1.y, c * a0.y - sn * a1.x);
          s[k1] = mk(c * a1.x + sn * a0.y, c * a1.y - sn * a0.x);
        } else {
          v[0] += abs2(a0);
          v[1] += abs2(a1);
          v[2] = fma(a0.x, a1.x, fma(a0.y, a1.y, v[2]));
          v[3] = fma(a0.x, a1.y, fma(-a0.y, a1.x, v[3]));
        }
      }
      if (MODE == 0) {
        __syncthreads();
      } else {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          for (int o = 32; o > 0; o >>= 1) v[x] += __shfl_xor(v[x], o, 64);
          if ((threadIdx.x & 63) == 0) sums[4 * (b - row) + x][threadIdx.x >> 6] = v[x];
        }
      }
    }
    if (MODE == 0) {
      for (int k = threadIdx.x; k < size; k += kSvThreads) psi[at(k)] = s[k];
      __syncthreads();
    }
  }
  if (MODE == 1) {   // one tile (n <= 10), so the sums are whole
    __syncthreads();
    for (int x = threadIdx.x; x < 4 * t; x += kSvThreads) {
      double v = 0.0;
      for (int w = 0; w < kSvThreads / 64; ++w) v += sums[x][w];
      part[(size_t)blockIdx.x * 4 * kSvTileBits + x] = v;
    }
  }
}

// Tile element of register j in the three layouts: the registers' tile bits are 8..11 (A), 4..7 (B) or 0..3 (C).
enum SvLayout { kSvA, kSvB, kSvC };
template <SvLayout L>
__device__ __forceinline__ int sv_element(int j) {
  const int t = threadIdx.x;
  return L == kSvA ? j << 8 | t : L == kSvB ? (t >> 4) << 8 | j << 4 | (t & 15) : t << 4 | j;
}
constexpr int sv_first_bit(SvLayout l) { return l == kSvA ? 8 : l == kSvB ? 4 : 0; }

// LDS position of tile element k: a linear permutation under which every layout's accesses spread over the banks.
__device__ __forceinline__ constexpr int sv_slot(int k) { return k ^ ((k >> 4) & 15) ^ (((k >> 8) & 1) << 4); }

// The tile from layout L to layout M, one component at a time through 32 KB of LDS (so four blocks share a CU).
template <SvLayout L, SvLayout M>
__device__ __forceinline__ void sv_exchange(cplx<double> (&a)[16], double* s) {
#pragma unroll
  for (int part = 0; part < 2; ++part) {
    // opaque: one position per layout is kept, not sixteen
    const int from = opaque(sv_slot(sv_element<L>(0))), to = opaque(sv_slot(sv_element<M>(0)));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; ++j) s[from ^ sv_slot(j << sv_first_bit(L))] = part ? a[j].y : a[j].x;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; ++j) (part ? a[j].y : a[j].x) = s[to ^ sv_slot(j << sv_first_bit(M))];
  }
}

// exp(-i xtime X) on the registers' tile bits of layout L that lie in [first, last).
template <SvLayout L>
__device__ __forceinline__ void sv_rotate(cplx<double> (&a)[16], int first, int last, double c, double sn) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (sv_first_bit(L) + b < first || sv_first_bit(L) + b >= last) continue;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (j >> b & 1) continue;
      const cplx<double> a0 = a[j], a1 = a[j | 1 << b];
      // (cos t) a - i (sin t) X a
      a[j] = mk(c * a0.x + sn * a1.y, c * a0.y - sn * a1.x);
      a[j | 1 << b] = mk(c * a1.x + sn * a0.y, c * a1.y - sn * a0.x);
    }
  }
}

// Readout sums of the registers' four tile bits, added to this thread's v[b]: r00, r11, Re r10, Im r10 with
// r10 = sum conj(psi0) psi1.
__device__ __forceinline__ void sv_sums(const cplx<double> (&a)[16], double (&v)[4][4]) {
  double norm[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) norm[j] = abs2(a[j]);
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (j >> b & 1) continue;
      const cplx<double> a0 = a[j], a1 = a[j | 1 << b];
      v[b][0] += norm[j];
      v[b][1] += norm[j | 1 << b];
      v[b][2] = fma(a0.x, a1.x, fma(a0.y, a1.y, v[b][2]));
      v[b][3] = fma(a0.x, a1.y, fma(-a0.y, a1.x, v[b][3]));
    }
}

// part[block][tile bit][4] of the bits of layout L from the threads' sums, always in the same order.
template <SvLayout L>
__device__ __forceinline__ void sv_store(const double (&v)[4][4], double* s, double* part) {
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    double r = v[x >> 2][x & 3];
    for (int o = 32; o > 0; o >>= 1) r += __shfl_xor(r, o, 64);
    if ((threadIdx.x & 63) == 0) s[x * (kSvThreads / 64) + (threadIdx.x >> 6)] = r;
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    double r = 0.0;
    for (int w = 0; w < kSvThreads / 64; ++w) r += s[threadIdx.x * (kSvThreads / 64) + w];
    part[(size_t)blockIdx.x * 4 * kSvTileBits + 4 * sv_first_bit(L) + threadIdx.x] = r;
  }
}

// Two waves a SIMD: the sixteen sincos of a thread then run interleaved (26 qubits: 0.70 ms; held to the registers of
// three or four waves 0.89 and 1.09 ms).
// First pass: tiles of 2^tb contiguous amplitudes (tb = min(n, 12); with fewer qubits the tile's other elements are
// zero).  MODE 0: diagonal phase exp(-i ztime Ez) (when ez != nullptr), then the X rotations of qubits 0..tb-1.
// MODE 1: readout sums of qubits 0..tb-1 into part.
template <int MODE>
__global__ __launch_bounds__(kSvThreads, 2) void k_sv_low(cplx<double>* __restrict__ psi, int n,
                                                       const double* __restrict__ ez, double ztime, double c,
                                                       double sn, double* part) {
  __shared__ double s[1 << kSvTileBits];
  const int tb = n < kSvTileBits ? n : kSvTileBits;
  const int size = 1 << tb;
  const unsigned long long tiles = 1ULL << (n - tb);
  double va[4][4] = {}, vb[4][4] = {}, vc[4][4] = {};
  for (unsigned long long T = blockIdx.x; T < tiles; T += gridDim.x) {
    cplx<double>* p = psi + (T << tb);
    cplx<double> a[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int k = sv_element<kSvA>(j);
      a[j] = k < size ? p[k] : mk(0.0, 0.0);
    }
    if (MODE == 0 && ez) {
      const double* e = ez + (T << tb);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int k = sv_element<kSvA>(j);
        double sp, cp;
        sincos(k < size ? -ztime * e[k] : 0.0, &sp, &cp);
        a[j] = a[j] * mk(cp, sp);
      }
    }
    if (MODE == 0) {
      sv_rotate<kSvA>(a, 0, tb, c, sn);
      sv_exchange<kSvA, kSvC>(a, s);
      sv_rotate<kSvC>(a, 0, tb, c, sn);
      sv_exchange<kSvC, kSvB>(a, s);
      sv_rotate<kSvB>(a, 0, tb, c, sn);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int k = sv_element<kSvB>(j);
        if (k < size) p[k] = a[j];
      }
    } else {
      sv_sums(a, va);
      sv_exchange<kSvA, kSvC>(a, s);
      sv_sums(a, vc);
      sv_exchange<kSvC, kSvB>(a, s);
      sv_sums(a, vb);
    }
  }
  if (MODE == 1) {
    sv_store<kSvA>(va, s, part);
    sv_store<kSvB>(vb, s, part);
    sv_store<kSvC>(vc, s, part);
  }
}

// Later passes: qubits b0..b0+t-1 (1 <= t <= 8, b0 >= 12 > cb = 12 - t).  Tile element k: bits below cb the lowest
// qubits, the t bits above them the pass's qubits; the tile number T the remaining bits (those between cb and b0,
// then those above b0 + t).  Readout sums of tile bits below cb are not used.
template <int MODE>
__global__ __launch_bounds__(kSvThreads, MODE == 0 ? 3 : 2) void k_sv_high(cplx<double>* __restrict__ psi, int n, int b0, int t,
                                                        double c, double sn, double* part) {
  __shared__ double s[1 << kSvTileBits];
  const int cb = kSvTileBits - t, mid = b0 - cb;
  const unsigned long long tiles = 1ULL << (n - kSvTileBits);
  double va[4][4] = {}, vb[4][4] = {};
  for (unsigned long long T = blockIdx.x; T < tiles; T += gridDim.x) {
    cplx<double>* p = psi + ((T & ((1ULL << mid) - 1ULL)) << cb) + ((T >> mid) << (b0 + t));
    auto at = [&](int k) { return (unsigned long long)(k & ((1 << cb) - 1)) | (unsigned long long)(k >> cb) << b0; };
    cplx<double> a[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = p[at(sv_element<kSvA>(j))];
    if (MODE == 0) {
      sv_rotate<kSvA>(a, cb, kSvTileBits, c, sn);
      if (t > 4) {
        sv_exchange<kSvA, kSvB>(a, s);
        sv_rotate<kSvB>(a, cb, kSvTileBits, c, sn);
#pragma unroll
        for (int j = 0; j < 16; ++j) p[at(sv_element<kSvB>(j))] = a[j];
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) p[at(sv_element<kSvA>(j))] = a[j];
      }
    } else {
      sv_sums(a, va);
      if (t > 4) {
        sv_exchange<kSvA, kSvB>(a, s);
        sv_sums(a, vb);
      }
    }
  }
  if (MODE == 1) {
    sv_store<kSvA>(va, s, part);
    if (t > 4) sv_store<kSvB>(vb, s, part);
  }
}

// Bloch vectors and densities of qubits q0.. from the block partials of one readout pass: block b takes tile bit
// bit0 + b, a wave each of its four sums.
__global__ __launch_bounds__(kSvThreads) void k_sv_finish(const double* __restrict__ part, int blocks, int q0, int bit0,
                                                          double* rho, double* bloch) {
  __shared__ double s[4];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  double v = 0.0;
  for (int blk = l; blk < blocks; blk += 64) v += part[(size_t)blk * 4 * kSvTileBits + 4 * (bit0 + blockIdx.x) + w];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (l == 0) s[w] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double tr = s[0] + s[1];
  const double r00 = s[0] / tr, r11 = s[1] / tr, r10r = s[2] / tr, r10i = s[3] / tr;
  const int q = q0 + blockIdx.x;
  // rho[p][q'] = sum psi_p conj(psi_q'): rho10 = r10, rho01 = conj(r10)
  if (rho) {
    double* ro = rho + 8 * (size_t)q;
    ro[0] = r00; ro[1] = 0.0; ro[2] = r10r; ro[3] = -r10i;
    ro[4] = r10r; ro[5] = r10i; ro[6] = r11; ro[7] = 0.0;
  }
  if (bloch) {
    double* bo = bloch + 3 * (size_t)q;
    bo[0] = 2.0 * r10r;
    bo[1] = 2.0 * r10i;
    bo[2] = r00 - r11;
  }
}

}  // namespace bqa
