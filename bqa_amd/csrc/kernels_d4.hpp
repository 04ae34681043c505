// BP sweep and extended messages for degree-4 nodes at chi = 8 (the 100x100 grid's interior, the
// d = 4 serving jobs) on MFMA, for both precisions.  A node tensor is 2 x 8^4 complex elements, so
// the kernels work on one physical half T_p (4096 elements) at a time.
//
// The reference computes out_k = Gram over every bond but k of conj(T) against T contracted with the
// three other incoming messages (backends.py:381-404).  Every message is Hermitian, so a message can
// act on the bra side instead: sum_a conj(T[..a..]) m[a][b] = conj((T x m)[..b..]).  With that, per half:
//   B = T x2 m2 x3 m3;  out_1 += conj(T x0 m0) . B;  out_0 += conj(T x1 m1) . B;
//   B = T x1 m1 x0 m0;  out_3 += conj(T x2 m2) . B;  out_2 += conj(T x3 m3) . B;
// eight mode products and four Grams per half (the reference's schedule: twelve and four).
//
// What bounds it: the twelve contractions are 6.3 MFLOP a node, 0.82 ms (FP64) and 0.40 ms (FP32) for the
// 9,604 interior nodes of the 100x100 grid at the matrix rates a large product reaches, against 0.24 and
// 0.12 ms for the tensors' bytes: the matrix cores, if they are kept fed.  So the products are chained
// in registers and LDS holds only T_p and B:
//   * a 16 x 16 MFMA result (rows: register and lane / 16; columns: lane % 16) is, register by register,
//     the B operand of a product over its rows, and the A or B operand of a Gram over them.  Components
//     sit with the column bond, so a product over the row bond computes m_r X and m_i X for both
//     components (the same number of MFMAs) and adds the two with one lane exchange (d4_combine);
//   * B's two products chain that way per tile of 128 elements, the first one straight from the global
//     loads of T_p (the same registers fill T_p's LDS copy), the second one's tiles from LDS;
//   * a Gram's bra (one mode product of T_p) goes from the product's registers into the Gram's MFMAs;
//     only its T_p and B operands come from LDS.
// Four barriers a half, T_p read from memory once, the next half's loads in flight during the last
// Grams of this one.  Measured, a sweep of the 9,604 nodes: FP64 1.18 ms with sixteen waves per node (1.30 with
// eight), FP32 0.60 ms with eight and two nodes per CU; the extended messages 1.35 and 0.88 ms (eight waves;
// sixteen in FP64: 1.38).  With every product and Gram through LDS in place, about twenty barriers a half and
// T_p reloaded six times: 2.49, 1.68, 3.18 and 1.84 ms.
#pragma once

#include "common.hpp"
#include "kernels_mfma.hpp"
#include "launch_grid.hpp"

namespace bqa {

// LDS position of half-tensor element (b0 b1 b2 b3), three bits each from bit 11 down: a GF(2)-linear
// permutation within aligned rows of 16 elements under which the elements that 32 lanes read or write
// together (eight values of the column bond and the low bit of the row bond, for every pair of bonds
// used here) fall on the 16 different slots of a row.
__device__ __forceinline__ constexpr int d4_sw(int idx) {
  const int b2 = idx >> 3, b1 = idx >> 6, b0 = idx >> 9;
  return idx ^ (b2 & 6) ^ (b1 & 7) ^ (b0 & 6) ^ ((b0 & 1) << 3);
}

constexpr int kD4Half = 4096;                          // elements of a physical half
constexpr int d4_shift(int bond) { return 3 * (3 - bond); }

__device__ __forceinline__ f4v d4_mm(float a, float b, f4v c) { return mfma4(a, b, c); }
__device__ __forceinline__ d4v d4_mm(double a, double b, d4v c) { return mfma4d(a, b, c); }

template <typename R>
struct D4Acc;
template <>
struct D4Acc<float> {
  using type = f4v;
};
template <>
struct D4Acc<double> {
  using type = d4v;
};

// The logical row or column kept at index i of a 16-wide tile side, so that result register v of lane l
// holds logical row l / 16 + 4 v in both precisions (the FP32 instruction's registers hold rows
// 4 (l / 16) + v).  Bit 3 of a logical row or column is its component, real part or half tile.
template <typename R>
__device__ __forceinline__ int d4_logical(int i) {
  return sizeof(R) == sizeof(double) ? i : (i >> 2) + 4 * (i & 3);
}

// Value of the lane whose column is the other component (logical columns in the order of GT).
template <typename GT>
__device__ __forceinline__ int d4_other32(int v) {
  if constexpr (sizeof(GT) == sizeof(double))
    return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);  // lane ^ 8: rotate the row by 8
  else
    return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);   // lane ^ 2: quad permutation
}
template <typename GT>
__device__ __forceinline__ double d4_other(double x) {
  return __hiloint2double(d4_other32<GT>(__double2hiint(x)), d4_other32<GT>(__double2loint(x)));
}
template <typename GT>
__device__ __forceinline__ float d4_other(float x) {
  return __int_as_float(d4_other32<GT>(__float_as_int(x)));
}

template <typename R, typename GT, int NW>
struct D4 {
  static_assert(NW == 8 || NW == 16, "eight or sixteen waves per node");
  static constexpr int H = kD4Half, NT = 64 * NW, TILES = 32 / NW;
  static constexpr int ES = 2 * sizeof(R);                         // bytes of an element
  static constexpr int BUF = H * ES;                               // bytes of T_p or B
  using Acc = typename D4Acc<R>::type;
  using GAcc = typename D4Acc<GT>::type;

  unsigned char *T, *B;    // T_p and B, swizzled
  int lane, w, i16, kq;    // w is the same for a whole wave
  int row, comp, cb;       // logical row of lane % 16; component and bond index of its column
  R sg;                    // what the other component's m_i product adds with

  __device__ __forceinline__ D4(unsigned char* lds) {
    T = lds;
    B = lds + BUF;
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

  // Byte position of element idx (and of its part `comp`): linear over XOR in idx.
  static __device__ __forceinline__ int at(int idx) { return d4_sw(idx) * ES; }

  // Message operand of a product over the row bond: m_r (logical rows 0..7) and m_i (8..15) of m[a][b].
  __device__ __forceinline__ void row_operand(const cplx<R>* m, R (&am)[2]) const {
    const int a = row & 7;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const cplx<R> v = m[a * 8 + kq + 4 * s];
      am[s] = (row >> 3) ? v.y : v.x;
    }
  }
  // Message operand of a product whose result's columns are the product's bond.
  __device__ __forceinline__ void col_operand(const cplx<R>* m, R (&bm)[4]) const {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const cplx<R> v = m[cb * 8 + kq + 4 * (s & 1)];
      bm[s] = (s >> 1) == comp ? v.x : (s >> 1) ? -v.y : v.y;
    }
  }
  // Both results of the row product am on the 8 x 16 operand (x0, x1): rows kq and kq + 4.
  __device__ __forceinline__ void row_product(const R (&am)[2], R x0, R x1, R& y0, R& y1) const {
    Acc d = {0, 0, 0, 0};
    d = d4_mm(am[0], x0, d);
    d = d4_mm(am[1], x1, d);
    y0 = fma(sg, d4_other<GT>(d[2]), d[0]);
    y1 = fma(sg, d4_other<GT>(d[3]), d[1]);
  }
  // Two chained products of one tile: rows (x, row bond) of xa times bm, then the row bond's am; the
  // results go to B at `base` (lane part included) + x * stx + 4 v * sty.
  __device__ __forceinline__ void chain_tile(const cplx<R> (&x)[2], const R (&bm)[4], const R (&am)[2], int pos, int stx,
                                             int st4) {
    Acc d = {0, 0, 0, 0};
    d = d4_mm(x[0].x, bm[0], d);
    d = d4_mm(x[1].x, bm[1], d);
    d = d4_mm(x[0].y, bm[2], d);
    d = d4_mm(x[1].y, bm[3], d);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      R y0, y1;
      row_product(am, d[2 * h], d[2 * h + 1], y0, y1);
      const int p = h ? pos ^ stx : pos;
      *reinterpret_cast<R*>(B + p) = y0;
      *reinterpret_cast<R*>(B + (p ^ st4)) = y1;
    }
  }

  // T_p tile t of this wave: (b0, upper bits of b1), rows (lowest bit of b1, b2), b3 = kq and kq + 4.
  __device__ __forceinline__ void load(const cplx<R>* __restrict__ Tp, cplx<R> (&xt)[TILES][2]) const {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const cplx<R>* p = Tp + (w * TILES + t) * 128 + row * 8 + kq;
      xt[t][0] = p[0];
      xt[t][1] = p[4];
    }
  }
  // T_p into LDS and B = T x3 m3 x2 m2.
  __device__ __forceinline__ void front(const cplx<R> (&xt)[TILES][2], const cplx<R>* M) {
    R bm[4], am[2];
    col_operand(M + 3 * 64, bm);
    row_operand(M + 2 * 64, am);
    const int ti = opaque(at(row * 8 + kq)), bi = opaque(at(kq * 8 + cb) + comp * (int)sizeof(R));
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int u = at((w * TILES + t) * 128);
      *reinterpret_cast<cplx<R>*>(T + (ti ^ u)) = xt[t][0];
      *reinterpret_cast<cplx<R>*>(T + (ti ^ u ^ at(4))) = xt[t][1];
      chain_tile(xt[t], bm, am, bi ^ u, at(64), at(32));
    }
  }
  // B = T x1 m1 x0 m0, tiles (b2, upper bits of b3) with rows (lowest bit of b3, b0).
  __device__ __forceinline__ void middle(const cplx<R>* M) {
    R bm[4], am[2];
    col_operand(M + 1 * 64, bm);
    row_operand(M, am);
    const int ti = opaque(at((row >> 3) | (row & 7) << 9 | kq << 6));
    const int bi = opaque(at(kq << 9 | cb << 6) + comp * (int)sizeof(R));
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int u = at((w * TILES + t) * 2);
      cplx<R> x[2];
      x[0] = *reinterpret_cast<const cplx<R>*>(T + (ti ^ u));
      x[1] = *reinterpret_cast<const cplx<R>*>(T + (ti ^ u ^ at(4 << 6)));
      chain_tile(x, bm, am, bi ^ u, at(1), at(4 << 9));
    }
  }
  // This wave's part of the Gram over all bonds but K of conj(T x_J m) and B: columns bond K, rows bond J,
  // the other two bonds' 64 pairs split over the waves.  Adds its entries (c, (part, e)) for c = kq and
  // kq + 4 and the lane's column to ge, in FP64 from two chains.
  template <int K, int J>
  __device__ __forceinline__ void gram(const cplx<R>* m, double (&ge)[2]) const {
    constexpr int O1 = K != 0 && J != 0 ? 0 : K != 1 && J != 1 ? 1 : 2;
    constexpr int O2 = 6 - K - J - O1;
    constexpr int S1 = d4_shift(O1), S2 = d4_shift(O2);
    R am[2];
    row_operand(m, am);
    // opaque: the addresses are formed next to their accesses, not hoisted out of the node loop
    const int li = opaque(at(cb << d4_shift(K) | kq << d4_shift(J)) + comp * (int)sizeof(R));
    GAcc g0 = {0, 0, 0, 0}, g1 = {0, 0, 0, 0};
#pragma unroll 4
    for (int q = 0; q < 64 / NW; ++q) {
      const int e = w * (64 / NW) + q;
      const int p0 = li ^ at((e >> 3) << S1 | (e & 7) << S2), p1 = p0 ^ at(4 << d4_shift(J));
      R y0, y1;
      row_product(am, *reinterpret_cast<const R*>(T + p0), *reinterpret_cast<const R*>(T + p1), y0, y1);
      const R b0 = *reinterpret_cast<const R*>(B + p0), b1 = *reinterpret_cast<const R*>(B + p1);
      g0 = d4_mm((GT)y0, (GT)b0, g0);
      g1 = d4_mm((GT)y1, (GT)b1, g1);
    }
    // conj(A) B: re = D[(0,c)][(0,e)] + D[(1,c)][(1,e)], im = D[(0,c)][(1,e)] - D[(1,c)][(0,e)]
    const double sgn = comp ? -1.0 : 1.0;
#pragma unroll
    for (int v = 0; v < 2; ++v)
      ge[v] += fma(sgn, d4_other<GT>((double)g0[v + 2] + (double)g1[v + 2]), (double)g0[v] + (double)g1[v]);
  }
};

// One physical half: adds the half's four Grams to ge[k].  xt holds the half's tiles; `next` runs
// before the last two Grams (the next half's loads into xt).
template <typename R, typename GT, int NW, typename Next>
__device__ __forceinline__ void d4_half(D4<R, GT, NW>& s, const cplx<R>* M, cplx<R> (&xt)[D4<R, GT, NW>::TILES][2],
                                        double (&ge)[4][2], Next next) {
  s.front(xt, M);
  __syncthreads();
  s.template gram<1, 0>(M, ge[1]);
  s.template gram<0, 1>(M + 64, ge[0]);
  __syncthreads();
  s.middle(M);
  next();
  __syncthreads();
  s.template gram<3, 2>(M + 2 * 64, ge[3]);
  s.template gram<2, 3>(M + 3 * 64, ge[2]);
  __syncthreads();
}

// T_p and B, the messages twice (this node's and the next one's).
template <typename R>
struct D4Lds {
  static constexpr int BYTES = (2 * kD4Half + 2 * 256) * (int)sizeof(cplx<R>);
};

// FP64: one block per CU (136 KB of LDS).  FP32: two.
template <typename R, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4 * (sizeof(R) == sizeof(float) ? 2 : 1)) void k_bp_d4c8(
    ClassView cv, const cplx<R>* __restrict__ T, cplx<R>* msgA, cplx<R>* msgB, BpStatus* st) {
  constexpr int H = kD4Half;
  extern __shared__ __align__(16) unsigned char d4_lds[];
  const int cur = bp_begin(st, cv.sweep);
  if (cur < 0) return;
  const cplx<R>* min = cur ? msgB : msgA;
  cplx<R>* mout = cur ? msgA : msgB;
  D4<R, R, NW> s(d4_lds);
  cplx<R>* M0 = reinterpret_cast<cplx<R>*>(d4_lds + 2 * s.BUF);
  double* red = reinterpret_cast<double*>(d4_lds);  // [k][wave][row][part][e]: 4 NW KB over T_p and B
  const int n = cv.n;
  const int t = threadIdx.x, o = t & 63;
  const bool io = s.w < 4;  // waves 0..3 move bond w's messages
  double dnum = 0.0, dden = 0.0;
  int i = blockIdx.x;
  if (i >= n) return;
  cplx<R> xt[s.TILES][2];
  s.load(T + (size_t)i * 2 * H, xt);
  if (io) M0[t] = min[(size_t)cv.in_pos[s.w * n + i] * 64 + o];
  __syncthreads();
  for (int turn = 0; i < n; i += gridDim.x, turn ^= 1) {
    const cplx<R>* M = M0 + turn * 256;
    const int ni = i + (int)gridDim.x;
    cplx<R> nm = mk((R)0, (R)0);
    double ge[4][2];
#pragma unroll
    for (int k = 0; k < 4; ++k) ge[k][0] = ge[k][1] = 0.0;
#pragma unroll 1
    for (int p = 0; p < 2; ++p) {
      d4_half(s, M, xt, ge, [&] {
        if (p == 0)
          s.load(T + (size_t)i * 2 * H + H, xt);
        else if (ni < n) {
          s.load(T + (size_t)ni * 2 * H, xt);
          if (io) nm = min[(size_t)cv.in_pos[s.w * n + ni] * 64 + o];
        }
      });
    }
    if (io) M0[(turn ^ 1) * 256 + t] = nm;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double* r = red + (k * NW + s.w) * 128 + s.comp * 8 + s.cb;
      r[s.kq * 16] = ge[k][0];
      r[(s.kq + 4) * 16] = ge[k][1];
    }
    __syncthreads();
    if (io) {
      const int k = s.w, c = o >> 3, e = o & 7;
      const size_t pos = (size_t)cv.out_pos[k * n + i];
      const cplx<double> od = cast<double>(min[pos * 64 + o]);
      double re = 0.0, im = 0.0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        const double* r = red + (k * NW + q) * 128 + c * 16 + e;
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
      mout[pos * 64 + o] = v;
    }
    __syncthreads();  // the sums are read, the next node's messages in place
  }
  bp_end_waves<4>(st, cv.sweep, dnum, dden, reinterpret_cast<double*>(d4_lds));
}

template <typename R, int NW>
inline void launch_bp_d4c8(ClassView cv, const cplx<R>* T, cplx<R>* mA, cplx<R>* mB, BpStatus* st, hipStream_t s) {
  constexpr int LDS = D4Lds<R>::BYTES;
  const int grid = node_grid_lds<k_bp_d4c8<R, NW>, 64 * NW, LDS>(cv.n, 1);
  hipLaunchKernelGGL((k_bp_d4c8<R, NW>), dim3(grid), dim3(64 * NW), LDS, s, cv, T, mA, mB, st);
}

// Extended messages (state.py:127-139, backends.py:393-404,519-526): the same products per physical half
// (FP32 jobs: FP32 mode products, the Grams on FP64 MFMA from the FP32 operands), the Grams G_p kept per
// half, and each 16 x 16 message assembled with the bond's ZZ-split gates g0, g1:
//   ext[(s,c),(s',e)] = conj(g_s) g_s' (G_0 +- G_1)[c][e] / (trace * (|g0|^2 + |g1|^2)),
// + for s + s' even.
template <typename R, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4 * (sizeof(R) == sizeof(float) ? 2 : 1)) void k_ext_d4c8(
    ClassView cv, const cplx<R>* __restrict__ T, const cplx<R>* __restrict__ msgs, cplx<double>* ext_out) {
  constexpr int H = kD4Half, NT = 64 * NW;
  // the sums [p][k][wave][128] over T_p and B
  static_assert(2 * 4 * NW * 128 * (int)sizeof(double) <= 2 * H * (int)sizeof(cplx<R>), "reduction fits T_p and B");
  extern __shared__ __align__(16) unsigned char d4_lds[];
  D4<R, double, NW> s(d4_lds);
  cplx<R>* M = reinterpret_cast<cplx<R>*>(d4_lds + 2 * s.BUF);
  double* red = reinterpret_cast<double*>(d4_lds);
  cplx<double>* gm = reinterpret_cast<cplx<double>*>(d4_lds);  // [k][p][64], once the sums are read
  const int n = cv.n;
  const int t = threadIdx.x, o = t & 63;
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    cplx<R> xt[s.TILES][2];
    s.load(T + (size_t)i * 2 * H, xt);
    if (s.w < 4) M[t] = msgs[(size_t)cv.in_pos[s.w * n + i] * 64 + o];
    __syncthreads();
    double ge[2][4][2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int k = 0; k < 4; ++k) ge[p][k][0] = ge[p][k][1] = 0.0;
      d4_half(s, M, xt, ge[p], [&] {
        if (p == 0) s.load(T + (size_t)i * 2 * H + H, xt);
      });
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        double* r = red + ((p * 4 + k) * NW + s.w) * 128 + s.comp * 8 + s.cb;
        r[s.kq * 16] = ge[p][k][0];
        r[(s.kq + 4) * 16] = ge[p][k][1];
      }
    __syncthreads();
    cplx<double> sum = mk(0.0, 0.0);
    const int x = t;  // (p, k, c, e), one a thread
    if (x < 512) {
      const double* r = red + ((x >> 8) * 4 + ((x >> 6) & 3)) * NW * 128 + ((x >> 3) & 7) * 16 + (x & 7);
      double re = 0.0, im = 0.0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        re += r[q * 128];
        im += r[q * 128 + 8];
      }
      sum = mk(re, im);
    }
    __syncthreads();
    if (x < 512) gm[(((x >> 6) & 3) * 2 + (x >> 8)) * 64 + (x & 63)] = sum;
    __syncthreads();
    for (int y = t; y < 4 * 256; y += NT) {
      const int k = y >> 8, e16 = y & 255, row = e16 >> 4, col = e16 & 15;
      const int s1 = row >> 3, c = row & 7, s2 = col >> 3, e = col & 7;
      cplx<double> tr = mk(0.0, 0.0);
#pragma unroll
      for (int d = 0; d < 8; ++d) tr = tr + gm[(k * 2) * 64 + d * 9] + gm[(k * 2 + 1) * 64 + d * 9];
      const cplx<double>* zg = cv.zz + 2 * (size_t)cv.lmbd_pos[k * n + i];
      const cplx<double> g0 = zg[0], g1 = zg[1];
      const cplx<double> inv = cinv(tr * mk(abs2(g0) + abs2(g1), 0.0));
      const cplx<double> a0 = gm[(k * 2) * 64 + c * 8 + e], a1 = gm[(k * 2 + 1) * 64 + c * 8 + e];
      const cplx<double> ga = s1 ? g1 : g0, gb = s2 ? g1 : g0;
      ext_out[(size_t)cv.out_pos[k * n + i] * 256 + e16] = conj(ga) * gb * (((s1 + s2) & 1) ? a0 - a1 : a0 + a1) * inv;
    }
    __syncthreads();  // the Grams are read
  }
}

template <typename R, int NW>
inline void launch_ext_d4c8(ClassView cv, const cplx<R>* T, const cplx<R>* msgs, cplx<double>* ext, hipStream_t s) {
  constexpr int LDS = D4Lds<R>::BYTES;
  const int grid = node_grid_lds<k_ext_d4c8<R, NW>, 64 * NW, LDS>(cv.n, 1);
  hipLaunchKernelGGL((k_ext_d4c8<R, NW>), dim3(grid), dim3(64 * NW), LDS, s, cv, T, msgs, ext);
}

}  // namespace bqa
