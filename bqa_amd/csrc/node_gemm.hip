// Node contractions as batched matrix products (interface and plan: node_gemm.hpp).
//
// A node tensor T[p, b_1 .. b_d] is too large for LDS at chi > 16 (512 KB at chi = 32, d = 3) and at
// degree 5 from chi = 8, and a block per node leaves the chip idle on small graphs.  Here every
// partial product of a class goes through a workspace in HBM (sized so a chunk of nodes stays in the
// 256 MB Infinity Cache), one launch per level over (node, product, tiles of fibres), and one launch
// of Grams over (node, output).  Both are complex products on MFMA tiles of 16 x 16 x 4 in the real
// form of eight complex rows (a row for each real and imaginary part), so chi need only be a multiple
// of 8 in the rows and of 4 in the summed index to waste nothing.  A wave keeps its message
// fragments in registers and streams fibres straight from memory: 16 lanes read 16 neighbouring
// fibres (128 bytes in FP32), nothing is staged through LDS, and the next tile is in flight
// while this one multiplies.
#include "node_gemm.hpp"

#include <algorithm>

namespace bqa {

namespace {

constexpr int kGemmThreads = 256;
constexpr int kGemmWaves = kGemmThreads / 64;

template <typename R>
struct Vec4T {
  typedef R type __attribute__((ext_vector_type(4)));
};
template <typename R>
using vec4 = typename Vec4T<R>::type;

__device__ __forceinline__ vec4<float> mfma4(float a, float b, vec4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ vec4<double> mfma4(double a, double b, vec4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Value of lane ^ 1 (a quad permutation).
__device__ __forceinline__ float swap1(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ double swap1(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Row r of a 16-row tile holds part ri (0 real, 1 imaginary) of complex row a of eight, such that a
// lane's four result registers are two whole complex numbers, rows a = 2 g and 2 g + 1 of its lane
// group g = lane / 16 (FP32 results lie in rows 4 g + v, FP64 in g + 4 v).
template <typename R>
__device__ __forceinline__ void tile_row(int r, int& a, int& ri);
template <>
__device__ __forceinline__ void tile_row<float>(int r, int& a, int& ri) {
  a = r >> 1;
  ri = r & 1;
}
template <>
__device__ __forceinline__ void tile_row<double>(int r, int& a, int& ri) {
  a = 2 * (r & 3) + (r >> 3);
  ri = (r >> 2) & 1;
}
// Result row of register v of lane group g.
template <typename R>
__device__ __forceinline__ int result_row(int g, int v) {
  return sizeof(R) == 4 ? 4 * g + v : g + 4 * v;
}

// A wave's fragments of the matrix W (rows a < ma, columns b < kb, element (a, b) at w[a * sa + b * sb]):
// re / im [mt][ks] multiply the real / imaginary part of source element b = 4 ks + g.
template <typename R, int KS, int MT>
struct MatFrag {
  R re[MT][KS], im[MT][KS];
  template <typename RM>
  __device__ __forceinline__ void load(const cplx<RM>* __restrict__ w, int ma, int kb, int sa, int sb) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    int al, ri;
    tile_row<R>(r, al, ri);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int a = 8 * mt + al, b = 4 * ks + g;
        cplx<RM> v = mk<RM>(0, 0);
        if (a < ma && b < kb) v = w[a * sa + b * sb];
        re[mt][ks] = (R)(ri == 0 ? v.x : v.y);
        im[mt][ks] = (R)(ri == 0 ? -v.y : v.x);
      }
  }
};

// dst[o, a, i] = sum_b W[a, b] src[o, b, i] for fibres f = o * inner + i in [f0, f1), 16 at a time;
// this wave takes tiles `wave`, `wave + step`, ...
template <typename R, typename RS, int KS, int MT>
__device__ __forceinline__ void product_tiles(const MatFrag<R, KS, MT>& w, const cplx<RS>* __restrict__ src,
                                              cplx<R>* __restrict__ dst, int kb, int ma, int inner, int f0, int f1,
                                              int wave, int step) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int tiles = (f1 - f0 + 15) >> 4;
  int soff = 0, doff = 0;
  bool live = false;
  cplx<RS> nx[KS];
  auto fetch = [&](int t) {
    const int f = f0 + 16 * t + r;
    live = f < f1;
    const int o = f / inner, i = f - o * inner;
    soff = o * kb * inner + i;
    doff = o * ma * inner + i;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int b = 4 * ks + g;
      nx[ks] = mk<RS>(0, 0);
      if (live && b < kb) nx[ks] = src[soff + b * inner];
    }
  };
  if (wave < tiles) fetch(wave);
  for (int t = wave; t < tiles; t += step) {
    R xr[KS], xi[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      xr[ks] = (R)nx[ks].x;
      xi[ks] = (R)nx[ks].y;
    }
    const int at = doff;
    const bool on = live;
    if (t + step < tiles) fetch(t + step);
    vec4<R> acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = vec4<R>{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma4(w.re[mt][ks], xr[ks], acc[mt]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma4(w.im[mt][ks], xi[ks], acc[mt]);
    }
    if (on) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int a = 8 * mt + 2 * g + h;
          if (a < ma) dst[at + a * inner] = mk<R>(acc[mt][2 * h], acc[mt][2 * h + 1]);
        }
    }
  }
}

// Two neighbouring elements in one access (an even element index).
template <typename R>
struct alignas(4 * sizeof(R) <= 16 ? 4 * sizeof(R) : 16) Pair {
  cplx<R> a, b;
};

// acc[mt][nt] += tile (rows: parts of X's free index, columns: parts of Y's) of the real products of
// X[f, c] and Y[f, e] over fibres [f0, f1), 16 at a time; this wave takes groups `wave`, `wave + step`.
// Lanes of a pair load two fibres each for one row of eight and swap the parts the other needs,
// so every element is read once and 16 fibres come as whole lines.
template <typename R, int MT, bool PAIR, typename RX, typename RY>
__device__ __forceinline__ void gram_tiles(vec4<R> (&acc)[MT][MT], const cplx<RX>* __restrict__ X,
                                           const cplx<RY>* __restrict__ Y, int chi, int inner, int f0, int f1,
                                           int wave, int step) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int cl = r >> 1, ri = r & 1;
  const int groups = (f1 - f0 + 15) >> 4;
  // groups in flight while one multiplies: more where a group is few loads
  constexpr int kAhead = MT == 1 ? 4 : MT == 2 ? 2 : 1;
  cplx<RX> bx[kAhead][MT][2];
  cplx<RY> by[kAhead][MT][2];
  auto fetch = [&](int q, cplx<RX>(&nx)[MT][2], cplx<RY>(&ny)[MT][2]) {
    const int f = f0 + 16 * q + 4 * g + 2 * ri;
    const int o0 = f / inner, i0 = f - o0 * inner;
    const int at0 = o0 * chi * inner + i0;
    int at1 = at0 + 1;
    if constexpr (!PAIR) {
      const int o1 = (f + 1) / inner;
      at1 = o1 * chi * inner + (f + 1 - o1 * inner);
    }
    const bool on0 = f < f1, on1 = f + 1 < f1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int c = 8 * mt + cl;
      nx[mt][0] = nx[mt][1] = mk<RX>(0, 0);
      ny[mt][0] = ny[mt][1] = mk<RY>(0, 0);
      if (c < chi) {
        if constexpr (PAIR) {
          if (on0) {
            const Pair<RX> px = *reinterpret_cast<const Pair<RX>*>(X + at0 + c * inner);
            const Pair<RY> py = *reinterpret_cast<const Pair<RY>*>(Y + at0 + c * inner);
            nx[mt][0] = px.a;
            nx[mt][1] = px.b;
            ny[mt][0] = py.a;
            ny[mt][1] = py.b;
          }
        } else {
          if (on0) {
            nx[mt][0] = X[at0 + c * inner];
            ny[mt][0] = Y[at0 + c * inner];
          }
          if (on1) {
            nx[mt][1] = X[at1 + c * inner];
            ny[mt][1] = Y[at1 + c * inner];
          }
        }
      }
    }
  };
  auto spread = [&](const auto& v, R (&out)[4]) {
    const R s0 = (R)(ri ? v[0].x : v[0].y), s1 = (R)(ri ? v[1].x : v[1].y);
    const R m0 = (R)(ri ? v[0].y : v[0].x), m1 = (R)(ri ? v[1].y : v[1].x);
    const R q0 = swap1(s0), q1 = swap1(s1);
    out[0] = ri ? q0 : m0;
    out[1] = ri ? q1 : m1;
    out[2] = ri ? m0 : q0;
    out[3] = ri ? m1 : q1;
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (wave + u * step < groups) fetch(wave + u * step, bx[u], by[u]);
  for (int q0 = wave; q0 < groups; q0 += kAhead * step) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int q = q0 + u * step;
      if (u > 0 && q >= groups) break;
      R a[MT][4], b[MT][4];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        spread(bx[u][mt], a[mt]);
        spread(by[u][mt], b[mt]);
      }
      if (q + kAhead * step < groups) fetch(q + kAhead * step, bx[u], by[u]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < MT; ++nt) acc[mt][nt] = mfma4(a[mt][t], b[nt][t], acc[mt][nt]);
    }
  }
}

template <typename R, int MT, typename RX, typename RY>
__device__ __forceinline__ void gram_range(vec4<R> (&acc)[MT][MT], const cplx<RX>* X, const cplx<RY>* Y, int chi,
                                           int inner, int f0, int f1, int wave, int step) {
  if ((inner & 1) == 0)
    gram_tiles<R, MT, true>(acc, X, Y, chi, inner, f0, f1, wave, step);
  else
    gram_tiles<R, MT, false>(acc, X, Y, chi, inner, f0, f1, wave, step);
}

// sum[row][col] (16 MT square) of the waves' tiles, one wave after the other, in FP64.
template <typename R, int MT>
__device__ __forceinline__ void add_tiles(double* sum, const vec4<R> (&acc)[MT][MT], bool first) {
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < MT; ++nt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double* s = sum + (16 * mt + result_row<R>(g, v)) * 16 * MT + 16 * nt + col;
        *s = first ? (double)acc[mt][nt][v] : *s + (double)acc[mt][nt][v];
      }
}

// LDS tile sums (2 MT^2 KB each) that WG waves share: 64 KB of them over `groups` groups of waves.
template <int MT, int WG>
constexpr int gram_slots(int groups) {
  int s = WG;
  while (s > 1 && s * groups * 2 * MT * MT > 64) s /= 2;
  return s;
}

// The sum of the WG waves' tiles of each of `groups` groups, in FP64 in slot 0 of the group: the waves add to the
// slots in turns, then all threads add the slots, always in the same order.
template <typename R, int MT, int WG>
__device__ __forceinline__ void sum_tiles(double* slots, const vec4<R> (&acc)[MT][MT], int group, int w, int groups) {
  constexpr int SZ = 256 * MT * MT;
  const int S = groups == 1 ? gram_slots<MT, WG>(1) : gram_slots<MT, WG>(2);
  double* own = slots + group * S * SZ;
#pragma unroll 1
  for (int turn = 0; turn < WG / S; ++turn) {
    if (w / S == turn) add_tiles<R, MT>(own + (w % S) * SZ, acc, turn == 0);
    __syncthreads();
  }
  if (S > 1) {
    for (int x = threadIdx.x; x < groups * SZ; x += groups * WG * 64) {
      double* at = slots + (x / SZ) * S * SZ + x % SZ;
      double v = at[0];
      for (int q = 1; q < S; ++q) v += at[q * SZ];
      at[0] = v;
    }
    __syncthreads();
  }
}

// Element (c, e) of the Gram sum conj(X) Y from the summed real products.
template <int MT>
__device__ __forceinline__ cplx<double> gram_at(const double* sum, int c, int e) {
  const double* u = sum + (2 * c) * 16 * MT + 2 * e;
  const double* v = u + 16 * MT;
  return mk(u[0] + v[1], u[1] - v[0]);
}

// Blocks of the same node follow each other on one XCD (blocks go to the eight XCDs in turn), so
// a node's tensor and products are re-read through that XCD's L2.
__device__ __forceinline__ bool node_item(int idx, int per, int count, int& node, int& sub) {
  node = (idx / per) * 8 + (blockIdx.x & 7);
  sub = idx % per;
  return node < count;
}

// The products of one level: block (node, product, part of the fibres).
template <typename R, typename RS, typename RM, int KS, int MT, bool BP>
__global__ __launch_bounds__(kGemmThreads) void k_gemm_product(ClassView cv, GemmPlan plan, int level, int parts,
                                                               int node0, int count, int chi,
                                                               const cplx<RS>* __restrict__ T, const cplx<RM>* mA,
                                                               const cplx<RM>* mB, BpStatus* st, cplx<R>* ws) {
  const cplx<RM>* msg = mA;
  if constexpr (BP) {
    const int cur = bp_begin(st, cv.sweep);
    if (cur < 0) return;
    msg = cur ? mB : mA;
  }
  const int q0 = plan.first[level], nq = plan.first[level + 1] - q0;
  int node, sub;
  if (!node_item(blockIdx.x >> 3, nq * parts, count, node, sub)) return;
  const int q = q0 + sub / parts, part = sub % parts;
  const int i = node0 + node, bond = plan.bond[q], src = plan.src[q];
  const long S = 2L * ipow(chi, plan.d);
  const int inner = ipow(chi, plan.d - 1 - bond);
  const int F = 2 * ipow(chi, plan.d - 1);
  MatFrag<R, KS, MT> w;
  w.load(msg + (size_t)cv.in_pos[bond * cv.n + i] * chi * chi, chi, chi, chi, 1);
  cplx<R>* base = ws + (size_t)node * plan.products * S;
  cplx<R>* dst = base + q * S;
  const int wave = part * kGemmWaves + (threadIdx.x >> 6), step = parts * kGemmWaves;
  if (src < 0)
    product_tiles<R, RS, KS, MT>(w, T + (size_t)i * S, dst, chi, chi, inner, 0, F, wave, step);
  else
    product_tiles<R, R, KS, MT>(w, base + src * S, dst, chi, chi, inner, 0, F, wave, step);
}

template <typename R, typename RS, int MT>
__device__ __forceinline__ void gram_sources(vec4<R> (&acc)[MT][MT], const GemmPlan& plan, int k, int chi,
                                             const cplx<RS>* Ti, const cplx<R>* base, long S, int f0, int f1,
                                             int wave, int step) {
  const int inner = ipow(chi, plan.d - 1 - k);
  const int bra = plan.bra[k], ket = plan.ket[k];
  if constexpr (sizeof(R) == sizeof(RS)) {
    const cplx<R>* X = bra < 0 ? reinterpret_cast<const cplx<R>*>(Ti) : base + bra * S;
    const cplx<R>* Y = ket < 0 ? reinterpret_cast<const cplx<R>*>(Ti) : base + ket * S;
    gram_range<R, MT>(acc, X, Y, chi, inner, f0, f1, wave, step);
  } else {
    if (bra >= 0)
      gram_range<R, MT>(acc, base + bra * S, base + ket * S, chi, inner, f0, f1, wave, step);
    else if (ket >= 0)
      gram_range<R, MT>(acc, Ti, base + ket * S, chi, inner, f0, f1, wave, step);
    else
      gram_range<R, MT>(acc, Ti, Ti, chi, inner, f0, f1, wave, step);
  }
}

// New messages: blocks of W waves take (node, output) items in turn and keep their distance maxima until the end.
template <typename R, int MT, int W>
__global__ __launch_bounds__(64 * W) void k_gemm_gram_bp(ClassView cv, GemmPlan plan, int node0, int count,
                                                               int chi, const cplx<R>* __restrict__ T, cplx<R>* mA,
                                                               cplx<R>* mB, BpStatus* st, const cplx<R>* ws) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double shred[16];
  double* sum = reinterpret_cast<double*>(smem_raw);
  const int cur = bp_begin(st, cv.sweep);
  if (cur < 0) return;
  const cplx<R>* min = cur ? mB : mA;
  cplx<R>* mout = cur ? mA : mB;
  const int cc = chi * chi, d = plan.d, wave = threadIdx.x >> 6;
  const long S = 2L * ipow(chi, d);
  const int F = 2 * ipow(chi, d - 1);
  double dnum = 0.0, dden = 0.0;
  int node, k;
  for (int idx = blockIdx.x >> 3; node_item(idx, d, count, node, k); idx += gridDim.x >> 3) {
    const int i = node0 + node;
    const long pos = cv.out_pos[k * cv.n + i];
    vec4<R> acc[MT][MT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b) acc[a][b] = vec4<R>{0, 0, 0, 0};
    gram_sources<R, R, MT>(acc, plan, k, chi, T + (size_t)i * S, ws + (size_t)node * plan.products * S, S, 0, F, wave, W);
    sum_tiles<R, MT, W>(sum, acc, 0, wave, 1);
    double tr = 0.0;
    for (int c = 0; c < chi; ++c) tr += gram_at<MT>(sum, c, c).x;
    const double inv = 0.5 / tr;
    for (int o = threadIdx.x; o < cc; o += 64 * W) {
      const int c = o / chi, e = o % chi;
      const cplx<double> a = gram_at<MT>(sum, c, e), b = gram_at<MT>(sum, e, c);
      const cplx<R> v = cast<R>(mk((a.x + b.x) * inv, (a.y - b.y) * inv));
      const cplx<R> old = min[pos * cc + o];
      dnum = fmax(dnum, abs2(cast<double>(v - old)));
      dden = fmax(dden, abs2(cast<double>(v + old)));
      mout[pos * cc + o] = v;
    }
    __syncthreads();
  }
  dnum = block_max(dnum, shred);
  dden = block_max(dden, shred);
  if (threadIdx.x == 0) bp_end(st, cv.sweep, sqrt(dnum), sqrt(dden));
}

// Extended messages: the Grams of the two physical halves (fibres [0, F / 2) and [F / 2, F), each
// over half of the waves), assembled with the bond's ZZ-split gates (backends.py:393-404,519-526).
template <typename RS, int MT, int W>
__global__ __launch_bounds__(64 * W) void k_gemm_gram_ext(ClassView cv, GemmPlan plan, int node0, int count,
                                                                int chi, const cplx<RS>* __restrict__ T,
                                                                cplx<double>* __restrict__ ext,
                                                                const cplx<double>* ws) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int kSide = 16 * MT, kHalf = W / 2, kAt = gram_slots<MT, W / 2>(2) * kSide * kSide;
  double* sum = reinterpret_cast<double*>(smem_raw);
  const int d = plan.d, wave = threadIdx.x >> 6, p = wave / kHalf, n2 = 2 * chi;
  const long S = 2L * ipow(chi, d);
  const int half = ipow(chi, d - 1);
  int node, k;
  for (int idx = blockIdx.x >> 3; node_item(idx, d, count, node, k); idx += gridDim.x >> 3) {
    const int i = node0 + node;
    vec4<double> acc[MT][MT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b) acc[a][b] = vec4<double>{0, 0, 0, 0};
    gram_sources<double, RS, MT>(acc, plan, k, chi, T + (size_t)i * S, ws + (size_t)node * plan.products * S, S,
                                 p * half, (p + 1) * half, wave % kHalf, kHalf);
    sum_tiles<double, MT, kHalf>(sum, acc, p, wave % kHalf, 2);
    const cplx<double>* g = cv.zz + 2 * (size_t)cv.lmbd_pos[k * cv.n + i];
    const cplx<double> gs[2] = {g[0], g[1]};
    const double weight = abs2(gs[0]) + abs2(gs[1]);
    cplx<double> tr = mk(0.0, 0.0);
    for (int c = 0; c < chi; ++c)
      tr = tr + gram_at<MT>(sum, c, c) + gram_at<MT>(sum + kAt, c, c);
    const cplx<double> inv = cinv(scale(tr, weight));
    cplx<double>* out = ext + (size_t)cv.out_pos[k * cv.n + i] * n2 * n2;
    for (int o = threadIdx.x; o < n2 * n2; o += 64 * W) {
      const int row = o / n2, col = o % n2;
      const int s = row / chi, c = row % chi, s2 = col / chi, e = col % chi;
      const cplx<double> g0 = gram_at<MT>(sum, c, e), g1 = gram_at<MT>(sum + kAt, c, e);
      out[o] = conj(gs[s]) * gs[s2] * (((s + s2) & 1) ? g0 - g1 : g0 + g1) * inv;
    }
    __syncthreads();
  }
}

// Fragments of the absorb operand of one physical half: W[c][a] = g0 C[c][a] + z g1 C[chi_in + c][a].
template <int KS, int MT>
__device__ __forceinline__ void absorb_frag(MatFrag<double, KS, MT>& w, const cplx<double>* __restrict__ C, int cols,
                                            int chi_in, int chi_out, cplx<double> g0, cplx<double> gz) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  int al, ri;
  tile_row<double>(r, al, ri);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int a = 8 * mt + al, c = 4 * ks + g;
      cplx<double> v = mk(0.0, 0.0);
      if (a < chi_out && c < chi_in) v = g0 * C[c * cols + a] + gz * C[(chi_in + c) * cols + a];
      w.re[mt][ks] = ri == 0 ? v.x : v.y;
      w.im[mt][ks] = ri == 0 ? -v.y : v.x;
    }
}

// The absorb along bond k: block (node, physical half, part of the half's fibres).
template <typename RS, int KS, int MT>
__global__ __launch_bounds__(kGemmThreads) void k_gemm_absorb(ClassView cv, int k, int parts, int node0, int count,
                                                              int chi_in, int chi_out, const cplx<RS>* __restrict__ src,
                                                              long src_stride, cplx<double>* dst, long dst_stride,
                                                              const cplx<double>* __restrict__ canon, int cols,
                                                              double zz_time) {
  int node, sub;
  if (!node_item(blockIdx.x >> 3, 2 * parts, count, node, sub)) return;
  const int p = sub / parts, part = sub % parts, i = node0 + node;
  const int inner = ipow(chi_in, cv.d - 1 - k), half = ipow(chi_out, k) * inner;
  cplx<double> g0, g1;
  if (cv.zz) {
    const cplx<double>* g = cv.zz + 2 * (size_t)cv.lmbd_pos[k * cv.n + i];
    g0 = g[0];
    g1 = g[1];
  } else {
    zz_split(cv.J[k * cv.n + i] * zz_time, g0, g1);
  }
  MatFrag<double, KS, MT> w;
  absorb_frag<KS, MT>(w, canon + (size_t)cv.in_pos[k * cv.n + i] * 2 * chi_in * cols, cols, chi_in, chi_out, g0,
                      p ? mk(-g1.x, -g1.y) : g1);
  product_tiles<double, RS, KS, MT>(w, src + (size_t)node * src_stride, dst + (size_t)node * dst_stride, chi_in,
                                    chi_out, inner, p * half, (p + 1) * half,
                                    part * kGemmWaves + (threadIdx.x >> 6), parts * kGemmWaves);
}

constexpr int kGaugeThreads = 512;

// Z and X gates, symmetric gauge, node normalisation and message re-initialisation of absorbed tensors
// (state.py:142-156, 219-227), a block per node: the norm in a first pass over the tensor, the scaled
// values in a second (a node's FP64 tensor is larger than the registers, and L2 still has it).  LDS: the
// products of sqrt(lambda) over the last two bonds, then sqrt(lambda) of every bond.
template <typename R>
__global__ __launch_bounds__(kGaugeThreads) void k_gemm_gauge(ClassView cv, int node0, int chi,
                                                              const cplx<double>* __restrict__ X, long stride,
                                                              cplx<R>* __restrict__ Tout, int flags, double z_time,
                                                              double x_time, const double* __restrict__ lmbd,
                                                              int lstride, cplx<R>* msgs_init) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double shred[16];
  double* low = reinterpret_cast<double*>(smem_raw);
  const int d = cv.d, n = cv.n, t = threadIdx.x, i = node0 + blockIdx.x, cc = chi * chi;
  double* root = low + cc;
  const int A = ipow(chi, d);
  const cplx<double>* x0 = X + (size_t)blockIdx.x * stride;
  const cplx<double>* x1 = x0 + A;
  const bool gates = flags & kGates, gauge = flags & kGauge;
  if (gauge) {
    for (int q = t; q < d * chi; q += kGaugeThreads)
      root[q] = sqrt(lmbd[(size_t)cv.lmbd_pos[(q / chi) * n + i] * lstride + q % chi]);
    __syncthreads();
    for (int q = t; q < cc; q += kGaugeThreads) low[q] = root[(d - 2) * chi + q / chi] * root[(d - 1) * chi + q % chi];
    __syncthreads();
  }
  const double phi = gates ? cv.h[i] * z_time : 0.0;
  const double cz = cos(phi), sz = sin(phi), cx = cos(x_time), sx = sin(x_time);
  const cplx<double> f0 = mk(cz, -sz), f1 = mk(cz, sz);
  auto values = [&](int a, cplx<double>& y0, cplx<double>& y1) {
    y0 = x0[a];
    y1 = x1[a];
    if (gates) {
      const cplx<double> t0 = y0 * f0, t1 = y1 * f1;
      // (cos x) t - i (sin x) X t
      y0 = mk(cx * t0.x + sx * t1.y, cx * t0.y - sx * t1.x);
      y1 = mk(cx * t1.x + sx * t0.y, cx * t1.y - sx * t0.x);
    }
    if (gauge) {
      int hi = a / cc;
      double f = low[a - hi * cc];
      for (int k = d - 3; k >= 0; --k) {
        f *= root[k * chi + hi % chi];
        hi /= chi;
      }
      y0 = scale(y0, f);
      y1 = scale(y1, f);
    }
  };
  double inv = 1.0;
  if (gauge) {
    double ss = 0.0;
    for (int a = t; a < A; a += kGaugeThreads) {
      cplx<double> y0, y1;
      values(a, y0, y1);
      ss += abs2(y0) + abs2(y1);
    }
    inv = 1.0 / sqrt(block_sum(ss, shred));
  }
  cplx<R>* out = Tout + (size_t)i * 2 * A;
  for (int a = t; a < A; a += kGaugeThreads) {
    cplx<double> y0, y1;
    values(a, y0, y1);
    out[a] = cast<R>(scale(y0, inv));
    out[A + a] = cast<R>(scale(y1, inv));
  }
  if (!gauge) return;
  for (int k = 0; k < d; ++k) {
    const double* lam = lmbd + (size_t)cv.lmbd_pos[k * n + i] * lstride;
    double tr = 0.0;
    for (int a = 0; a < chi; ++a) tr += lam[a];
    const size_t pos = cv.in_pos[k * n + i];
    for (int o = t; o < cc; o += kGaugeThreads) {
      const int a = o / chi, b = o % chi;
      msgs_init[pos * cc + o] = mk<R>(a == b ? (R)(lam[a] / tr) : (R)0, (R)0);
    }
  }
}

// Calls f.template operator()<KS, MT>() with the tile counts of bond dimension chi.
template <typename F>
void by_chi(int chi, F&& f) {
  switch ((chi + 3) / 4) {
    case 1: f.template operator()<1, 1>(); break;
    case 2: f.template operator()<2, 1>(); break;
    case 3: f.template operator()<3, 2>(); break;
    case 4: f.template operator()<4, 2>(); break;
    case 5: f.template operator()<5, 3>(); break;
    case 6: f.template operator()<6, 3>(); break;
    case 7: f.template operator()<7, 4>(); break;
    default: f.template operator()<8, 4>(); break;
  }
}

// rho[p, q] = sum_a X[p, a] conj(Z[q, a]), trace one, and the Bloch vector by qubit id: a block per node, X the last
// product of the first chain and Z of the second (the node tensor for an empty one).  Sums in FP64.
template <typename R>
__global__ __launch_bounds__(kGemmThreads) void k_gemm_density(ClassView cv, int node0, int chi, int x_at, int z_at,
                                                               int products, const cplx<R>* __restrict__ T,
                                                               const cplx<R>* __restrict__ ws, double* rho_out,
                                                               double* bloch_out) {
  __shared__ double part[8][kGemmWaves];
  const int i = node0 + blockIdx.x, t = threadIdx.x;
  const long A = ipow(chi, cv.d), S = 2 * A;
  const cplx<R>* base = ws + (size_t)blockIdx.x * products * S;
  const cplx<R>* X = x_at < 0 ? T + (size_t)i * S : base + x_at * S;
  const cplx<R>* Z = z_at < 0 ? T + (size_t)i * S : base + z_at * S;
  cplx<double> r[4] = {};
#pragma unroll 4
  for (long a = t; a < A; a += kGemmThreads) {
    const cplx<double> x0 = cast<double>(X[a]), x1 = cast<double>(X[A + a]);
    const cplx<double> z0 = cast<double>(Z[a]), z1 = cast<double>(Z[A + a]);
    cfma_cj(r[0], z0, x0);
    cfma_cj(r[1], z1, x0);
    cfma_cj(r[2], z0, x1);
    cfma_cj(r[3], z1, x1);
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    double v = q & 1 ? r[q >> 1].y : r[q >> 1].x;
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((t & 63) == 0) part[q][t >> 6] = v;
  }
  __syncthreads();
  if (t == 0) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      v[q] = part[q][0];
#pragma unroll
      for (int w = 1; w < kGemmWaves; ++w) v[q] += part[q][w];
    }
    const cplx<double> inv = cinv(mk(v[0] + v[6], v[1] + v[7]));
    const cplx<double> r00 = mk(v[0], v[1]) * inv, r01 = mk(v[2], v[3]) * inv;
    const cplx<double> r10 = mk(v[4], v[5]) * inv, r11 = mk(v[6], v[7]) * inv;
    const long id = cv.node_ids[i];
    double* ro = rho_out + id * 8;
    ro[0] = r00.x; ro[1] = r00.y; ro[2] = r01.x; ro[3] = r01.y;
    ro[4] = r10.x; ro[5] = r10.y; ro[6] = r11.x; ro[7] = r11.y;
    double* bo = bloch_out + id * 3;
    bo[0] = r01.x + r10.x;
    bo[1] = r10.y - r01.y;
    bo[2] = r00.x - r11.x;
  }
}

// Parts of a node's fibres: about eight tiles a wave to pay for the message fragments, fewer where
// the launch would not give every CU four blocks.
int product_parts(int count, int products, long fibres) {
  const long tiles = (fibres + 15) / 16;
  const long most = std::max<long>(1, (tiles + kGemmWaves - 1) / kGemmWaves);
  const long least = std::max<long>(1, (tiles + 8 * kGemmWaves - 1) / (8 * kGemmWaves));
  const long want = (1024 + (long)count * products - 1) / ((long)count * products);
  return (int)std::min(most, std::max(least, want));
}

int padded8(int n) { return (n + 7) / 8 * 8; }

template <typename R, typename RS, typename RM, bool BP>
void launch_products(const ClassView& cv, const GemmPlan& plan, int chi, int node0, int count, const cplx<RS>* T,
                     const cplx<RM>* mA, const cplx<RM>* mB, BpStatus* st, cplx<R>* ws, hipStream_t s) {
  const long fibres = 2L * ipow(chi, plan.d - 1);
  for (int level = 0; level < plan.levels; ++level) {
    const int nq = plan.first[level + 1] - plan.first[level];
    const int parts = product_parts(count, nq, fibres);
    const dim3 grid((unsigned)(padded8(count) * nq * parts));
    by_chi(chi, [&]<int KS, int MT>() {
      hipLaunchKernelGGL((k_gemm_product<R, RS, RM, KS, MT, BP>), grid, dim3(kGemmThreads), 0, s, cv, plan, level,
                         parts, node0, count, chi, T, mA, mB, st, ws);
    });
  }
}

// The same with independent counts for the summed index (chi_in) and the rows (chi_out).
template <int KS, typename F>
void by_rows(int rows, F&& f) {
  switch ((rows + 7) / 8) {
    case 1: f.template operator()<KS, 1>(); break;
    case 2: f.template operator()<KS, 2>(); break;
    case 3: f.template operator()<KS, 3>(); break;
    default: f.template operator()<KS, 4>(); break;
  }
}
template <typename F>
void by_chi_pair(int chi_in, int chi_out, F&& f) {
  switch ((chi_in + 3) / 4) {
    case 1: by_rows<1>(chi_out, f); break;
    case 2: by_rows<2>(chi_out, f); break;
    case 3: by_rows<3>(chi_out, f); break;
    case 4: by_rows<4>(chi_out, f); break;
    case 5: by_rows<5>(chi_out, f); break;
    case 6: by_rows<6>(chi_out, f); break;
    case 7: by_rows<7>(chi_out, f); break;
    default: by_rows<8>(chi_out, f); break;
  }
}

// Waves per Gram: with few (node, output) items a Gram of four waves leaves most of the chip waiting for the loads of
// its long fibre loop, so up to sixteen share it, to six waves a SIMD over the chip, as long as each has a group of
// 16 fibres.  (Wider tiles need the registers of eight waves a CU, the widest FP64 ones of four.)
template <typename R, int MT, typename F>
void by_waves(int items, long fibres, F&& f) {
  const long most = std::min<long>(6144 / std::max(items, 1), (fibres + 15) / 16);
  constexpr int kMost = MT <= 2 ? 16 : sizeof(R) == 8 && MT == 4 ? 4 : 8;
  if (kMost >= 16 && most >= 16) f.template operator()<(kMost >= 16 ? 16 : 4)>();
  else if (kMost >= 8 && most >= 8) f.template operator()<(kMost >= 8 ? 8 : 4)>();
  else f.template operator()<4>();
}

constexpr int kGramBlocks = 2048;   // eight blocks a CU; each keeps its maxima over its items

}  // namespace

GemmPlan gemm_plan(int d) {
  GemmPlan p{};
  p.d = d;
  // index sets of the products made so far; a product of a set multiplies one more bond onto the
  // product of the set without it
  int sets[kGemmMaxProducts], level[kGemmMaxProducts], n = 0;
  auto find = [&](int set) {
    for (int q = 0; q < n; ++q)
      if (sets[q] == set) return q;
    return -1;
  };
  struct Item {
    int set, src, bond, level;
  };
  auto make = [&](auto&& self, int set) -> int {
    if (set == 0) return -1;
    const int have = find(set);
    if (have >= 0) return have;
    int from = -1, bond = -1;
    for (int b = 0; b < d && bond < 0; ++b)
      if ((set >> b & 1) && (set & (set - 1)) && find(set & ~(1 << b)) >= 0) bond = b;
    if (bond < 0)
      for (int b = d - 1; b >= 0 && bond < 0; --b)
        if (set >> b & 1) bond = b;
    from = self(self, set & ~(1 << bond));
    sets[n] = set;
    level[n] = from < 0 ? 0 : level[from] + 1;
    p.src[n] = (int8_t)from;
    p.bond[n] = (int8_t)bond;
    return n++;
  };
  const int all = (1 << d) - 1;
  const int low = (1 << (d / 2)) - 1, high = all & ~low;
  for (int k = 0; k < d; ++k) {
    int bra, ket;
    if (d <= 3) {   // one message on each side
      const int rest = all & ~(1 << k);
      ket = rest & -rest;
      bra = rest & ~ket;
    } else {        // the other half whole, this half without k
      ket = (low >> k & 1) ? high : low;
      bra = all & ~ket & ~(1 << k);
    }
    p.ket[k] = (int8_t)make(make, ket);
    p.bra[k] = (int8_t)make(make, bra);
  }
  p.products = n;
  // order by level, renumbering the sources
  int order[kGemmMaxProducts], place[kGemmMaxProducts], m = 0;
  for (int l = 0; m < n; ++l) {
    p.first[l] = m;
    for (int q = 0; q < n; ++q)
      if (level[q] == l) {
        place[q] = m;
        order[m++] = q;
      }
    p.levels = l + 1;
    p.first[l + 1] = m;
  }
  GemmPlan out = p;
  for (int x = 0; x < n; ++x) {
    out.src[x] = p.src[order[x]] < 0 ? (int8_t)-1 : (int8_t)place[p.src[order[x]]];
    out.bond[x] = p.bond[order[x]];
  }
  for (int k = 0; k < d; ++k) {
    out.bra[k] = p.bra[k] < 0 ? (int8_t)-1 : (int8_t)place[p.bra[k]];
    out.ket[k] = p.ket[k] < 0 ? (int8_t)-1 : (int8_t)place[p.ket[k]];
  }
  return out;
}

template <typename R>
void gemm_bp(ClassView cv, int chi, const cplx<R>* T, cplx<R>* mA, cplx<R>* mB, BpStatus* st, void* ws, int chunk,
             hipStream_t s) {
  const GemmPlan plan = gemm_plan(cv.d);
  cplx<R>* w = reinterpret_cast<cplx<R>*>(ws);
  for (int node0 = 0; node0 < cv.n; node0 += chunk) {
    const int count = std::min(chunk, cv.n - node0);
    launch_products<R, R, R, true>(cv, plan, chi, node0, count, T, mA, mB, st, w, s);
    const int items = padded8(count) * cv.d;
    by_chi(chi, [&]<int KS, int MT>() {
      by_waves<R, MT>(items, 2L * ipow(chi, cv.d - 1), [&]<int W>() {
        hipLaunchKernelGGL((k_gemm_gram_bp<R, MT, W>), dim3(std::min(items, kGramBlocks)), dim3(64 * W),
                           (sizeof(double) * 256 * MT * MT * gram_slots<MT, W>(1)), s, cv, plan, node0, count, chi, T, mA,
                           mB, st, w);
      });
    });
  }
}

template <typename R>
void gemm_ext(ClassView cv, int chi, const cplx<R>* T, const cplx<R>* msgs, cplx<double>* ext, void* ws, int chunk,
              hipStream_t s) {
  const GemmPlan plan = gemm_plan(cv.d);
  cplx<double>* w = reinterpret_cast<cplx<double>*>(ws);
  for (int node0 = 0; node0 < cv.n; node0 += chunk) {
    const int count = std::min(chunk, cv.n - node0);
    launch_products<double, R, R, false>(cv, plan, chi, node0, count, T, msgs, msgs, nullptr, w, s);
    const int items = padded8(count) * cv.d;
    by_chi(chi, [&]<int KS, int MT>() {
      by_waves<double, MT>(items, 2L * ipow(chi, cv.d - 1), [&]<int W>() {
        hipLaunchKernelGGL((k_gemm_gram_ext<R, MT, W>), dim3(std::min(items, kGramBlocks)), dim3(64 * W),
                           (2 * sizeof(double) * 256 * MT * MT * gram_slots<MT, W / 2>(2)), s, cv, plan, node0, count, chi,
                           T, ext, w);
      });
    });
  }
}

template <typename R>
void gemm_local(ClassView cv, int chi_in, int chi_out, const cplx<R>* Tin, cplx<R>* Tout, const cplx<double>* canon,
                int canon_cols, double zz_time, int flags, double z_time, double x_time, const double* lmbd,
                int lstride, cplx<R>* msgs_init, void* ws, int chunk, hipStream_t s) {
  const int d = cv.d, most = std::max(chi_in, chi_out);
  const long S_in = 2L * ipow(chi_in, d), S = 2L * ipow(most, d);
  cplx<double>* buf[2] = {reinterpret_cast<cplx<double>*>(ws), reinterpret_cast<cplx<double>*>(ws) + chunk * S};
  for (int node0 = 0; node0 < cv.n; node0 += chunk) {
    const int count = std::min(chunk, cv.n - node0);
    for (int k = 0; k < d; ++k) {
      const long half = (long)ipow(chi_out, k) * ipow(chi_in, d - 1 - k);
      const int parts = product_parts(count, 2, half);
      const dim3 grid((unsigned)(padded8(count) * 2 * parts));
      by_chi_pair(chi_in, chi_out, [&]<int KS, int MT>() {
        if (k == 0)
          hipLaunchKernelGGL((k_gemm_absorb<R, KS, MT>), grid, dim3(kGemmThreads), 0, s, cv, k, parts, node0, count,
                             chi_in, chi_out, Tin + node0 * S_in, S_in, buf[0], S, canon, canon_cols, zz_time);
        else
          hipLaunchKernelGGL((k_gemm_absorb<double, KS, MT>), grid, dim3(kGemmThreads), 0, s, cv, k, parts, node0,
                             count, chi_in, chi_out, buf[(k + 1) & 1], S, buf[k & 1], S, canon, canon_cols, zz_time);
      });
    }
    const size_t lds = sizeof(double) * (chi_out * chi_out + d * chi_out);
    hipLaunchKernelGGL((k_gemm_gauge<R>), dim3(count), dim3(kGaugeThreads), lds, s, cv, node0, chi_out,
                       buf[(d + 1) & 1], S, Tout, flags, z_time, x_time, lmbd, lstride, msgs_init);
  }
}

template <typename R>
void gemm_density(ClassView cv, int chi, const cplx<R>* T, const cplx<R>* msgs, double* rho, double* bloch, void* ws,
                  int chunk, hipStream_t s) {
  // two chains of products, level by level: the upper half of the bonds from the last one down, and the lower half
  const int d = cv.d, low = d / 2;
  GemmPlan plan{};
  plan.d = d;
  int last_low = -1, last_high = -1;
  for (int l = 0; l < d - low; ++l) {
    plan.first[l] = plan.products;
    plan.src[plan.products] = (int8_t)last_high;
    plan.bond[plan.products] = (int8_t)(d - 1 - l);
    last_high = plan.products++;
    if (l < low) {
      plan.src[plan.products] = (int8_t)last_low;
      plan.bond[plan.products] = (int8_t)(low - 1 - l);
      last_low = plan.products++;
    }
    plan.levels = l + 1;
    plan.first[l + 1] = plan.products;
  }
  cplx<R>* w = reinterpret_cast<cplx<R>*>(ws);
  for (int node0 = 0; node0 < cv.n; node0 += chunk) {
    const int count = std::min(chunk, cv.n - node0);
    launch_products<R, R, R, false>(cv, plan, chi, node0, count, T, msgs, msgs, nullptr, w, s);
    hipLaunchKernelGGL((k_gemm_density<R>), dim3(count), dim3(kGemmThreads), 0, s, cv, node0, chi, last_high, last_low,
                       plan.products, T, w, rho, bloch);
  }
}

template void gemm_density<float>(ClassView, int, const cplx<float>*, const cplx<float>*, double*, double*, void*, int,
                                  hipStream_t);
template void gemm_density<double>(ClassView, int, const cplx<double>*, const cplx<double>*, double*, double*, void*,
                                   int, hipStream_t);
template void gemm_local<float>(ClassView, int, int, const cplx<float>*, cplx<float>*, const cplx<double>*, int, double,
                                int, double, double, const double*, int, cplx<float>*, void*, int, hipStream_t);
template void gemm_local<double>(ClassView, int, int, const cplx<double>*, cplx<double>*, const cplx<double>*, int,
                                 double, int, double, double, const double*, int, cplx<double>*, void*, int,
                                 hipStream_t);
template void gemm_bp<float>(ClassView, int, const cplx<float>*, cplx<float>*, cplx<float>*, BpStatus*, void*, int,
                             hipStream_t);
template void gemm_bp<double>(ClassView, int, const cplx<double>*, cplx<double>*, cplx<double>*, BpStatus*, void*,
                              int, hipStream_t);
template void gemm_ext<float>(ClassView, int, const cplx<float>*, const cplx<float>*, cplx<double>*, void*, int,
                              hipStream_t);
template void gemm_ext<double>(ClassView, int, const cplx<double>*, const cplx<double>*, cplx<double>*, void*, int,
                               hipStream_t);

}  // namespace bqa
