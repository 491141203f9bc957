// kernels_coarse16.hpp -- the V-cycle's levels 16^3, 8^3 and 4^3 in one workgroup, laid out for latency.
//
// cw_cycle (kernels_coarse.hpp) runs these levels point by point from index arithmetic and memory:
// some 2-3 us per colour phase, 140 to 7000 barrier-separated phases per cycle.  A phase's own
// arithmetic is 0.2 us, so everything that can be prepared once per visit to a level is held on
// chip by the thread that needs it:
//  - 4^3: one point per lane of wavefront 0, no barriers (64 points);
//  - 8^3: one point per thread, wavefront w owning colour class w;
//  - 16^3: one 2x2x2 cell per thread, its 8 points one of each class.
// The iterate is in LDS (sub-lattice layout).  Coefficients are in registers: the face averages, the
// diagonal and its reciprocal and the cross-term factors of the 19-point operator, or the 27 Galerkin
// coefficients.  Those of the 16^3 level that do not fit (registers: 256 per lane) are in LDS (FP64
// 19-point: the three cross-term fields; FP32 27-point: the eight corners) or, FP64 27-point (0.9 MB),
// streamed from the L2 one colour ahead.
// Colours c and c ^ 7 are not coupled by the 19-point operator (it has no corner offsets), so the fourth
// and fifth colour of a sweep, and the last of a sweep with the first of the next, share a phase:
// 6 phases per sweep instead of 8, the same values.
// The per-point arithmetic, the order of every sum and the schedule are cw_cycle's, so results are
// bit-identical.  Measured (MI355X), per cycle: FP32 reference schedule 1124 -> 246 us at NG = 64 and
// 5.87 -> 1.22 ms at NG = 512 (0.24 us per phase); FP64 Krylov schedule with Galerkin levels 408 -> 126 us;
// in a batch, one workgroup per grid, 614 -> 128 us.
#pragma once
#include <limits>

#include "kernels_coarse.hpp"

namespace mmh {

// a / b for y = 1 / b rounded to nearest: two residual corrections give the correctly rounded
// quotient (P. Markstein, IBM J. Res. Dev. 34, 1990), 5 dependent operations where the compiler's
// division takes 11; div_fixup gives zeros, infinities and NaN their IEEE results.  It is exact while y, the
// quotient and the residuals stay normal numbers: in FP32 |a| from 2^-100 (the residual is a multiple of 2^-47
// |a|, and 2^-149 the smallest step), |b| and |q| from 2^-126, |b| up to 2^126.  The bounds kept here, |a| from
// 2^-80 and |b| up to 2^44 (FP64 2^-600, 2^400), make |q| large enough too.  A Range holds the
// smallest dividend but zero of a thread, in two integer operations a quotient; where it or a divisor is out
// of bounds, or the iterate is not finite (a quotient that overflows leaves it so), the cycle is run
// again with plain divisions.  A test on every quotient that chose the division there cost 9 % of
// the FP32 cycle, flags of three comparisons 6 %.
template <bool PLAIN> struct Range {
  static constexpr bool plain = PLAIN;  // the cycle run again: plain divisions
  unsigned key = ~0u;  // of the smallest dividend: its bits without the sign, less one
  static __device__ __forceinline__ unsigned key_of(float a) { return (__float_as_uint(a) << 1) - 1u; }
  static __device__ __forceinline__ unsigned key_of(double a) {  // of the high word; one more below it if the low is set
    return ((unsigned)__double2hiint(a) << 1) + min((unsigned)__double2loint(a), 1u) - 1u;
  }
  template <class T> __device__ __forceinline__ void dividend(T a) { key = min(key, key_of(a)); }
  __device__ __forceinline__ void divisor(float b) {
    if (!(fabs(b) >= 0x1p-126f && fabs(b) <= 0x1p44f)) key = 0u;
  }
  __device__ __forceinline__ void divisor(double b) {
    if (!(fabs(b) >= 0x1p-1022 && fabs(b) <= 0x1p400)) key = 0u;
  }
  template <class T> __device__ __forceinline__ void iterate(T u) {
    if constexpr (PLAIN) return;
    if (!(fabs(u) <= std::numeric_limits<T>::max())) key = 0u;
  }
  template <class T> __device__ __forceinline__ bool out() const { return key < key_of(sizeof(T) == 4 ? T(0x1p-80) : T(0x1p-600)); }
};
__device__ __forceinline__ float corrected(float a, float b, float y, float q) {
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
}
__device__ __forceinline__ double corrected(double a, double b, double y, double q) {
  return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}
__device__ __forceinline__ float fixup(float q, float b, float a) { return __builtin_amdgcn_div_fixupf(q, b, a); }
__device__ __forceinline__ double fixup(double q, double b, double a) { return __builtin_amdgcn_div_fixup(q, b, a); }
template <class T, class R> __device__ __forceinline__ T recip(T b, R& off) {
  if constexpr (R::plain) return T(0);
  off.divisor(b);
  return T(1) / b;
}
template <class T, class R> __device__ __forceinline__ T quotient(T a, T b, T y, R& off) {
  if constexpr (R::plain) return a / b;
  off.dividend(a);
  T q = a * y;
  q = corrected(a, b, y, q);
  q = corrected(a, b, y, q);
  return fixup(q, b, a);
}

// Offsets of the 18 neighbours of the 19-point operator in the order of its terms: faces (+-x, +-y, +-z),
// then the corners of the cross terms (x, y), (y, z), (x, z).
constexpr int NB19[18][3] = {{1, 0, 0},  {-1, 0, 0},  {0, 1, 0},  {0, -1, 0}, {0, 0, 1},  {0, 0, -1},
                             {1, 1, 0},  {-1, 1, 0},  {1, -1, 0}, {-1, -1, 0}, {0, 1, 1}, {0, -1, 1},
                             {0, 1, -1}, {0, -1, -1}, {1, 0, 1},  {-1, 0, 1}, {1, 0, -1}, {-1, 0, -1}};
// Neighbours (of NB19) whose G2, G5, G3 multiply the 12 cross differences, in the terms' order, with
// the G field (0-based component).
constexpr int XG19[12][2] = {{2, 1}, {3, 1}, {0, 1}, {1, 1}, {4, 4}, {5, 4}, {2, 4}, {3, 4}, {4, 2}, {5, 2}, {0, 2}, {1, 2}};

// Faces b11p, b11m, b22p, b22m, b33p, b33m, then the diagonal, as stencil19 forms them; o: index of the
// point, nb: of its neighbours.
template <class T> __device__ __forceinline__ void faces19(T (&w)[7], const T* G, int n3, int o, const int (&nb)[18]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const T* g = G + (d == 0 ? 0 : d == 1 ? 3 : 5) * n3;
    w[2 * d] = (g[nb[2 * d]] + g[o]) / T(2);
    w[2 * d + 1] = (g[nb[2 * d + 1]] + g[o]) / T(2);
  }
  w[6] = -(w[0] + w[1] + w[2] + w[3] + w[4] + w[5]);
}
// t1 and t2 of stencil19 from the neighbours' values and the 12 cross factors.
template <class T>
__device__ __forceinline__ void terms19(T& t1, T& t2, const T (&w)[7], const T (&x)[12], const T (&p)[18]) {
  t1 = (w[0] * p[0] + w[1] * p[1] + w[2] * p[2] + w[3] * p[3] + w[4] * p[4] + w[5] * p[5]);
  t2 = ((p[6] - p[7]) * x[0]
      - (p[8] - p[9]) * x[1]
      + (p[6] - p[8]) * x[2]
      - (p[7] - p[9]) * x[3]
      + (p[10] - p[11]) * x[4]
      - (p[12] - p[13]) * x[5]
      + (p[10] - p[12]) * x[6]
      - (p[11] - p[13]) * x[7]
      + (p[14] - p[15]) * x[8]
      - (p[16] - p[17]) * x[9]
      + (p[14] - p[16]) * x[10]
      - (p[15] - p[17]) * x[11]) / T(4);
}

// Colour phases of ns sweeps (reversed order when rev): f(mask) updates the classes whose bit is set
// (class bit = i&1 | (j&1)<<1 | (k&1)<<2), a barrier or its like included.
template <class F> __device__ __forceinline__ void phases19(int ns, bool rev, F&& f) {
  if (ns < 1) return;
  const unsigned m3 = 1u << 3 | 1u << 4;
  if (!rev) {
    f(1u << 0);
    for (int s = 0; s < ns; ++s) {
      f(1u << 2); f(1u << 1); f(m3); f(1u << 6); f(1u << 5);
      f(s + 1 < ns ? 1u << 7 | 1u << 0 : 1u << 7);
    }
  } else {
    f(1u << 7);
    for (int s = 0; s < ns; ++s) {
      f(1u << 5); f(1u << 6); f(m3); f(1u << 1); f(1u << 2);
      f(s + 1 < ns ? 1u << 7 | 1u << 0 : 1u << 0);
    }
  }
}
template <class F> __device__ __forceinline__ void phases27(int ns, bool rev, F&& f) {
  for (int s = 0; s < ns; ++s) {
    if (!rev) {
      f(1u << 0); f(1u << 2); f(1u << 1); f(1u << 3); f(1u << 4); f(1u << 6); f(1u << 5); f(1u << 7);
    } else {
      f(1u << 7); f(1u << 5); f(1u << 6); f(1u << 4); f(1u << 3); f(1u << 1); f(1u << 2); f(1u << 0);
    }
  }
}

// ---- one point per thread (4^3, 8^3) ---------------------------------------------------------------
// The point p (sub-lattice index) of an N^3 level, its neighbours' indices and its coefficients.
template <class T, int N, bool GAL> struct PointOp;
template <class T, int N> struct PointOp<T, N, false> {
  int nb[18];
  T w[7], x[12], y, b, b2;
  T di2;
  template <class R> __device__ __forceinline__ void load(const T* G, const T* rhs, int p, T dx, R& off) {
    int i, j, k;
    point_of<1, true>(p, N, i, j, k);
#pragma unroll
    for (int e = 0; e < 18; ++e)
      nb[e] = (int)lx<1, true>((i + NB19[e][0]) & (N - 1), (j + NB19[e][1]) & (N - 1), (k + NB19[e][2]) & (N - 1), N);
    faces19<T>(w, G, N * N * N, p, nb);
#pragma unroll
    for (int e = 0; e < 12; ++e) x[e] = G[XG19[e][1] * N * N * N + nb[XG19[e][0]]];
    y = recip(w[6], off);
    b = rhs[p];
    b2 = b * (dx * dx);
    di2 = T(1) / (dx * dx);
  }
  template <class R> __device__ __forceinline__ T update(const T* u, R& off) const {
    T q[18], t1, t2;
#pragma unroll
    for (int e = 0; e < 18; ++e) q[e] = u[nb[e]];
    terms19<T>(t1, t2, w, x, q);
    return quotient(b2 - t1 - t2, w[6], y, off);
  }
  __device__ __forceinline__ T resid(const T* u, int p) const {
    T q[18], t1, t2;
#pragma unroll
    for (int e = 0; e < 18; ++e) q[e] = u[nb[e]];
    terms19<T>(t1, t2, w, x, q);
    return b - (t1 + t2 + w[6] * u[p]) * di2;
  }
  template <class F> static __device__ __forceinline__ void phases(int ns, bool rev, F&& f) { phases19(ns, rev, f); }
};
template <class T, int N> struct PointOp<T, N, true> {
  int nb[27];
  T a[27], y, b;
  template <class R> __device__ __forceinline__ void load(const T* A, const T* rhs, int p, T, R& off) {
    int i, j, k;
    point_of<1, true>(p, N, i, j, k);
#pragma unroll
    for (int e = 0; e < 27; ++e) {
      nb[e] = (int)lx<1, true>((i + e % 3 - 1) & (N - 1), (j + e / 3 % 3 - 1) & (N - 1), (k + e / 9 - 1) & (N - 1), N);
      a[e] = A[e * N * N * N + p];
    }
    y = recip(a[13], off);
    b = rhs[p];
  }
  __device__ __forceinline__ T offsum(const T* u) const {
    T q[27], s = T(0);
#pragma unroll
    for (int e = 0; e < 27; ++e)
      if (e != 13) q[e] = u[nb[e]];
#pragma unroll
    for (int e = 0; e < 27; ++e)
      if (e != 13) s = s + a[e] * q[e];
    return s;
  }
  template <class R> __device__ __forceinline__ T update(const T* u, R& off) const { return quotient(b - offsum(u), a[13], y, off); }
  __device__ __forceinline__ T resid(const T* u, int p) const { return b - (offsum(u) + a[13] * u[p]); }
  template <class F> static __device__ __forceinline__ void phases(int ns, bool rev, F&& f) { phases27(ns, rev, f); }
};

// Sum over lanes of the halving tree's last levels (h = 32 .. 1), in lane 0.
__device__ __forceinline__ double tree64(double a) {
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) a = a + __shfl_down(a, h);
  return a;
}
__device__ __forceinline__ double max64(double a) {
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) a = dmax(a, __shfl_xor(a, h));
  return a;
}

// Scratch of the workgroup's sums and maxima.
struct Cc16Scratch {
  double s[CW];
  double v[CW / 64];
  int off;  // a quotient was out of range (Range)
};

// max over the workgroup, in every thread.
__device__ __forceinline__ double cc_max(double a, Cc16Scratch& S) {
  a = max64(a);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) S.v[threadIdx.x >> 6] = a;
  __syncthreads();
  double m = S.v[0];
#pragma unroll
  for (int v = 1; v < CW / 64; ++v) m = dmax(m, S.v[v]);
  return m;
}

// reduce()'s sum (op 0) of u[0..N^3) in LDS, in every thread: blocks of RB*RPT values, thread t of a block
// adds values t, t + RB, ... in order, then the halving tree; the block sums once more.
template <class T, int N> __device__ __forceinline__ double cc_sum(const T* u, Cc16Scratch& S) {
  constexpr int N3 = N * N * N, NB = (N3 + RB * RPT - 1) / (RB * RPT);
  static_assert(NB <= 2, "two blocks at most");
  const int t = threadIdx.x & (RB - 1), g = threadIdx.x / RB;
  double a = 0.0;
  if (g < NB) {
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const int q = g * RB * RPT + m * RB + t;
      if (q < N3) a = a + (double)u[q];
    }
  }
  __syncthreads();
  S.s[threadIdx.x] = a;
  __syncthreads();
  if (t < 128) S.s[threadIdx.x] = a = a + S.s[threadIdx.x + 128];
  __syncthreads();
  if (t < 64) {
    a = tree64(a + S.s[threadIdx.x + 64]);
    if (t == 0) S.v[g] = a;
  }
  __syncthreads();
  return NB == 1 ? S.v[0] : (0.0 + S.v[0]) + (0.0 + S.v[1]);
}

// zerosum or the guard's szero (cw_zerosum) of the level in LDS.
template <class T, int N>
__device__ __forceinline__ void cc_zerosum(T* u, double* scal, int* guard, int mode, double r1, double re, Cc16Scratch& S) {
  const double sum = cc_sum<T, N>(u, S);
  bool g = false;
  if (mode == 1) g = (T)re > (T)r1;
  else if (mode == 2) g = ((T)re > (T)r1 * T(1.001) && (T)r1 > T(1.e-5));
  if (threadIdx.x == 0) {
    scal[2] = sum;
    if (guard) *guard = g ? 1 : 0;
  }
  const double m = sum / (double)(N * N * N);
  for (int p = threadIdx.x; p < N * N * N; p += CW) u[p] = g ? T(0) : (T)((double)u[p] - m);
  __syncthreads();
}

// The 4^3 level (cw_bottom), by wavefront 0: u4 holds the result.  Its mean's tree has one block of
// which 64 threads hold a value, so the levels above h = 32 add zeros.
template <class T, bool GAL, bool PLAIN>
__device__ __forceinline__ void cc_bottom(T* u4, const T* rhs4, const T* op, T dx, int nc, bool rev, double* scal, int* guard,
                                          int ref, int mode, Cc16Scratch& S) {
  if (threadIdx.x >= 64) return;
  const int p = threadIdx.x;
  Range<PLAIN> off;
  PointOp<T, 4, GAL> P;
  P.load(op, rhs4, p, dx, off);
  auto phase = [&](unsigned mask) {
    if ((mask >> (p >> 3)) & 1u) u4[p] = P.update(u4, off);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  double r1 = 0.0, re = 0.0;
  PointOp<T, 4, GAL>::phases(nc, false, phase);
  if (ref) r1 = max64((double)fabs(P.resid(u4, p)));
  PointOp<T, 4, GAL>::phases(nc, rev, phase);
  if (ref) re = max64((double)fabs(P.resid(u4, p)));
  off.iterate(u4[p]);
  if (off.template out<T>()) S.off = 1;
  double sum = tree64(0.0 + (double)u4[p]);
  sum = __shfl(sum, 0);
  bool g = false;
  if (mode == 2) g = ((T)re > (T)r1 * T(1.001) && (T)r1 > T(1.e-5));
  if (p == 0) {
    if (ref) { scal[0] = r1; scal[1] = re; }
    scal[2] = sum;
    if (guard) *guard = g ? 1 : 0;
  }
  const double m = sum / 64.0;
  u4[p] = g ? T(0) : (T)((double)u4[p] - m);
}

// Sweeps of the 8^3 level; want: 0 none, 1 the residual into r8 (its maximum returned when norm), 2 the
// maximum only.
template <class T, bool GAL, bool PLAIN>
__device__ __forceinline__ double cc_level8(T* u, const T* rhs, T* r8, const T* op, T dx, int ns, bool rev, int want, int norm,
                                            Cc16Scratch& S) {
  const int p = threadIdx.x;
  Range<PLAIN> off;
  PointOp<T, 8, GAL> P;
  P.load(op, rhs, p, dx, off);
  const int cls = __builtin_amdgcn_readfirstlane(p >> 6);
  PointOp<T, 8, GAL>::phases(ns, rev, [&](unsigned mask) {
    if ((mask >> cls) & 1u) u[p] = P.update(u, off);
    __syncthreads();
  });
  off.iterate(u[p]);
  if (off.template out<T>()) S.off = 1;
  if (!want) return 0.0;
  const T rv = P.resid(u, p);
  if (want == 1) r8[p] = rv;
  return norm ? cc_max((double)fabs(rv), S) : 0.0;
}

// ---- 16^3: one cell per thread ---------------------------------------------------------------------
// In-class index of the cell shifted by (-1, 0, 1)^3; a class's neighbour in direction d lies in the
// class with that axis's bit flipped, at the shift that the point's own bit gives.
struct Cell16 {
  int o[3][3][3];
  __device__ __forceinline__ void set(int q) {
    const int x = q & 7, y = (q >> 3) & 7, z = q >> 6;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) o[c][b][a] = ((x + a - 1) & 7) + 8 * ((y + b - 1) & 7) + 64 * ((z + c - 1) & 7);
  }
};
// shift (0, 1, 2 for -1, 0, +1) of the neighbour at step s of a point with parity bit b
__host__ __device__ constexpr int shift16(int b, int s) { return s == 0 ? 1 : (b ? (s > 0 ? 2 : 1) : (s > 0 ? 1 : 0)); }
__host__ __device__ constexpr int class16(int c, int sx, int sy, int sz) { return c ^ ((sx ? 1 : 0) | (sy ? 2 : 0) | (sz ? 4 : 0)); }
// index of the neighbour of the cell's class-C point (C a constant after unrolling)
__device__ __forceinline__ int nb16(const Cell16& K, int c, int sx, int sy, int sz) {
  return class16(c, sx, sy, sz) * 512 + K.o[shift16(c >> 2, sz)][shift16((c >> 1) & 1, sy)][shift16(c & 1, sx)];
}

// f(integral_constant) for the classes in mask, wave-uniform.
template <int C = 0, class F> __device__ __forceinline__ void each_class(unsigned mask, F&& f) {
  if constexpr (C < 8) {
    if ((mask >> C) & 1u) f(std::integral_constant<int, C>());
    each_class<C + 1>(mask, f);
  }
}

// Sweeps of the 16^3 level, then the residual (want and norm as cc_level8).  The residual's values are
// formed before any is stored, since r may share LDS with staged coefficients (big).
// 19-point: faces and the diagonal's reciprocal in registers; in FP32 the diagonal, the right-hand side and
// the cross factors too; in FP64 (256 registers hold half as many values) the cross factors come from
// G2, G3, G5 in LDS (big).
template <class T, bool PLAIN>
__device__ __forceinline__ double cc_level16_19(T* u, const T* rhs, T* r, T* big, const T* G, T dx, int ns, bool rev, int want,
                                                int norm, Cc16Scratch& S) {
  constexpr bool REG = sizeof(T) == 4;
  const int q = threadIdx.x;
  Cell16 K;
  K.set(q);
  Range<PLAIN> off;
  T w[8][REG ? 7 : 6], y[8], b2[REG ? 8 : 1], x[REG ? 8 : 1][12];
  if constexpr (!REG) {
    for (int t = q; t < 4096; t += CW) {
      big[t] = G[4096 + t];              // G2
      big[4096 + t] = G[2 * 4096 + t];   // G3
      big[8192 + t] = G[4 * 4096 + t];   // G5
    }
    __syncthreads();
  }
  const T dx2 = dx * dx;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    int nb[18];
#pragma unroll
    for (int e = 0; e < 18; ++e) nb[e] = nb16(K, c, NB19[e][0], NB19[e][1], NB19[e][2]);
    T f[7];
    faces19<T>(f, G, 4096, c * 512 + q, nb);
#pragma unroll
    for (int e = 0; e < (REG ? 7 : 6); ++e) w[c][e] = f[e];
    y[c] = recip(f[6], off);
    if constexpr (REG) {
      b2[c] = rhs[c * 512 + q] * dx2;
#pragma unroll
      for (int e = 0; e < 12; ++e) x[c][e] = G[XG19[e][1] * 4096 + nb[XG19[e][0]]];
    }
  }
  // t1, t2 and the diagonal; FP64: the diagonal is summed again rather than held, and the cell's offsets
  // pass through empty asm, which keeps the 240 LDS addresses of the 8 classes from being held too
  auto terms = [&](auto cc, T& t1, T& t2, T& diag) {
    constexpr int c = decltype(cc)::value;
    T p[18];
    if constexpr (REG) {
#pragma unroll
      for (int e = 0; e < 18; ++e) p[e] = u[nb16(K, c, NB19[e][0], NB19[e][1], NB19[e][2])];
      diag = w[c][6];
      terms19<T>(t1, t2, w[c], x[c], p);
    } else {
      Cell16 L = K;
#pragma unroll
      for (int e = 0; e < 27; ++e) asm volatile("" : "+v"(L.o[e / 9][e / 3 % 3][e % 3]));
      T xc[12], f[7];
#pragma unroll
      for (int e = 0; e < 18; ++e) p[e] = u[nb16(L, c, NB19[e][0], NB19[e][1], NB19[e][2])];
#pragma unroll
      for (int e = 0; e < 12; ++e) {
        const int g = XG19[e][0], comp = XG19[e][1];
        xc[e] = big[(comp == 1 ? 0 : comp == 2 ? 4096 : 8192) + nb16(L, c, NB19[g][0], NB19[g][1], NB19[g][2])];
      }
#pragma unroll
      for (int e = 0; e < 6; ++e) f[e] = w[c][e];
      diag = f[6] = -(f[0] + f[1] + f[2] + f[3] + f[4] + f[5]);
      terms19<T>(t1, t2, f, xc, p);
    }
  };
  auto scaled_rhs = [&](auto cc) -> T {
    constexpr int c = decltype(cc)::value;
    if constexpr (REG) return b2[c];
    else return rhs[c * 512 + q] * dx2;
  };
  phases19(ns, rev, [&](unsigned mask) {
    each_class(mask, [&](auto cc) {
      constexpr int c = decltype(cc)::value;
      T t1, t2, d;
      const T b = scaled_rhs(cc);
      terms(cc, t1, t2, d);
      u[c * 512 + q] = quotient(b - t1 - t2, d, y[c], off);
    });
    __syncthreads();
  });
#pragma unroll
  for (int c = 0; c < 8; ++c) off.iterate(u[c * 512 + q]);
  if (off.template out<T>()) S.off = 1;
  if (!want) return 0.0;
  const T di2 = T(1) / dx2;
  T rv[8];
  double a = 0.0;
  each_class(0xFFu, [&](auto cc) {
    constexpr int c = decltype(cc)::value;
    T t1, t2, d;
    terms(cc, t1, t2, d);
    rv[c] = rhs[c * 512 + q] - (t1 + t2 + d * u[c * 512 + q]) * di2;
    a = dmax(a, (double)fabs(rv[c]));
  });
  if (norm) a = cc_max(a, S);
  if (want == 1) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; ++c) r[c * 512 + q] = rv[c];
  }
  return a;
}

// 27-point, FP32: the eight corner coefficients of every point in LDS (big), the others in registers.
// FP64: the coefficients of one class at a time, loaded a phase ahead of their use.
constexpr int corner27(int e) { return ((e % 3 != 1) && (e / 3 % 3 != 1) && (e / 9 != 1)) ? 1 : 0; }
constexpr int rank27(int e, int corner) {  // index of offset e among the corners, or among the others
  int r = 0;
  for (int f = 0; f < e; ++f) r += corner27(f) == corner ? 1 : 0;
  return r;
}
template <class T, bool PLAIN>
__device__ __forceinline__ double cc_level16_27(T* u, const T* rhs, T* r, T* big, const T* A, int ns, bool rev, int want,
                                                int norm, Cc16Scratch& S) {
  constexpr bool REG = sizeof(T) == 4;
  const int q = threadIdx.x;
  Cell16 K;
  K.set(q);
  T rv[8];
  double am = 0.0;
  if constexpr (REG) {
    Range<PLAIN> off;
    T a[8][19], y[8], b[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int e = 0; e < 27; ++e) {
        const T v = A[e * 4096 + c * 512 + q];
        if (corner27(e)) big[rank27(e, 1) * 4096 + c * 512 + q] = v;  // read back by this thread only
        else a[c][rank27(e, 0)] = v;
      }
      y[c] = recip(a[c][rank27(13, 0)], off);
      b[c] = rhs[c * 512 + q];
    }
    auto offsum = [&](auto cc) -> T {
      constexpr int c = decltype(cc)::value;
      T p[27], s = T(0);
#pragma unroll
      for (int e = 0; e < 27; ++e)
        if (e != 13) p[e] = u[nb16(K, c, e % 3 - 1, e / 3 % 3 - 1, e / 9 - 1)];
#pragma unroll
      for (int e = 0; e < 27; ++e)
        if (e != 13) s = s + (corner27(e) ? big[rank27(e, 1) * 4096 + c * 512 + q] : a[c][rank27(e, 0)]) * p[e];
      return s;
    };
    phases27(ns, rev, [&](unsigned mask) {
      each_class(mask, [&](auto cc) {
        constexpr int c = decltype(cc)::value;
        u[c * 512 + q] = quotient(b[c] - offsum(cc), a[c][rank27(13, 0)], y[c], off);
      });
      __syncthreads();
    });
#pragma unroll
    for (int c = 0; c < 8; ++c) off.iterate(u[c * 512 + q]);
    if (off.template out<T>()) S.off = 1;
    if (!want) return 0.0;
    each_class(0xFFu, [&](auto cc) {
      constexpr int c = decltype(cc)::value;
      rv[c] = b[c] - (offsum(cc) + a[c][rank27(13, 0)] * u[c * 512 + q]);
      am = dmax(am, (double)fabs(rv[c]));
    });
  } else {
    T a[27], bc;
    auto fetch = [&](int c) {  // scalar base (field and class) + 32-bit lane offset
      uint32_t o = (uint32_t)q * (uint32_t)sizeof(T);
      asm volatile("" : "+v"(o));
#pragma unroll
      for (int e = 0; e < 27; ++e) a[e] = *(const T*)((const char*)(A + e * 4096 + c * 512) + o);
      bc = *(const T*)((const char*)(rhs + c * 512) + o);
    };
    auto offsum = [&](auto cc, const T (&w)[27]) -> T {
      constexpr int c = decltype(cc)::value;
      T p[27], s = T(0);
#pragma unroll
      for (int e = 0; e < 27; ++e)
        if (e != 13) p[e] = u[nb16(K, c, e % 3 - 1, e / 3 % 3 - 1, e / 9 - 1)];
#pragma unroll
      for (int e = 0; e < 27; ++e)
        if (e != 13) s = s + w[e] * p[e];
      return s;
    };
    // class after mask's in the sweep order (the last one's is the first's)
    auto next = [rev](unsigned mask) -> int {
      const int c = __builtin_ctz(mask);
      constexpr int fwd[8] = {2, 3, 1, 4, 6, 7, 5, 0}, bwd[8] = {7, 2, 0, 1, 3, 6, 4, 5};
      int r = 0;
#pragma unroll
      for (int t = 0; t < 8; ++t) r = c == t ? (rev ? bwd[t] : fwd[t]) : r;
      return r;
    };
    if (ns > 0) fetch(rev ? 7 : 0);
    phases27(ns, rev, [&](unsigned mask) {
      T w[27], bw = bc;
#pragma unroll
      for (int e = 0; e < 27; ++e) w[e] = a[e];
      fetch(next(mask));
      each_class(mask, [&](auto cc) {
        constexpr int c = decltype(cc)::value;
        u[c * 512 + q] = (bw - offsum(cc, w)) / w[13];
      });
      __syncthreads();
    });
    if (!want) return 0.0;
    each_class(0xFFu, [&](auto cc) {
      constexpr int c = decltype(cc)::value;
      fetch(c);
      rv[c] = bc - (offsum(cc, a) + a[13] * u[c * 512 + q]);
      am = dmax(am, (double)fabs(rv[c]));
    });
  }
  if (norm) am = cc_max(am, S);
  if (want == 1) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; ++c) r[c * 512 + q] = rv[c];
  }
  return am;
}

// ---- the cycle -------------------------------------------------------------------------------------
template <class T> struct Cc16Lds {
  T u16[4096], u8[512], rhs8[512], r8[512], u4[64], rhs4[64];
  double du[64], drhs[64];
  Cc16Scratch S;
  T big[sizeof(T) == 4 ? 8 * 4096 : 3 * 4096];  // staged coefficients, and r16 between its sweeps and the restriction
};

__host__ __device__ constexpr int relax_plane(int pre, int n) {  // calcresid's plane order (relax_dev)
  const int nrmax = (n / 4 < 1 ? 1 : n / 4) < 4 ? (n / 4 < 1 ? 1 : n / 4) : 4;
  return (pre > nrmax ? (pre % nrmax ? pre % nrmax : nrmax) : pre) % (n / 2);
}

// p, known to be the same in every lane, in scalar registers.
template <class P> __device__ __forceinline__ P* uniform(P* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (P*)((uint64_t)hi << 32 | lo);
}

// Levels C.n[0] (16, 8 or 4) .. 4 of the cycle C (cw_cycle's schedule), by CW threads, up to the entry
// level's iterate, which is left in LDS; M.S.off is set where a quotient was out of range.
template <class T, bool PLAIN> __device__ __forceinline__ void cc16_levels(const CoarseCycle<T>& C, Cc16Lds<T>& M) {
  static_assert(CW == 512, "one 16^3 cell, and one 8^3 point, per thread");
  const int t = threadIdx.x, lb = C.nl - 1, l8 = C.nl - 2, l16 = C.nl - 3;
  T* r16 = M.big;
  double r1_16 = 0.0, r1_8 = 0.0;
  // the entry level's iterate and right-hand side; coarser levels start from 0
  if (l16 >= 0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) M.u16[c * 512 + t] = C.u[l16][c * 512 + t];
  } else if (l8 >= 0) {
    M.u8[t] = C.u[l8][t];
    M.rhs8[t] = C.rhs[l8][t];
  } else if (t < 64) {
    M.u4[t] = C.u[lb][t];
    M.rhs4[t] = C.rhs[lb][t];
  }
  __syncthreads();
  if (l16 >= 0) {
    if (C.A[l16]) r1_16 = cc_level16_27<T, PLAIN>(M.u16, uniform(C.rhs[l16]), r16, M.big, uniform(C.A[l16]), C.sw[l16], false, 1, C.ref, M.S);
    else r1_16 = cc_level16_19<T, PLAIN>(M.u16, uniform(C.rhs[l16]), r16, M.big, uniform(C.G[l16]), C.dx[l16], C.sw[l16], false, 1, C.ref, M.S);
    if (C.ref && t == 0) C.scal[l16][0] = r1_16;
    __syncthreads();
    restrict_point<T, 1, true>(M.rhs8, r16, 16, relax_plane(C.sw[l16], 16), t);
    M.u8[t] = T(0);
    __syncthreads();
  }
  if (l8 >= 0) {
    if (C.A[l8]) r1_8 = cc_level8<T, true, PLAIN>(M.u8, M.rhs8, M.r8, C.A[l8], C.dx[l8], C.sw[l8], false, 1, C.ref, M.S);
    else r1_8 = cc_level8<T, false, PLAIN>(M.u8, M.rhs8, M.r8, C.G[l8], C.dx[l8], C.sw[l8], false, 1, C.ref, M.S);
    if (C.ref && t == 0) C.scal[l8][0] = r1_8;
    __syncthreads();
    if (t < 64) {
      restrict_point<T, 1, true>(M.rhs4, M.r8, 8, relax_plane(C.sw[l8], 8), t);
      M.u4[t] = T(0);
    }
    __syncthreads();
  }
  const int mode_b = (C.ref && !(C.top && lb == 0)) ? 2 : 0;
  if (C.mixed) {
    if (t < 64) {
      M.drhs[t] = (double)M.rhs4[t];
      M.du[t] = 0.0;
    }
    __syncthreads();
    if (C.dA) cc_bottom<double, true, PLAIN>(M.du, M.drhs, C.dA, C.ddx, C.coarse, C.symmetric, C.dscal, C.dguard, C.ref, mode_b, M.S);
    else cc_bottom<double, false, PLAIN>(M.du, M.drhs, C.dG, C.ddx, C.coarse, C.symmetric, C.dscal, C.dguard, C.ref, mode_b, M.S);
    if (t < 64) M.u4[t] = (T)M.du[t];
  } else {
    if (C.A[lb]) cc_bottom<T, true, PLAIN>(M.u4, M.rhs4, C.A[lb], C.dx[lb], C.coarse, C.symmetric, C.scal[lb], C.guard[lb], C.ref, mode_b, M.S);
    else cc_bottom<T, false, PLAIN>(M.u4, M.rhs4, C.G[lb], C.dx[lb], C.coarse, C.symmetric, C.scal[lb], C.guard[lb], C.ref, mode_b, M.S);
  }
  __syncthreads();
  if (l8 < 0) return;
  if (t < 64) prolong_cell<T, true>(M.u8, M.u4, 8, 1, t);
  __syncthreads();
  double re;
  if (C.A[l8]) re = cc_level8<T, true, PLAIN>(M.u8, M.rhs8, M.r8, C.A[l8], C.dx[l8], C.sw[l8], C.symmetric != 0, C.ref ? 2 : 0, C.ref, M.S);
  else re = cc_level8<T, false, PLAIN>(M.u8, M.rhs8, M.r8, C.G[l8], C.dx[l8], C.sw[l8], C.symmetric != 0, C.ref ? 2 : 0, C.ref, M.S);
  if (C.ref && t == 0) C.scal[l8][1] = re;
  cc_zerosum<T, 8>(M.u8, C.scal[l8], C.guard[l8], (C.ref && !(C.top && l8 == 0)) ? 1 : 0, r1_8, re, M.S);
  if (l16 < 0) return;
  prolong_cell<T, true>(M.u16, M.u8, 16, 1, t);
  __syncthreads();
  if (C.A[l16]) re = cc_level16_27<T, PLAIN>(M.u16, uniform(C.rhs[l16]), r16, M.big, uniform(C.A[l16]), C.sw[l16], C.symmetric != 0, C.ref ? 2 : 0, C.ref, M.S);
  else re = cc_level16_19<T, PLAIN>(M.u16, uniform(C.rhs[l16]), r16, M.big, uniform(C.G[l16]), C.dx[l16], C.sw[l16], C.symmetric != 0, C.ref ? 2 : 0, C.ref, M.S);
  if (C.ref && t == 0) C.scal[l16][1] = re;
  cc_zerosum<T, 16>(M.u16, C.scal[l16], C.guard[l16], (C.ref && !(C.top && l16 == 0)) ? 1 : 0, r1_16, re, M.S);
}

// The cycle; off the quotients' range once more with plain divisions, from the caller's arrays, which the
// levels on chip have only read but for the per-level scalars and guards, formed again.
template <class T> __device__ __forceinline__ void cc16_cycle(const CoarseCycle<T>& C, Cc16Lds<T>& M) {
  const int t = threadIdx.x;
  if (t == 0) M.S.off = 0;  // every level starts behind a barrier
  cc16_levels<T, false>(C, M);
  __syncthreads();
  if (M.S.off) cc16_levels<T, true>(C, M);
  if (C.nl == 1) {
    if (t < 64) C.u[0][t] = M.u4[t];
  } else if (C.nl == 2) {
    C.u[0][t] = M.u8[t];
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) C.u[0][c * 512 + t] = M.u16[c * 512 + t];
  }
}

template <class T> __global__ __launch_bounds__(CW) void k_coarse16(CoarseCycle<T> C) {
  __shared__ Cc16Lds<T> M;
  cc16_cycle<T>(C, M);
}

// One workgroup per grid of a batched group (k_coarse_stack's levels and skip rule).
__global__ __launch_bounds__(CW) void k_coarse16_stack(StackLevels L, const int* __restrict__ act) {
  __shared__ Cc16Lds<double> M;
  __shared__ CoarseCycle<double> C;
  if (act && !act[blockIdx.x]) return;
  stack_table(C, L, blockIdx.x);
  __syncthreads();
  cc16_cycle<double>(C, M);
}

}  // namespace mmh
