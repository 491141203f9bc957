// kernels_fft.hpp -- the real 3-D FFT of the spectral stages (rlft3/fourn, mmh/recipes12.f90:1-135).
//
// Every transform is the radix-2 Stockham recurrence of the CPU restatement, its twiddles W[q] =
// exp(s 2 pi i q / L) from a host table, so each butterfly rounds as the restatement's does.  The
// kernels run three radix-2 steps per pass on 8 values held in registers (the remainder of log2 L in
// a first pass of one or two steps) and exchange through LDS between passes: the same butterflies
// in the same order of operations, two or three exchanges per line instead of log2 L.
//
// All three axes are bound by memory: one read and one write of the array per axis.  Lines along x
// are contiguous.  Lines along y and z take 128 B of adjacent columns per workgroup, so every access
// is a full 128 B segment.  Measured at 512^3 FP32 (MI355X): 214 us per strided axis, 199 us along x
// (1.07 GB moved, 5.0-5.4 TB/s, what a large copy reaches), against 1449 us for an axis on average with
// one line per workgroup and log2 L exchanges, where a strided line took 8 B of each segment it touched.
#pragma once
#include "kernels.hpp"

namespace mmh {

template <class T> struct C2 { T r, i; };

template <int L> struct FftShape {
  static constexpr int E = L < 8 ? L : 8;  // values per thread
  static constexpr int TL = L / E;         // threads per line
  static constexpr int lg = __builtin_ctz(L);
  static constexpr int R0 = lg <= 3 ? L : (lg % 3 == 0 ? 8 : 1 << (lg % 3));  // radix of the first pass
};

// One pass of radix R on the thread's values: element (t + q TL) + m L/R of the line is v[q + m E/R].
// Step s of the pass pairs (b, m) with (b, m + R/2^(s+1)): u0 +- w u1 with w = W[(k + b P) L / (2^(s+1) P)],
// k = t' mod P.  The result b of butterfly q is left in v[q + b E/R].
template <class T, int L, int P, int R>
__device__ __forceinline__ void fft_pass(C2<T>* v, const C2<T>* tw, int t) {
  constexpr int E = FftShape<L>::E, TL = FftShape<L>::TL, Q = E / R;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k = (t + q * TL) & (P - 1);
    C2<T> x[R];
#pragma unroll
    for (int m = 0; m < R; ++m) x[m] = v[q + m * Q];
#pragma unroll
    for (int S = 1; S < R; S <<= 1) {  // S = 2^s results per butterfly so far, x[m S + b]
      C2<T> y[R];
#pragma unroll
      for (int b = 0; b < S; ++b) {
        const C2<T> w = tw[(k + b * P) * (L / (2 * S * P))];
#pragma unroll
        for (int m = 0; m < R / (2 * S); ++m) {
          const C2<T> u0 = x[m * S + b], u1 = x[(m + R / (2 * S)) * S + b];
          const T tr = w.r * u1.r - w.i * u1.i;
          const T ti = w.r * u1.i + w.i * u1.r;
          y[m * 2 * S + b] = C2<T>{u0.r + tr, u0.i + ti};
          y[m * 2 * S + b + S] = C2<T>{u0.r - tr, u0.i - ti};
        }
      }
#pragma unroll
      for (int m = 0; m < R; ++m) x[m] = y[m];
    }
#pragma unroll
    for (int m = 0; m < R; ++m) v[q + m * Q] = x[m];
  }
}

// The passes from stride P on.  Between passes the results go to their Stockham positions in LDS,
// lds[ix(pos)], and the next pass reads elements t + s TL.  Every thread of the workgroup calls it.
template <class T, int L, int P, class IX>
__device__ __forceinline__ void fft_line(C2<T>* v, C2<T>* lds, const C2<T>* tw, int t, IX ix) {
  constexpr int E = FftShape<L>::E, TL = FftShape<L>::TL;
  constexpr int R = P == 1 ? FftShape<L>::R0 : 8;
  fft_pass<T, L, P, R>(v, tw, t);
  if constexpr (P * R < L) {
    __syncthreads();  // the line's previous contents have been read
#pragma unroll
    for (int q = 0; q < E / R; ++q) {
      const int tp = t + q * TL, k = tp & (P - 1), base = (tp - k) * R + k;
#pragma unroll
      for (int b = 0; b < R; ++b) lds[ix(base + b * P)] = v[q + b * (E / R)];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < E; ++s) v[s] = lds[ix(t + s * TL)];
    fft_line<T, L, P * R>(v, lds, tw, t, ix);
  }
}

// Lines along x: contiguous, 256 threads per workgroup, 256 / TL lines.
template <class T, int L>
__global__ __launch_bounds__(256) void k_fft_x(C2<T>* out, const C2<T>* in, const C2<T>* __restrict__ W, i64 nl) {
  constexpr int E = FftShape<L>::E, TL = FftShape<L>::TL, NL = 256 / TL, LP = L + L / 8 + 1;
  __shared__ C2<T> lds[NL * LP];
  __shared__ C2<T> tw[L / 2];
  for (int q = threadIdx.x; q < L / 2; q += 256) tw[q] = W[q];
  const int t = threadIdx.x % TL, ln = threadIdx.x / TL;
  const i64 l = (i64)blockIdx.x * NL + ln;
  C2<T> v[E];
#pragma unroll
  for (int s = 0; s < E; ++s) v[s] = l < nl ? in[l * L + t + s * TL] : C2<T>{T(0), T(0)};
  __syncthreads();
  fft_line<T, L, 1>(v, lds + ln * LP, tw, t, [](int p) { return p + (p >> 3); });
  if (l < nl)
#pragma unroll
    for (int s = 0; s < E; ++s) out[l * L + t + s * TL] = v[s];
}

// Lines of stride `inner` (a power of two, 2^lgi): line l starts at (l mod inner) + (l / inner) inner L.  A
// workgroup takes C adjacent lines, C the columns of a 128 B segment where LDS (64 KiB per
// workgroup, two of them per CU) and 1024 threads allow.  scale > 0: the inverse's normalisation,
// x 2 / n / n / n as three multiplications by 1 / n (n a power of two, so 1 / n is exact and each
// product rounds as the division does).
template <class T, int L> struct FftCols {
  static constexpr int a = 128 / (int)sizeof(C2<T>), b = 65536 / (L * (int)sizeof(C2<T>)), d = 1024 / FftShape<L>::TL;
  static constexpr int ab = a < b ? a : b, C = ab < d ? ab : d;
  static constexpr int NT = C * FftShape<L>::TL;
};
template <class T, int L>
__global__ __launch_bounds__((FftCols<T, L>::NT)) void k_fft_cols(C2<T>* out, const C2<T>* in, const C2<T>* __restrict__ W,
                                                              i64 nl, int lgi, T scale) {
  constexpr int E = FftShape<L>::E, TL = FftShape<L>::TL, C = FftCols<T, L>::C, NT = FftCols<T, L>::NT;
  __shared__ C2<T> lds[L * C];
  __shared__ C2<T> tw[L / 2];
  for (int q = threadIdx.x; q < L / 2; q += NT) tw[q] = W[q];
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  const i64 l = (i64)blockIdx.x * C + c, st = (i64)1 << lgi;
  const i64 base = (l & (st - 1)) + ((l >> lgi) << lgi) * L;
  C2<T> v[E];
#pragma unroll
  for (int s = 0; s < E; ++s) v[s] = l < nl ? in[base + (t + s * TL) * st] : C2<T>{T(0), T(0)};
  __syncthreads();
  fft_line<T, L, 1>(v, lds, tw, t, [c](int p) { return p * C + c; });
  if (l >= nl) return;
#pragma unroll
  for (int s = 0; s < E; ++s) {
    C2<T> x = v[s];
    if (scale > T(0)) {
      x.r = x.r * T(2.) * scale * scale * scale;
      x.i = x.i * T(2.) * scale * scale * scale;
    }
    out[base + (t + s * TL) * st] = x;
  }
}

// ------------------------------------------------------------------------------------------------
// rlft3 recombination between the half-length complex transform and the real spectrum
// (mmh/recipes12.f90:100-127), of one pair: X at (i1, i2, i3) and Y at (h - i1, -i2, -i3), w =
// exp(isign 2 pi i i1 / n); i1 = 0 pairs with the Nyquist plane (no twiddle).  c2i = -isign / 2.
template <class T> __device__ __forceinline__ void rlft_pair0(C2<T>& X, C2<T>& Y, T c2i) {
  const C2<T> s{X.r + Y.r, X.i - Y.i}, d{X.r - Y.r, X.i + Y.i};
  const C2<T> H1{T(0.5) * s.r, T(0.5) * s.i};
  const C2<T> H2{-c2i * d.i, c2i * d.r};
  X = C2<T>{H1.r + H2.r, H1.i + H2.i};
  Y = C2<T>{H1.r - H2.r, -(H1.i - H2.i)};
}
template <class T> __device__ __forceinline__ void rlft_pair(C2<T>& X, C2<T>& Y, T wr, T wi, T c2i) {
  const C2<T> s{X.r + Y.r, X.i - Y.i}, d{X.r - Y.r, X.i + Y.i};
  const C2<T> H1{T(0.5) * s.r, T(0.5) * s.i};
  const C2<T> H2{-c2i * d.i, c2i * d.r};
  const C2<T> WH{wr * H2.r - wi * H2.i, wr * H2.i + wi * H2.r};
  X = C2<T>{H1.r + WH.r, H1.i + WH.i};
  Y = C2<T>{H1.r - WH.r, -(H1.i - WH.i)};
}

// Pass A of a transform by itself: k1 = 0 with the Nyquist plane speq.  One thread per pair of
// (i2, i3) and its mirror image (both roles), so the plane is read before it is overwritten.
// forward: the previous speq is the k1 = 0 plane itself.
template <class T>
__global__ void k_rlft_k0(C2<T>* __restrict__ z, C2<T>* __restrict__ sq, int h1, int n, int forward, T c2i) {
  const i64 q = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (i64)n * n) return;
  const int i2 = (int)(q % n), i3 = (int)(q / n);
  const i64 m = (i64)((n - i2) & (n - 1)) + (i64)n * ((n - i3) & (n - 1));
  if (m < q) return;
  C2<T> X = z[h1 * q], Xm = z[h1 * m];
  C2<T> Y = forward ? Xm : sq[m], Ym = forward ? X : sq[q];
  rlft_pair0(X, Y, c2i);
  z[h1 * q] = X;
  sq[m] = Y;
  if (m == q) return;
  rlft_pair0(Xm, Ym, c2i);
  z[h1 * m] = Xm;
  sq[q] = Ym;
}

// Pass B: the pairs 1 <= i1 < h1 - i1.
template <class T>
__global__ void k_rlft_pairs(C2<T>* __restrict__ z, const C2<T>* __restrict__ wtab, int h1, int n2, int n3, T c2i) {
  const int npair = (h1 - 1) / 2;  // number of i1 values with i1 < h1 - i1, i1 >= 1
  const i64 q = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (i64)npair * n2 * n3) return;
  const int i1 = 1 + (int)(q % npair);
  const i64 r = q / npair;
  const int i2 = (int)(r % n2), i3 = (int)(r / n2);
  const int j1 = h1 - i1, j2 = i2 == 0 ? 0 : n2 - i2, j3 = i3 == 0 ? 0 : n3 - i3;
  C2<T>& Xr = z[(i64)i1 + (i64)h1 * ((i64)i2 + (i64)n2 * i3)];
  C2<T>& Yr = z[(i64)j1 + (i64)h1 * ((i64)j2 + (i64)n2 * j3)];
  C2<T> X = Xr, Y = Yr;
  rlft_pair(X, Y, wtab[i1].r, wtab[i1].i, c2i);
  Xr = X;
  Yr = Y;
}

// Spectral multiplier at (ic, j, k) of the real spectrum (ic = n/2 the Nyquist plane).
// mode 0: divide by the 7-point symbol 2cos kx + 2cos ky + 2cos kz - 6 (mmh/limiter.f90:560-575)
// from host cosine tables; mode 1: multiply by |k|^2 (mmh/reconstruct.f90:14-36);
// mode 2/3/4: multiply by i k_x, i k_y, i k_z (mmh/gradient.f90:16-26, 34-48, 56-70).
template <class T>
__device__ __forceinline__ void spectral_mul(C2<T>& a, int ic, int j, int k, int n, int mode, const T* __restrict__ cs, T pi) {
  const int h = n / 2;
  const T rn = T(1) / T(n);  // exact (n a power of two): x rn rounds as x / n
  if (mode == 0) {
    T ak = T(2) * cs[ic] + T(2) * cs[n + j] + T(2) * cs[2 * n + k] - T(6);
    if (fabs(ak) < T(1e-10)) ak = 1;
    a.r = a.r / ak;
    a.i = a.i / ak;
  } else if (mode == 1) {
    T k3 = (k + 1 <= h + 1) ? T(k) : T(k - n);
    k3 = k3 * rn * T(2.) * pi;
    T k2 = (j + 1 <= h + 1) ? T(j) : T(j - n);
    k2 = k2 * rn * T(2.) * pi;
    T k1 = T(ic);
    k1 = k1 * rn * T(2.) * pi;
    const T f = k1 * k1 + k2 * k2 + k3 * k3;
    a.r = a.r * f;
    a.i = a.i * f;
  } else {
    T km;
    if (mode == 2) km = T(ic);
    else if (mode == 3) km = (j + 1 <= h + 1) ? T(j) : T(j - n);
    else km = (k + 1 <= h + 1) ? T(k) : T(k - n);
    const T cr = a.r * T(0) - a.i * km, ci = a.r * km + a.i * T(0);
    a.r = cr * rn * T(2.) * pi;
    a.i = ci * rn * T(2.) * pi;
  }
}

// The middle of a spectral operation in one pass over the spectrum: forward recombination, the
// multiplier, inverse recombination and the inverse transform's x lines, from the forward complex
// transform `in` (before its recombination) to `out` (in may equal out).  The recombination couples
// line (j, k) with line (-j, -k) only, so a workgroup takes such pairs whole: 256 / (2 TL) of them.
// As separate launches this was five reads and writes of the spectrum (two recombinations of the
// pairs, the multiplier, the x lines, the Nyquist planes besides).  512^3 FP32: 264 us (4.1 TB/s)
// against 170 + 276 + 170 + 21 us before the x lines.  sqout (may be null) receives the
// Nyquist plane as the inverse recombination leaves it.  zero_dc: real part of entry (0, 0, 0) set to 0
// after the multiplier (mmh/limiter.f90:576).
// Wp, Wm: twiddles of length n = 2 L, signs + and - (for the recombinations); W: of length L, sign -.
template <class T, int L>
__global__ __launch_bounds__(256) void k_rlft_mid(C2<T>* out, const C2<T>* in, const C2<T>* __restrict__ Wp,
                                                  const C2<T>* __restrict__ Wm, const C2<T>* __restrict__ W,
                                                  C2<T>* __restrict__ sqout, int mode, int zero_dc,
                                                  const T* __restrict__ cs, T pi) {
  constexpr int E = FftShape<L>::E, TL = FftShape<L>::TL, NP = 128 / TL, LP = L + L / 8 + 1, n = 2 * L;
  __shared__ C2<T> lds[2 * NP * LP];
  __shared__ C2<T> tw[L / 2];
  for (int q = threadIdx.x; q < L / 2; q += 256) tw[q] = W[q];
  const int t = threadIdx.x % TL, ln = threadIdx.x / TL, side = ln & 1;
  // pair q: planes 0 < k < n/2 with every j, then j <= n/2 of the planes k = 0 and k = n/2
  const i64 q = (i64)blockIdx.x * NP + (ln >> 1), body = (i64)(L - 1) * n, total = body + 2 * (L + 1);
  int j, k;
  if (q < body) {
    k = 1 + (int)(q / n);
    j = (int)(q % n);
  } else {
    const int r = (int)(q - body);
    k = r < L + 1 ? 0 : L;
    j = r % (L + 1);
  }
  const int mj = (n - j) & (n - 1), mk = (n - k) & (n - 1);
  const bool self = mj == j && mk == k;
  const bool live = q < total && !(self && side);
  if (side) { j = mj; k = mk; }
  const int oj = (n - j) & (n - 1), ok = (n - k) & (n - 1);  // the partner line
  const i64 l = (i64)j + (i64)n * k;
  auto ix = [](int p) { return p + (p >> 3); };
  C2<T>* me = lds + ln * LP;
  C2<T>* other = self ? me : lds + (ln ^ 1) * LP;
  if (live)
#pragma unroll
    for (int s = 0; s < E; ++s) me[ix(t + s * TL)] = in[l * L + t + s * TL];
  __syncthreads();
  const T cf = T(-0.5), ci = T(0.5);
  C2<T> z0{T(0), T(0)};
  if (live) {
    for (int i1 = t == 0 ? TL : t; i1 < L / 2; i1 += TL) {  // (X here, Y in the partner line), i1 >= 1
      C2<T> X = me[ix(i1)], Y = other[ix(L - i1)];
      rlft_pair(X, Y, Wp[i1].r, Wp[i1].i, cf);
      spectral_mul(X, i1, j, k, n, mode, cs, pi);
      spectral_mul(Y, L - i1, oj, ok, n, mode, cs, pi);
      rlft_pair(X, Y, Wm[i1].r, Wm[i1].i, ci);
      me[ix(i1)] = X;
      other[ix(L - i1)] = Y;
    }
    if (t == 0) {
      C2<T> X = me[ix(0)], Y = other[ix(0)];
      rlft_pair0(X, Y, cf);
      spectral_mul(X, 0, j, k, n, mode, cs, pi);
      if (zero_dc && j == 0 && k == 0) X.r = T(0);
      spectral_mul(Y, L, oj, ok, n, mode, cs, pi);
      rlft_pair0(X, Y, ci);
      z0 = X;
      if (sqout) sqout[oj + (i64)n * ok] = Y;
      C2<T> m = me[ix(L / 2)];  // k1 = n/4 pairs with itself and is not recombined
      spectral_mul(m, L / 2, j, k, n, mode, cs, pi);
      me[ix(L / 2)] = m;
    }
  }
  __syncthreads();
  if (live && t == 0) me[ix(0)] = z0;
  __syncthreads();
  C2<T> v[E];
#pragma unroll
  for (int s = 0; s < E; ++s) v[s] = live ? me[ix(t + s * TL)] : C2<T>{T(0), T(0)};
  fft_line<T, L, 1>(v, me, tw, t, ix);
  if (live)
#pragma unroll
    for (int s = 0; s < E; ++s) out[l * L + t + s * TL] = v[s];
}

}  // namespace mmh
