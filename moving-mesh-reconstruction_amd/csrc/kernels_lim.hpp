// kernels_lim.hpp -- grid limiter (calcdefp), and relaxing-TVD transport kernels.
// Same conventions as kernels.hpp: column-major, periodic, reference association order,
// built with -ffp-contract=off.
#pragma once
#include "kernels.hpp"

namespace mmh {

template <class T> struct Hs { T xx, yy, zz, xy, yz, xz; };

// Point threadIdx.x of the 256-point chunk `chunk` of a field whose n is a power of two and n^2 a multiple of
// 256: the chunk lies in one plane, so plane bases are scalars and a lane adds its 32-bit offset.
struct PlanePoint {
  int lg, m, k;
  i64 pl;      // first point of the plane
  unsigned r;  // index in the plane
  int xs[3], ys[3];
  __device__ __forceinline__ PlanePoint(int n, i64 chunk) : lg(__builtin_ctz(n)), m(n - 1) {
    const i64 p0 = chunk * 256;
    k = (int)(p0 >> (2 * lg));
    pl = (i64)k << (2 * lg);
    r = (unsigned)(p0 - pl) + threadIdx.x;
    const int i = (int)r & m, j = (int)(r >> lg);
    xs[0] = (i - 1) & m; xs[1] = i; xs[2] = (i + 1) & m;
    ys[0] = ((j - 1) & m) << lg; ys[1] = j << lg; ys[2] = ((j + 1) & m) << lg;
  }
  template <class T> __device__ __forceinline__ T at(const T* f, int di, int dj, int dk) const {
    return *(const T*)((const char*)(f + ((i64)((k + dk) & m) << (2 * lg))) +
                       (uint32_t)(xs[di + 1] + ys[dj + 1]) * (uint32_t)sizeof(T));
  }
  template <class T> __device__ __forceinline__ void put(T* f, T v) const {
    *(T*)((char*)(f + pl) + r * (uint32_t)sizeof(T)) = v;
  }
};
// Hessian stencil without grid scaling (mmh/limiter.f90:268-273, mmh/relaxing.f90:876-881).
template <class T> __device__ __forceinline__ Hs<T> hess(const T* __restrict__ f, const PlanePoint& P) {
  const T f0 = P.at(f, 0, 0, 0);
  Hs<T> h;
  h.xx = (P.at(f, 1, 0, 0) - T(2) * f0 + P.at(f, -1, 0, 0));
  h.yy = (P.at(f, 0, 1, 0) - T(2) * f0 + P.at(f, 0, -1, 0));
  h.zz = (P.at(f, 0, 0, 1) - T(2) * f0 + P.at(f, 0, 0, -1));
  h.xy = (P.at(f, 1, 1, 0) - P.at(f, -1, 1, 0) - P.at(f, 1, -1, 0) + P.at(f, -1, -1, 0)) / T(4);
  h.yz = (P.at(f, 0, 1, 1) - P.at(f, 0, 1, -1) - P.at(f, 0, -1, 1) + P.at(f, 0, -1, -1)) / T(4);
  h.xz = (P.at(f, 1, 0, 1) - P.at(f, -1, 0, 1) - P.at(f, 1, 0, -1) + P.at(f, -1, 0, -1)) / T(4);
  return h;
}

// Smallest eigenvalue of symmetric C by the trigonometric method; returns 1/lambda_min
// (mmh/limiter.f90:346-358).
template <class T>
__device__ __forceinline__ T compression_of(T c11, T c12, T c13, T c22, T c23, T c33, T pi) {
  T trace = c11 + c22 + c33;
  T d11 = c11 - trace / T(3);
  T d22 = c22 - trace / T(3);
  T a = -(d11 * d11 + c12 * c12 + c13 * c13 + d11 * d22 + d22 * d22 + c23 * c23);
  T b = -(d11 * (c12 * c12)) + (d11 * d11) * d22 - (c12 * c12) * d22 + (c13 * c13) * d22 + d11 * (d22 * d22)
        - T(2) * c12 * c13 * c23 + d11 * (c23 * c23);
  if (fabs(a) < T(1.e-20)) a = T(1.e-20);
  T am = T(2) * sqrt(fabs(-a) / T(3));
  T arg = T(3) * b / a / am;
  arg = dmax(T(-1.), dmin(T(1.), arg));
  T theta = acos(arg) / T(3);
  // The three roots are am cos(theta + 0, 2 pi/3, 4 pi/3) with theta in [0, pi/3]: the first is the largest,
  // and the third exceeds the second by sqrt(3) am sin(theta), far above rounding unless theta is
  // small, so only there is the third formed (and the smaller taken); the value is that of the
  // minimum over all three.
  T t3 = trace / T(3);
  T l2 = am * cos(theta + T(2) * pi / T(3.)) + t3;
  if (!(theta > T(0.01))) {
    T l3 = am * cos(theta + T(4) * pi / T(3.)) + t3;
    l2 = dmin(l2, l3);
  }
  return T(1) / l2;
}

// Step 1 of calcdefp: clipped, scaled mass mismatch (mmh/limiter.f90:134-169).  rho (may be null): the
// density itself, contiguous, for the metric's box mean (u is read once for both).
template <class T>
__global__ void k_mismatch(T* __restrict__ tmp, T* __restrict__ rho, const T* __restrict__ u, int nf, i64 n3, T dtold) {
  const i64 p = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n3) return;
  const T u1 = u[(i64)nf * p];
  if (rho) rho[p] = u1;
  T t1 = T(1.0f) - u1;
  const T xhigh = 2;
  if (fabs(t1) > xhigh) t1 = copysign(xhigh, t1);
  tmp[p] = t1 / T(30) / dtold;
}

// Diagnostics of a workgroup: thread values combined over the wavefront and then the workgroup, stored
// at part[f gridDim.x + block].  Maxima, minima and counts do not depend on the order: a value that is
// NaN is passed over (a, the value so far, never is one).
template <int OP> __device__ __forceinline__ double stat_op(double a, double b) {
  return OP == 0 ? a + b : (OP == 1 ? (b > a ? b : a) : (b < a ? b : a));
}
template <int OP> __device__ __forceinline__ void block_stat(double a, double* part, int f) {
  __shared__ double w[4];
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) a = stat_op<OP>(a, __shfl_xor(a, h));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0)
    part[(i64)f * gridDim.x + blockIdx.x] = stat_op<OP>(stat_op<OP>(w[0], w[1]), stat_op<OP>(w[2], w[3]));
}
// The same over nb block results per field, in field order, by gridDim.x workgroups of 256.
__global__ __launch_bounds__(256) void k_stats(double* __restrict__ out, const double* __restrict__ part, i64 nb, int nf,
                                               unsigned ops) {
  for (int f = 0; f < nf; ++f) {
    const unsigned op = (ops >> (2 * f)) & 3u;
    i64 b = (i64)blockIdx.x * 256 + threadIdx.x;
    double a = op == 0 ? 0.0 : part[f * nb + (b < nb ? b : 0)];  // a repeated value changes no maximum or minimum
    if (op == 0 && b < nb) a = part[f * nb + b];
    for (b += (i64)gridDim.x * 256; b < nb; b += (i64)gridDim.x * 256) {
      const double v = part[f * nb + b];
      a = op == 0 ? stat_op<0>(a, v) : (op == 1 ? stat_op<1>(a, v) : stat_op<2>(a, v));
    }
    if (op == 0) block_stat<0>(a, out, f);
    else if (op == 1) block_stat<1>(a, out, f);
    else block_stat<2>(a, out, f);
  }
}

// Points of a thread of the limiter's kernels (n >= 16, so n^3 is a multiple of 256 LIM_PT): 256 LIM_PT
// consecutive points per workgroup, so that the
// block results stay few (at one point per thread the host read and combined 20 MB of them at 512^3).
constexpr int LIM_PT = 4;

// Step 3 of calcdefp (mmh/limiter.f90:238-381), pointwise part: the three components of the fluid's flux,
// s_d = (b_d . momentum) / rho with b = adj(A)/det, A = I + H(def) (limiter.f90:274-286), and which of
// the expansion limiter (det > 10, flag bit 0) and the compression gate (bit 1) hold at the point.
// The metric is formed and used in one pass; forming it at the flux's six neighbours from a stored
// metric took 5.1 ms with that pass at 512^3 FP32, the two passes now 1.43 + 0.50 ms.
// part: per workgroup nexpand, detmax, detmin.  n a power of two, n^2 a multiple of 256.
template <class T>
__global__ __launch_bounds__(256) void k_lim_point(T* __restrict__ s, unsigned char* __restrict__ flag,
                                                   const T* __restrict__ def, const T* __restrict__ u, int nf, int n, T dtold,
                                                   T cmpmaxglobal, T pi, double* __restrict__ part) {
  const i64 n3 = (i64)n * n * n;
  double nexp = 0.0, dhi = 0.0, dlo = 1.0;
  const i64 chunk0 = (i64)xcd_remap(blockIdx.x, gridDim.x) * LIM_PT;
  for (int q = 0; q < LIM_PT; ++q) {
    const PlanePoint P(n, chunk0 + q);
    const Hs<T> h = hess(def, P);
    const T a11 = T(1) + h.xx, a12 = h.xy, a13 = h.xz, a22 = T(1) + h.yy, a23 = h.yz, a33 = T(1) + h.zz;
    const T det = a11 * a22 * a33 + T(2) * a12 * a13 * a23 - (a13 * a13) * a22 - a11 * (a23 * a23) - (a12 * a12) * a33;
    const T b11 = (a22 * a33 - a23 * a23) / det;
    const T b12 = (a13 * a23 - a12 * a33) / det;
    const T b13 = (a12 * a23 - a13 * a22) / det;
    const T b22 = (a11 * a33 - a13 * a13) / det;
    const T b23 = (a12 * a13 - a11 * a23) / det;
    const T b33 = (a11 * a22 - a12 * a12) / det;
    const T* ul = u + (i64)nf * (P.pl + P.r);
    const T u0 = ul[0], u1 = ul[1], u2 = ul[2], u3 = ul[3];
    P.put(s, (b11 * u1 + b12 * u2 + b13 * u3) / u0);
    P.put(s + n3, (b12 * u1 + b22 * u2 + b23 * u3) / u0);
    P.put(s + 2 * n3, (b13 * u1 + b23 * u2 + b33 * u3) / u0);
    const T compression = compression_of(a11, a12, a13, a22, a23, a33, pi);
    const T cmpmax = cmpmaxglobal * T(1);
    const T tlim = T(3) * (T(1) / cmpmax - T(1) / compression) / dtold;
    const bool ex = det > T(10.0f);
    P.put(flag, (unsigned char)((ex ? 1 : 0) | (tlim > T(0) ? 2 : 0)));
    nexp += ex ? 1.0 : 0.0;
    dhi = stat_op<1>(dhi, (double)det);
    dlo = stat_op<2>(dlo, (double)det);
  }
  block_stat<0>(nexp, part, 0);
  block_stat<1>(dhi, part, 1);
  block_stat<2>(dlo, part, 2);
}

// The eflux of a point from the fluxes of its neighbours and the gates of the point one plane above
// it (limiter.f90:330-381); gate: the derivative of this eflux with respect to the smoothed mismatch
// tmp at fixed def (the expansion limiter's -2|.|, the compression gate's max(0, .) and the clamp, each
// taken on the branch the forward pass took; the e.v terms vanish with u(2:4) = 0).
// part: per workgroup fluxmax, fluxmin.
template <class T>
__global__ __launch_bounds__(256) void k_eflux(T* __restrict__ eflux, const T* __restrict__ tmp, const T* __restrict__ s,
                                               const unsigned char* __restrict__ flag, int n, T dtold, T dtaumesh,
                                               double* __restrict__ part, T* __restrict__ gate) {
  const i64 n3 = (i64)n * n * n;
  double fhi = 0.0, flo = 0.0;
  const i64 chunk0 = (i64)xcd_remap(blockIdx.x, gridDim.x) * LIM_PT;
  for (int q = 0; q < LIM_PT; ++q) {
    const PlanePoint P(n, chunk0 + q);
    const T s1p = P.at(s, 1, 0, 0), s1m = P.at(s, -1, 0, 0);
    const T s2p = P.at(s + n3, 0, 1, 0), s2m = P.at(s + n3, 0, -1, 0);
    const T s3p = P.at(s + 2 * n3, 0, 0, 1), s3m = P.at(s + 2 * n3, 0, 0, -1);
    T ef = (s1p + s2p + s3p - s1m - s2m - s3m) / T(2);
    ef = ef + P.at(tmp, 0, 0, 0);
    const unsigned g = P.at(flag, 0, 0, 1);
    T dm = T(1);
    if (g & 1u) {
      dm = ef > T(0) ? -T(2) : (ef < T(0) ? T(2) : T(0));
      ef = -T(2) * fabs(ef);
    }
    if (g & 2u) {
      if (!(ef > T(0))) dm = T(0);
      ef = dmax(T(0.), ef);
    }
    if (!(ef < T(1.) / dtaumesh && ef > -T(1.) / dtaumesh)) dm = T(0);
    ef = dmin(T(1.) / dtaumesh, ef);
    ef = dmax(-T(1.) / dtaumesh, ef);
    P.put(eflux, ef);
    if (gate) P.put(gate, dm);
    fhi = stat_op<1>(fhi, (double)(ef * dtold));
    flo = stat_op<2>(flo, (double)(ef * dtold));
  }
  block_stat<1>(fhi, part, 0);
  block_stat<2>(flo, part, 1);
}

// Step 5 of calcdefp: compression limiter source (mmh/limiter.f90:425-533).  lim = tlim where
// lambda_min(I + H(def) + dtold*H(defp)) < 1/cmpmax; part: per workgroup ncompress, cmax.
template <class T>
__global__ __launch_bounds__(256) void k_complim(T* __restrict__ lim, const T* __restrict__ defp, const T* __restrict__ def,
                                                 int n, T dtold, T cmpmaxglobal, T pi, double* __restrict__ part) {
  double c0 = 0.0, c1 = 0.0;
  const i64 chunk0 = (i64)xcd_remap(blockIdx.x, gridDim.x) * LIM_PT;
  for (int q = 0; q < LIM_PT; ++q) {
    const PlanePoint P(n, chunk0 + q);
    Hs<T> hp = hess(defp, P), hd = hess(def, P);
    T pxx = hp.xx * dtold, pyy = hp.yy * dtold, pzz = hp.zz * dtold;
    T pxy = hp.xy * dtold, pyz = hp.yz * dtold, pxz = hp.xz * dtold;
    pxx = pxx + hd.xx; pyy = pyy + hd.yy; pzz = pzz + hd.zz;
    pxy = pxy + hd.xy; pyz = pyz + hd.yz; pxz = pxz + hd.xz;
    T compression = compression_of(T(1) + pxx, pxy, pxz, T(1) + pyy, pyz, T(1) + pzz, pi);
    T cmpmax = cmpmaxglobal * T(1);
    T tlim = T(3) * (T(1) / cmpmax - T(1) / compression) / dtold;
    T v = T(0.);
    if (tlim > T(0)) { v = tlim; c0 += 1.0; }
    P.put(lim, v);
    c1 = stat_op<1>(c1, (double)compression);
  }
  block_stat<0>(c0, part, 0);
  block_stat<1>(c1, part, 1);
}

// The compression limiter's correction x (its inverse transform, unnormalised): v = x 2 / n / n / n
// (mmh/limiter.f90:579,592) is added to defp and stored in tmp2, leading dimension n + 2
// (limiter.f90:43).  1 / n is exact (n a power of two), so each product rounds as the division does.
template <class T>
__global__ void k_limit_apply(T* __restrict__ defp, T* __restrict__ tmp2, const T* __restrict__ x, int n, i64 n3) {
  const i64 p = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n3) return;
  const T rn = T(1) / T(n);
  const T v = x[p] * T(2.) * rn * rn * rn;
  defp[p] = defp[p] + v;
  const i64 i = p & (n - 1), r = p >> __builtin_ctz(n);
  tmp2[i + (i64)(n + 2) * r] = v;
}

template <class T> __global__ void k_add(T* __restrict__ y, const T* __restrict__ x, i64 n3) {
  const i64 p = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n3) y[p] = y[p] + x[p];
}

// ------------------------------------------------------------------------------------------------
// relaxing-TVD (mmh/relaxing.f90), whole-volume two-stage form.  Each stage is two passes: the
// fluxes of every point (k_tvd_flux, pointwise in the fluid), then the limited differences along the
// three axes (k_tvd_march).  The fluid is held as 5 fields (SoA) between the passes; the caller's
// interleaved array is read by the first flux pass and updated by the last march.  The metric is
// recomputed from def in both flux passes (its 7 fields cost more to store and read than their
// arithmetic).  Memory bound: 28 + 26 + 23 + 31 words per point for the four passes.

// Fluxes (910-996 with fluxeuler 999-1063): V[(d*5 + l)*n3 + p] = (vt_d / c) for component l, stored
// already divided by c, which is how dpv consumes it (326, 400, 444).  FIRST: the fluid is the
// caller's u(5, ...), copied into U, and the freezing speed c (cflkeuler, 1067-1139) is formed and
// stored; otherwise the fluid is U and c is read.  n is a power of two, n^2 a multiple of 256, so a
// workgroup's points lie in one plane: plane bases are scalars and a lane adds its offset in the plane.
// 512^3 FP32: 3.77 ms first, 2.70 ms second (4.0-4.5 TB/s); 256^3 FP64: 0.89, 0.71 ms.
template <class T, bool FIRST>
__global__ __launch_bounds__(256) void k_tvd_flux(T* __restrict__ V, T* __restrict__ U, T* __restrict__ c,
                                                  const T* __restrict__ u, const T* __restrict__ def,
                                                  const T* __restrict__ defp, int n) {
  const PlanePoint P(n, blockIdx.x);
  const i64 n3 = (i64)1 << (3 * P.lg), pl = P.pl;
  const uint32_t o = P.r * (uint32_t)sizeof(T);
  // b = adj(A) / det, A = I + H (882-901)
  const Hs<T> h = hess(def, P);
  const T a12 = h.xy, a23 = h.yz, a13 = h.xz;
  const T a11 = T(1) + h.xx, a22 = T(1) + h.yy, a33 = T(1) + h.zz;
  const T rg = a11 * a22 * a33 + T(2) * a12 * a13 * a23 - (a13 * a13) * a22 - a11 * (a23 * a23) - (a12 * a12) * a33;
  const T B1 = (a22 * a33 - a23 * a23) / rg;
  const T B2 = (a13 * a23 - a12 * a33) / rg;
  const T B3 = (a12 * a23 - a13 * a22) / rg;
  const T B4 = (a11 * a33 - a13 * a13) / rg;
  const T B5 = (a12 * a13 - a11 * a23) / rg;
  const T B6 = (a11 * a22 - a12 * a12) / rg;
  const T pdx = (P.at(defp, 1, 0, 0) - P.at(defp, -1, 0, 0)) / T(2);
  const T pdy = (P.at(defp, 0, 1, 0) - P.at(defp, 0, -1, 0)) / T(2);
  const T pdz = (P.at(defp, 0, 0, 1) - P.at(defp, 0, 0, -1)) / T(2);
  T ul[5];
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    if constexpr (FIRST) ul[l] = *(const T*)((const char*)(u + 5 * pl) + (5u * o + (uint32_t)(l * sizeof(T))));
    else ul[l] = *(const T*)((const char*)(U + l * n3 + pl) + o);
  }
  const T gamma = T(5.) / T(3.);
  T cp;
  if constexpr (FIRST) {
#pragma unroll
    for (int l = 0; l < 5; ++l) P.put(U + l * n3, ul[l]);
    const T vx = ul[1] / ul[0], vy = ul[2] / ul[0], vz = ul[3] / ul[0];
    const T rho = ul[0] / rg;
    const T kin = rho * (vx * vx + vy * vy + vz * vz) / T(2);
    const T ed = ul[4] / rg - kin;
    const T pressure = (gamma - T(1)) * ed;
    const T cs = sqrt(gamma * fabs(pressure / rho));
    const T v1 = vx - pdx, v2 = vy - pdy, v3 = vz - pdz;
    const T vv1 = B1 * v1 + B2 * v2 + B3 * v3;
    const T vv2 = B2 * v1 + B4 * v2 + B5 * v3;
    const T vv3 = B3 * v1 + B5 * v2 + B6 * v3;
    const T blim1 = cs * sqrt(B1 * B1 + B2 * B2 + B3 * B3) + fabs(vv1);
    const T blim2 = cs * sqrt(B2 * B2 + B4 * B4 + B5 * B5) + fabs(vv2);
    const T blim3 = cs * sqrt(B3 * B3 + B5 * B5 + B6 * B6) + fabs(vv3);
    cp = dmax(dmax(blim1, blim2), blim3);
    P.put(c, cp);
  } else {
    cp = *(const T*)((const char*)(c + pl) + o);
  }
  const T rho = ul[0] / rg, mx = ul[1] / rg, my = ul[2] / rg, mz = ul[3] / rg;
  const T vx = mx / rho, vy = my / rho, vz = mz / rho;
  const T engy = ul[4] / rg;
  const T kinetic = rho * (vx * vx + vy * vy + vz * vz) / T(2);
  T pressure = (gamma - T(1)) * (engy - kinetic);
  pressure = dmax(T(0.), pressure);
  const T econv = engy + pressure;
  const T v1[3][5] = {{mx, mx * vx + pressure, my * vx, mz * vx, econv * vx},
                      {my, mx * vy, my * vy + pressure, mz * vy, econv * vy},
                      {mz, mx * vz, my * vz, mz * vz + pressure, econv * vz}};
  const T pdxg = pdx / rg, pdyg = pdy / rg, pdzg = pdz / rg;
  const T b11 = B1 * rg, b12 = B2 * rg, b13 = B3 * rg;
  const T b22 = B4 * rg, b23 = B5 * rg, b33 = B6 * rg;
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    const T ulv = ul[l];
    const T vtt1 = v1[0][l] - ulv * pdxg;
    const T vtt2 = v1[1][l] - ulv * pdyg;
    const T vtt3 = v1[2][l] - ulv * pdzg;
    P.put(V + (0 * 5 + l) * n3, (b11 * vtt1 + b12 * vtt2 + b13 * vtt3) / cp);
    P.put(V + (1 * 5 + l) * n3, (b12 * vtt1 + b22 * vtt2 + b23 * vtt3) / cp);
    P.put(V + (2 * 5 + l) * n3, (b13 * vtt1 + b23 * vtt2 + b33 * vtt3) / cp);
  }
}

// base + minmod(a, b)/2 (neg: base - minmod(b, a)/2), the limiter of wphalfx (514-516) with wslopelim =
// 1.5, wbee = 1 (mmh/relaxgl.f90:8): (sign a + sign b) m / 2 with m = min(1.5 x, y + 0 x), x and y
// the smaller and larger of |a|, |b|.  The sign factor is chosen from the sign bits (0 or +-1/2) and the
// multiply-adds are explicit where the product is exact, so this rounds, and passes on
// infinities and NaN, as the plain expression does.  Halvings are exact on normal numbers: below 2^-125 in
// FP32 (2^-1021) the plain form rounds halves that this form keeps, by a subnormal step at most, and
// doubled values overflow one binade sooner.
__device__ __forceinline__ float half_sign(float a, float b) {
  const int sa = __float_as_int(a), sb = __float_as_int(b);
  return (sa ^ sb) < 0 ? 0.f : __int_as_float((sa & (int)0x80000000) | 0x3f000000);
}
__device__ __forceinline__ double half_sign(double a, double b) {
  const int sa = __double2hiint(a), sb = __double2hiint(b);
  return __hiloint2double((sa ^ sb) < 0 ? 0 : ((sa & (int)0x80000000) | 0x3fe00000), 0);
}
template <bool NEG, class T> __device__ __forceinline__ T limited(T base, T a, T b) {
  const T aa = fabs(a), ab = fabs(b);
  const T x = dmin(aa, ab), y = dmax(aa, ab);
  const T m = dmin(T(1.5) * x, __builtin_elementwise_fma(T(0), x, y));
  const T h = half_sign(a, b);
  return __builtin_elementwise_fma(NEG ? -h : h, m, base);
}

// dpv (269-496) + stepu/stepuu (774-837): out = base - res(U, V, c)*dt.  A workgroup takes a tile of
// TI x 256/TI columns (TI = min(64, n)) and walks KS planes.  With A = u + v and B = u - v the flux
// through the face after point q of a line is (ap(q) - bp(q+1))/2, ap and bp the limited values of
// wphalf (502-560) at one point (all doubled: the halvings of wphalf are exact and taken together
// in the face weights w = (c + c')/4): along z each is formed once and carried in registers with the
// plane's A, B and differences, so a step loads one new plane for z; the in-plane neighbours
// are read at unit stride and mostly hit the caches.  One thread per point reading all 15 + 13
// neighbours, the fluid interleaved, ran at 0.8 TB/s.
// LAST: out is the caller's interleaved u, updated in place; otherwise 5 fields, from U.
// 512^3 FP32: 4.8 ms, LAST 5.6 ms, against 20.3 ms for that kernel; 256^3 FP64: 1.44, 1.67 ms against
// 4.45 ms (2.4-2.9 TB/s: about 1000 vector instructions per point are as long as the memory time).
// Four waves per SIMD at least: the FP64 form would take 3 (at 132 registers), 4 % slower.
template <class T, bool LAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tvd_march(T* __restrict__ out, const T* __restrict__ U, const T* __restrict__ V,
                                                   const T* __restrict__ c, int n, T dt, int KS) {
  const int lg = __builtin_ctz(n), m = n - 1;
  const i64 n3 = (i64)1 << (3 * lg);
  const int lti = lg < 6 ? lg : 6, TI = 1 << lti, TJ = 256 >> lti;
  const int tpr = n >> lti, tiles = tpr * (n / TJ);  // tiles of a row of tiles, and of a plane
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(b % (unsigned)tiles), k0 = (int)(b / (unsigned)tiles) * KS;
  const int i = (tile % tpr) * TI + ((int)threadIdx.x & (TI - 1)), j = (tile / tpr) * TJ + ((int)threadIdx.x >> lti);
  const uint32_t z = sizeof(T);
  const uint32_t o0 = (uint32_t)(i + (j << lg)) * z;
  const uint32_t oip = (uint32_t)(((i + 1) & m) + (j << lg)) * z, oipp = (uint32_t)(((i + 2) & m) + (j << lg)) * z;
  const uint32_t oim = (uint32_t)(((i - 1) & m) + (j << lg)) * z, oimm = (uint32_t)(((i - 2) & m) + (j << lg)) * z;
  const uint32_t ojp = (uint32_t)(i + (((j + 1) & m) << lg)) * z, ojpp = (uint32_t)(i + (((j + 2) & m) << lg)) * z;
  const uint32_t ojm = (uint32_t)(i + (((j - 1) & m) << lg)) * z, ojmm = (uint32_t)(i + (((j - 2) & m) << lg)) * z;
  auto ld = [](const T* base, uint32_t off) -> T { return *(const T*)((const char*)base + off); };
  auto plane = [&](int k) { return (i64)(k & m) << (2 * lg); };
  T A[5] = {}, B[5] = {}, dA[5] = {}, dB[5] = {}, ap[5] = {}, fl[5] = {};
  T ckm, ck = ld(c + plane(k0 - 1), o0), ckp = ld(c + plane(k0), o0);
  // plane s of component l enters the z pipeline; returns the flux through the face s-2 | s-1
  auto enter = [&](int l, int s, uint32_t o) -> T {
    const T us = ld(U + l * n3 + plane(s), o), vs = ld(V + (10 + l) * n3 + plane(s), o);
    const T An = us + vs, Bn = us - vs;
    const T dAn = An - A[l], dBn = Bn - B[l];
    const T apn = limited<false>(A[l], dA[l], dAn);
    const T bpn = limited<true>(B[l], dBn, dB[l]);
    const T fln = ap[l] - bpn;
    A[l] = An; B[l] = Bn; dA[l] = dAn; dB[l] = dBn; ap[l] = apn;
    return fln;
  };
  for (int s = k0 - 2; s < k0 + 2; ++s)
#pragma unroll
    for (int l = 0; l < 5; ++l) fl[l] = enter(l, s, o0);
  for (int k = k0; k < k0 + KS; ++k) {
    // The lane offsets pass through empty asm so that each load of the step takes the form scalar base +
    // 32-bit lane offset: hoisted out of the loop as 64-bit values they cost an address add per load.
    uint32_t q0 = o0, qip = oip, qipp = oipp, qim = oim, qimm = oimm, qjp = ojp, qjpp = ojpp, qjm = ojm, qjmm = ojmm;
    asm volatile("" : "+v"(q0), "+v"(qip), "+v"(qipp), "+v"(qim), "+v"(qimm), "+v"(qjp), "+v"(qjpp), "+v"(qjm), "+v"(qjmm));
    const T* cpl = c + plane(k);
    ckm = ck; ck = ckp; ckp = ld(c + plane(k + 1), q0);
    const T wzp = (ckp + ck) * T(0.25), wzm = (ck + ckm) * T(0.25);
    const T wxp = (ld(cpl, qip) + ck) * T(0.25), wxm = (ck + ld(cpl, qim)) * T(0.25);
    const T wyp = (ld(cpl, qjp) + ck) * T(0.25), wym = (ck + ld(cpl, qjm)) * T(0.25);
    // the caller's five values of the point, adjacent in memory: one wide read here, one write at the end
    T w[5];
    T* wp = (T*)((char*)(out + 5 * plane(k)) + 5u * q0);
    if constexpr (LAST)
#pragma unroll
      for (int l = 0; l < 5; ++l) w[l] = wp[l];
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      const T fln = enter(l, k + 2, q0);
      T r = wzp * fln - wzm * fl[l];
      fl[l] = fln;
      const T* Up = U + l * n3 + plane(k);
      const T u0 = ld(Up, q0);
      // fluxes through the two faces of the point along one axis
      auto faces = [&](const T* Vp, uint32_t omm, uint32_t om, uint32_t op, uint32_t opp, T& fp, T& fm) {
        const T umm = ld(Up, omm), um = ld(Up, om), up = ld(Up, op), upp = ld(Up, opp);
        const T vmm = ld(Vp, omm), vm = ld(Vp, om), v0 = ld(Vp, q0), vp = ld(Vp, op), vpp = ld(Vp, opp);
        const T Amm = umm + vmm, Am = um + vm, A0 = u0 + v0, Ap = up + vp;
        const T Bm = um - vm, B0 = u0 - v0, Bp = up - vp, Bpp = upp - vpp;
        const T dAm = Am - Amm, dA0 = A0 - Am, dA1 = Ap - A0;
        const T dB0 = B0 - Bm, dB1 = Bp - B0, dB2 = Bpp - Bp;
        fp = limited<false>(A0, dA0, dA1) - limited<true>(Bp, dB2, dB1);
        fm = limited<false>(Am, dAm, dA0) - limited<true>(B0, dB1, dB0);
      };
      T xp, xm, yp, ym;
      faces(V + l * n3 + plane(k), qimm, qim, qip, qipp, xp, xm);
      r = r + wxp * xp - wxm * xm;
      faces(V + (5 + l) * n3 + plane(k), qjmm, qjm, qjp, qjpp, yp, ym);
      r = r + wyp * yp - wym * ym;
      if constexpr (LAST) w[l] = w[l] - r * dt;
      else *(T*)((char*)(out + l * n3 + plane(k)) + q0) = u0 - r * dt;
    }
    if constexpr (LAST)
#pragma unroll
      for (int l = 0; l < 5; ++l) wp[l] = w[l];
  }
}

}  // namespace mmh
