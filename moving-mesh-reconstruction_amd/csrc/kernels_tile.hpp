// kernels_tile.hpp -- a whole Gauss-Seidel sweep of a small level in one launch.
//
// A colour launch of a 32^3 level is a few hundred nanoseconds of work and 3.6 us of launch, and eight of
// them are a sweep.  Here a workgroup owns a tile of 8 x 8 x TK points and sweeps all eight colours on
// the tile plus a halo, from the level's old values, in LDS: a colour reads what earlier colours of the
// sweep left one point away, so values near the region's rim go wrong, further in with each colour, by
// at most 4 points in i, 6 in j and 2 in k (the longest chains of the colour order k, i, j).  The
// halo is that wide, so the tile's own values are those of the eight launches, bit for bit.  Workgroups
// never wait for each other: old values come from one buffer and new ones go to another.  The region's
// metric is staged in LDS too (each value is read by up to three updates, and from memory a
// wavefront's 8 x 8 cells are eight lines per load).
// The halo costs 15 updates per point kept (TK = 2), bound by vector instructions, so this pays only
// where launches are the cost.  Measured per sweep: 32^3 FP32 25.8 -> 7.2 us, FP64 29.9 -> 8.0 us (TK = 4:
// 7.8, 8.3; 8: 9.8); 64^3 FP32 23.9 us at best (TK = 8) against 25.4 and FP64 39 against 30, so only 32^3
// is swept this way.
#pragma once
#include "kernels.hpp"
#include "kernels_coarse16.hpp"

namespace mmh {

template <int TK, bool GAL = false> struct TileShape {
  static constexpr int HI = 4, HJ = GAL ? 8 : 6, HK = 2;             // halo, in points
  static constexpr int CI = 4 + HI, CJ = 4 + HJ, CK = (TK + 2 * HK) / 2;  // region, in 2x2x2 cells
  static constexpr int CELLS = CI * CJ * CK;                          // one per thread
  static constexpr int NT = (CELLS + 63) / 64 * 64;
};

// out = one sweep of `in` (sub-lattice layout, n a multiple of 8), colours reversed with REV.
template <class T, class TG, bool REV, int TK>
__global__ __launch_bounds__((TileShape<TK>::NT)) void k_sweep_tile(T* __restrict__ out, const T* __restrict__ in,
                                                                 const T* __restrict__ rhs, const TG* __restrict__ G,
                                                                 int n, T dx2) {
  using S = TileShape<TK>;
  constexpr int CI = S::CI, CJ = S::CJ, CELLS = S::CELLS;
  __shared__ T u[8 * CELLS];
  __shared__ T g[6 * 8 * CELLS];
  const int h = n >> 1, hm = h - 1, lg = __builtin_ctz(h), h3 = h * h * h, nt = n >> 3;
  const int b = (int)xcd_remap(blockIdx.x, gridDim.x);
  const int bi = b % nt, bj = (b / nt) % nt, bk = b / (nt * nt);
  const int t = threadIdx.x, ci = t % CI, cj = (t / CI) % CJ, ck = t / (CI * CJ);
  const int gi = 4 * bi - S::HI / 2 + ci, gj = 4 * bj - S::HJ / 2 + cj, gk = TK / 2 * bk - S::HK / 2 + ck;
  // the thread's cell within a class of the level, as a byte offset (threads past the region's cells
  // wrap to some cell too, and use nothing)
  const uint32_t q = (uint32_t)((gi & hm) + ((gj & hm) << lg) + ((gk & hm) << (2 * lg)));
  auto cls = [](const T* a, i64 o, uint32_t x) -> T { return *(const T*)((const char*)(a + o) + x * (uint32_t)sizeof(T)); };
  auto clg = [](const TG* a, i64 o, uint32_t x) -> T {
    return gl<T>((const TG*)((const char*)(a + o) + x * (uint32_t)sizeof(TG)), 0);
  };
  const bool cell = t < CELLS;
  T b2[8];
  {
    T v[8], w[6];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = cls(in, (i64)c * h3, q);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int f = 0; f < 6; ++f) w[f] = clg(G, (i64)(f * 8 + c) * h3, q);
      b2[c] = cls(rhs, (i64)c * h3, q) * dx2;
      if (cell)
#pragma unroll
        for (int f = 0; f < 6; ++f) g[(f * 8 + c) * CELLS + t] = w[f];
    }
    if (cell)
#pragma unroll
      for (int c = 0; c < 8; ++c) u[c * CELLS + t] = v[c];
  }
  __syncthreads();
  // a point on the region's rim (no neighbour beyond it) keeps its old value
  const bool lo[3] = {ci == 0, cj == 0, ck == 0}, hi[3] = {ci == CI - 1, cj == CJ - 1, ck == S::CK - 1};
  auto colour = [&](auto cc) {
    constexpr int c = decltype(cc)::value;
    const bool rim = ((c & 1) ? hi[0] : lo[0]) || ((c & 2) ? hi[1] : lo[1]) || ((c & 4) ? hi[2] : lo[2]);
    if (!cell || rim) return;
    // index, among the region's class arrays, of the point's neighbour
    auto nb = [&](int sx, int sy, int sz) -> int {
      return class16(c, sx, sy, sz) * CELLS + t + (shift16(c & 1, sx) - 1) + CI * (shift16((c >> 1) & 1, sy) - 1) +
             CI * CJ * (shift16(c >> 2, sz) - 1);
    };
    int o[18];
#pragma unroll
    for (int e = 0; e < 18; ++e) o[e] = nb(NB19[e][0], NB19[e][1], NB19[e][2]);
    T p[18], w[7], x[12], t1, t2;
#pragma unroll
    for (int e = 0; e < 18; ++e) p[e] = u[o[e]];
    faces19<T>(w, g, 8 * CELLS, c * CELLS + t, o);
#pragma unroll
    for (int e = 0; e < 12; ++e) x[e] = g[XG19[e][1] * 8 * CELLS + o[XG19[e][0]]];
    terms19<T>(t1, t2, w, x, p);
    u[c * CELLS + t] = (b2[c] - t1 - t2) / w[6];
  };
  // classes 3 and 4 (the fourth and fifth colour) are not coupled: no barrier between them
#define TILE_C(C) colour(std::integral_constant<int, C>())
  if constexpr (!REV) {
    TILE_C(0); __syncthreads(); TILE_C(2); __syncthreads(); TILE_C(1); __syncthreads();
    TILE_C(3); TILE_C(4); __syncthreads(); TILE_C(6); __syncthreads(); TILE_C(5); __syncthreads(); TILE_C(7);
  } else {
    TILE_C(7); __syncthreads(); TILE_C(5); __syncthreads(); TILE_C(6); __syncthreads();
    TILE_C(4); TILE_C(3); __syncthreads(); TILE_C(1); __syncthreads(); TILE_C(2); __syncthreads(); TILE_C(0);
  }
#undef TILE_C
  const int ti = ci - S::HI / 2, tj = cj - S::HJ / 2, tk = ck - S::HK / 2;
  if (cell && ti >= 0 && ti < 4 && tj >= 0 && tj < 4 && tk >= 0 && tk < TK / 2)
#pragma unroll
    for (int c = 0; c < 8; ++c) *(T*)((char*)(out + (i64)c * h3) + q * (uint32_t)sizeof(T)) = u[c * CELLS + t];
}

// The same for a 27-point (Galerkin) level, whose classes are all coupled: 8 points of halo in j.  Its 27
// coefficients per point stay in memory; a colour's are loaded while the colour before it is updated.
// Per sweep of 32^3 FP64 36 -> 14 us, FP32 with
// bfloat16 coefficients 32 -> 8.4 us; 64^3 takes 34 us at best (TK = 8), as the launches do, so only 32^3 is
// swept this way.
template <class T, class TG, bool REV, int TK>
__global__ __launch_bounds__((TileShape<TK, true>::NT)) void k_sweep_tile_gal(T* __restrict__ out, const T* __restrict__ in,
                                                                            const T* __restrict__ rhs,
                                                                            const TG* __restrict__ A, int n) {
  using S = TileShape<TK, true>;
  constexpr int CI = S::CI, CJ = S::CJ, CELLS = S::CELLS;
  __shared__ T u[8 * CELLS];
  const int h = n >> 1, hm = h - 1, lg = __builtin_ctz(h), h3 = h * h * h, nt = n >> 3;
  const int b = (int)xcd_remap(blockIdx.x, gridDim.x);
  const int bi = b % nt, bj = (b / nt) % nt, bk = b / (nt * nt);
  const int t = threadIdx.x, ci = t % CI, cj = (t / CI) % CJ, ck = t / (CI * CJ);
  const int gi = 4 * bi - S::HI / 2 + ci, gj = 4 * bj - S::HJ / 2 + cj, gk = TK / 2 * bk - S::HK / 2 + ck;
  const uint32_t q = (uint32_t)((gi & hm) + ((gj & hm) << lg) + ((gk & hm) << (2 * lg)));
  const uint32_t qt = q * (uint32_t)sizeof(T), qg = q * (uint32_t)sizeof(TG);
  const bool cell = t < CELLS;
  if (cell)
#pragma unroll
    for (int c = 0; c < 8; ++c) u[c * CELLS + t] = *(const T*)((const char*)(in + (i64)c * h3) + qt);
  const bool lo[3] = {ci == 0, cj == 0, ck == 0}, hi[3] = {ci == CI - 1, cj == CJ - 1, ck == S::CK - 1};
  T a[27], bn;
  auto load = [&](int c) {
    if constexpr (std::is_same<TG, bf16x2>::value) {
#pragma unroll
      for (int f = 0; f < 14; ++f) {
        const unsigned w = ((const TG*)((const char*)(A + (i64)(f * 8 + c) * h3) + qg))->w;
        a[2 * f] = bf16_lo(w);
        if (2 * f + 1 < 27) a[2 * f + 1] = bf16_hi(w);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 27; ++e) a[e] = *(const T*)((const char*)(A + (i64)(e * 8 + c) * h3) + qg);
    }
    bn = *(const T*)((const char*)(rhs + (i64)c * h3) + qt);
  };
  load(REV ? 7 : 0);
  __syncthreads();
  auto colour = [&](auto cc, int next) {
    constexpr int c = decltype(cc)::value;
    T w[27];
    const T bc = bn;
#pragma unroll
    for (int e = 0; e < 27; ++e) w[e] = a[e];
    if (next >= 0) load(next);
    const bool rim = ((c & 1) ? hi[0] : lo[0]) || ((c & 2) ? hi[1] : lo[1]) || ((c & 4) ? hi[2] : lo[2]);
    if (cell && !rim) {
      T p[27], s = T(0);
#pragma unroll
      for (int e = 0; e < 27; ++e) {
        const int sx = e % 3 - 1, sy = e / 3 % 3 - 1, sz = e / 9 - 1;
        p[e] = u[class16(c, sx, sy, sz) * CELLS + t + (shift16(c & 1, sx) - 1) + CI * (shift16((c >> 1) & 1, sy) - 1) +
                 CI * CJ * (shift16(c >> 2, sz) - 1)];
      }
#pragma unroll
      for (int e = 0; e < 27; ++e)
        if (e != 13) s = s + w[e] * p[e];
      u[c * CELLS + t] = (bc - s) / w[13];
    }
    __syncthreads();
  };
#define TILE_C(C, N) colour(std::integral_constant<int, C>(), N)
  if constexpr (!REV) {
    TILE_C(0, 2); TILE_C(2, 1); TILE_C(1, 3); TILE_C(3, 4); TILE_C(4, 6); TILE_C(6, 5); TILE_C(5, 7); TILE_C(7, -1);
  } else {
    TILE_C(7, 5); TILE_C(5, 6); TILE_C(6, 4); TILE_C(4, 3); TILE_C(3, 1); TILE_C(1, 2); TILE_C(2, 0); TILE_C(0, -1);
  }
#undef TILE_C
  const int ti = ci - S::HI / 2, tj = cj - S::HJ / 2, tk = ck - S::HK / 2;
  if (cell && ti >= 0 && ti < 4 && tj >= 0 && tj < 4 && tk >= 0 && tk < TK / 2)
#pragma unroll
    for (int c = 0; c < 8; ++c) *(T*)((char*)(out + (i64)c * h3) + qt) = u[c * CELLS + t];
}

}  // namespace mmh
