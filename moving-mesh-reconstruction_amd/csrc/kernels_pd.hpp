// kernels_pd.hpp -- particle to grid density assignment of haloden.f90 (mmh's input generation
// from N-body particles): nearest-grid-point counting plus a nearest-particle fill of empty cells,
// each particle's unit mass shared equally between its own cell and the empty cells it fills.
#pragma once
#include "kernels.hpp"

namespace mmh {

// Position of particle p in grid units and its cell (haloden.f90:84-99): x = modulo(x, nf) * ng / nf,
// cell = floor(x) (0-based; clamped to ng-1 where the scaled position rounds up to ng, and to 0).
__global__ void k_pd_cells(float* __restrict__ xs, int* __restrict__ cell, int* __restrict__ idx,
                           const float* __restrict__ xp, i64 np, int ng, float nf) {
  const i64 p = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  int c[3];
  for (int d = 0; d < 3; ++d) {
    float x = xp[3 * p + d];
    x = x - floorf(x / nf) * nf;  // modulo(x, real(nf))
    x = x * (float)ng / nf;
    xs[3 * p + d] = x;
    c[d] = x >= 1.f ? (x < (float)ng ? (int)x : ng - 1) : 0;  // NaN: 0
  }
  cell[p] = c[0] + ng * (c[1] + ng * c[2]);
  idx[p] = (int)p;
}

// [start, end) of every non-empty cell in the cell-sorted particle list.
__global__ void k_pd_ranges(int* __restrict__ start, int* __restrict__ end, const int* __restrict__ key, i64 np) {
  const i64 q = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  const int k = key[q];
  if (q == 0 || key[q - 1] != k) start[k] = (int)q;
  if (q == np - 1 || key[q + 1] != k) end[k] = (int)q + 1;
}

// Scaled positions in cell order: xo[q] = position and index of particle order[q].  *out is set if any lies
// outside [0, ng] (coordinates some 2^23 boxes out, whose modulo in FP32 has lost the fraction), or is NaN.
__global__ void k_pd_sorted(float4* __restrict__ xo, int* __restrict__ out, const int* __restrict__ order,
                            const float* __restrict__ xs, i64 np, float fng) {
  const i64 q = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  const int p = order[q];
  const float x = xs[3 * (i64)p], y = xs[3 * (i64)p + 1], z = xs[3 * (i64)p + 2];
  xo[q] = make_float4(x, y, z, __int_as_float(p));
  auto in = [fng](float v) { return v >= 0.f && v <= fng; };
  if (!(in(x) && in(y) && in(z))) *out = 1;  // every writer stores the same value
}

// Occupancy bits, a row of words per (j, k): bit x + 32 of a row is set if cell x (periodic, from -32 to
// past ng + 31) holds a particle, so any run of up to 32 cells around a cell is two words.
__host__ __device__ inline int pd_row_words(int ng) { return (ng + 64 + 31) / 32 + 1; }
// One thread per bit, a wavefront per two words.
__global__ __launch_bounds__(256) void k_pd_bits(unsigned* __restrict__ bits, const int* __restrict__ start,
                                                 const int* __restrict__ end, int ng, i64 nwords) {
  const i64 w = ((i64)blockIdx.x * blockDim.x + threadIdx.x) >> 5;
  bool on = false;
  if (w < nwords) {
    const int rw = pd_row_words(ng);
    const i64 row = w / rw;
    int x = (int)(w - row * rw) * 32 - 32 + (int)(threadIdx.x & 31);
    while (x < 0) x += ng;
    x %= ng;
    on = end[row * ng + x] > start[row * ng + x];
  }
  const uint64_t m = __ballot(on);
  if (w < nwords && (threadIdx.x & 31) == 0) bits[w] = (unsigned)(m >> (threadIdx.x & 32));
}

// near[r - 1]: the bits or-ed over the (2r + 1)^2 rows around each row, r = 1 .. PD_NEAR: one window of it
// tells whether a cube holds any particle.
constexpr int PD_NEAR = 4;
__global__ __launch_bounds__(256) void k_pd_bits_near(unsigned* __restrict__ near, const unsigned* __restrict__ bits, int ng,
                                                      i64 nwords) {
  const i64 w = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nwords) return;
  const int rw = pd_row_words(ng);
  const i64 row = w / rw;
  const int x = (int)(w - row * rw), k = (int)(row / ng), j = (int)(row - (i64)k * ng);
  unsigned o[PD_NEAR + 1] = {};
#pragma unroll
  for (int dk = -PD_NEAR; dk <= PD_NEAR; ++dk)
#pragma unroll
    for (int dj = -PD_NEAR; dj <= PD_NEAR; ++dj) {
      const int aj = dj < 0 ? -dj : dj, ak = dk < 0 ? -dk : dk;
      const int kk = (k + dk + PD_NEAR * ng) % ng, jj = (j + dj + PD_NEAR * ng) % ng;
      o[aj > ak ? aj : ak] |= bits[((i64)kk * ng + jj) * rw + x];
    }
#pragma unroll
  for (int r = 1; r <= PD_NEAR; ++r) {
    o[r] |= o[r - 1];
    near[(r - 1) * nwords + w] = o[r];
  }
}

// Nearest particle of every empty cell (haloden.f90:119-167): cubes of growing half-width r
// around the cell are scanned in (k, j, i) order, each cell's particles in the reference's
// linked-list order (newest first, i.e. decreasing index); the first particle with the smallest
// periodic squared distance to the cell centre wins, and the scan stops after the first cube that
// holds any particle.  near[c] = particle index, or -1 for a non-empty cell; wp[p] counts cells.
// Bound by vector instructions and the divergence of a wavefront's cells.  A cube's row of 2r + 1 cells is
// one window of the occupancy bits (r <= 15; wider cubes go cell by cell); one window of the or-ed
// rows tells that a cube of r <= 4 is empty; the 27 cells of r = 1 are one mask; and the cells that
// need r >= 2 (13 %) go to a pass of their own.  200^3 cells, 10^6 particles: 2450 us with start and
// end of every cell read in turn, 907 with the windows, 706 with the or-ed rows, 385 + 151 us in two
// passes.
struct PdSearch {
  const int* start;
  const int* end;
  const float4* xo;
  const unsigned* bits;
  const unsigned* near;  // bits_near, nwords per level
  const int* out;        // whether any position lies outside [0, ng]: the search is k_pd_far's alone
  i64 nwords;
  int ng, rmax;
};

// The empty cell c's particle, searched from half-width r0 on (FIRST: only r = 1; -1 if its cube is empty).
// OUT: positions may lie outside [0, ng].
template <bool FIRST, bool OUT = false> __device__ __forceinline__ int pd_search(const PdSearch& P, unsigned c, int r0) {
  const int ng = P.ng, rw = pd_row_words(ng);
  const unsigned row = c / (unsigned)ng;
  const int i = (int)(c - row * ng), k = (int)(row / (unsigned)ng), j = (int)(row - (unsigned)k * ng);
  // 1-based cell (i+1, j+1, k+1) has centre (i+1, j+1, k+1) - 0.5
  const float gx = (float)(i + 1) - 0.5f, gy = (float)(j + 1) - 0.5f, gz = (float)(k + 1) - 0.5f;
  const float half = (float)(ng / 2), fng = (float)ng;
  float r2min = (float)(1000 * ng * ng);
  int best = -1;
  auto scan_cell = [&](int cc) {
    const int q0 = P.start[cc];
    for (int q = P.end[cc] - 1; q >= q0; --q) {
      const float4 x = P.xo[q];
      float d[3] = {x.x - gx, x.y - gy, x.z - gz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        // modulo(dpos + ng/2, real(ng)) - ng/2: for positions in [0, ng] t lies in (-ng, 2 ng), where the
        // floor of the rounded t / ng is -1, 0 or 1 as t < 0, t < ng or not (a float below ng divides to
        // one below 1)
        const float t = d[a] + half;
        if constexpr (OUT) d[a] = (t - floorf(t / fng) * fng) - half;
        else d[a] = (t < 0.f ? t + fng : (t >= fng ? t - fng : t)) - half;
      }
      const float r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
      if (r2 < r2min) { r2min = r2; best = __float_as_int(x.w); }
    }
  };
  auto wrapped = [&](int x) -> int { return x < 0 ? x + ng : (x >= ng ? x - ng : x); };
  auto window = [&](int rj, int r) -> unsigned {  // cells i - r .. i + r of row rj
    const int x0 = i - r + 32;
    const unsigned* w = P.bits + rj * rw + (x0 >> 5);
    return (unsigned)((((uint64_t)w[1] << 32) | w[0]) >> ((unsigned)x0 & 31u)) & ((2u << (2 * r)) - 1u);
  };
  if constexpr (FIRST) {
    // the 27 cells in one mask, in scan order: one loop, as many steps as the fullest lane has cells
    const int xs[3] = {wrapped(i - 1), i, wrapped(i + 1)}, ys[3] = {wrapped(j - 1), j, wrapped(j + 1)};
    const int zs[3] = {wrapped(k - 1), k, wrapped(k + 1)};
    unsigned m = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q) m |= window(ys[q % 3] + ng * zs[q / 3], 1) << (3 * q);
    while (m) {
      const unsigned b = (unsigned)__builtin_ctz(m), rowb = (b * 11u) >> 5, dx = b - 3u * rowb;
      const unsigned dk = (rowb * 11u) >> 5, dj = rowb - 3u * dk;
      m &= m - 1u;
      const int x = dx == 0 ? xs[0] : (dx == 1 ? xs[1] : xs[2]), y = dj == 0 ? ys[0] : (dj == 1 ? ys[1] : ys[2]);
      const int z = dk == 0 ? zs[0] : (dk == 1 ? zs[1] : zs[2]);
      scan_cell(x + ng * (y + ng * z));
    }
    return best;
  }
  for (int r = r0; r <= P.rmax && best < 0; ++r) {
    if (r <= 15 && 2 * r < ng) {
      for (int ks = k - r; ks <= k + r; ++ks) {
        const int kk = wrapped(ks) * ng;
        for (int js = j - r; js <= j + r; ++js) {
          const int rj = wrapped(js) + kk;
          unsigned m = window(rj, r);
          while (m) {
            const int b = __builtin_ctz(m);
            m &= m - 1u;
            scan_cell(rj * ng + wrapped(i - r + b));
          }
        }
      }
      continue;
    }
    for (int ks = k - r; ks <= k + r; ++ks)
      for (int js = j - r; js <= j + r; ++js)
        for (int is = i - r; is <= i + r; ++is) {
          const int kk = ((ks % ng) + ng) % ng, jj = ((js % ng) + ng) % ng, ii = ((is % ng) + ng) % ng;
          scan_cell(ii + ng * (jj + ng * kk));
        }
  }
  return best;
}

// First pass over all cells, PD_CH x 256 of them per workgroup at most: -1 for the non-empty ones, the
// cells whose cube r = 1 holds a particle, and the others into far (their count in far[0]) for a second
// pass, where the wider searches fill whole wavefronts instead of a few lanes of each.  The list is
// gathered in LDS and takes one atomic of the workgroup: an atomic per wavefront on the one counter
// cost 1.2 ms at 200^3.
constexpr int PD_CH = 16;
__global__ __launch_bounds__(256) void k_pd_nearest(int* __restrict__ near, int* __restrict__ wp, int* __restrict__ far,
                                                    PdSearch P, int chunks) {
  __shared__ int list[PD_CH * 256];
  __shared__ int count, base;
  if (*P.out) return;
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  const unsigned ncell = (unsigned)P.ng * P.ng * P.ng;
  const int lane = threadIdx.x & 63, rw = pd_row_words(P.ng);
  for (int ch = 0; ch < chunks; ++ch) {
    // cell and word indices in 32 bits (ng <= 1024)
    const unsigned c = (blockIdx.x * (unsigned)chunks + (unsigned)ch) * 256u + threadIdx.x;
    const bool empty = c < ncell && P.end[c] <= P.start[c];
    bool wide = empty;
    int best = -1;
    if (empty && P.ng > 2) {
      const unsigned row = c / (unsigned)P.ng;
      const int x0 = (int)(c - row * P.ng) - 1 + 32;
      const unsigned* w = P.near + (int)row * rw + (x0 >> 5);
      wide = !((unsigned)((((uint64_t)w[1] << 32) | w[0]) >> ((unsigned)x0 & 31u)) & 7u);
      if (!wide) best = pd_search<true>(P, c, 1);
    }
    if (c < ncell) near[c] = best;
    if (wide) list[atomicAdd(&count, 1)] = (int)c;
    // neighbouring cells of a row often share their particle: one atomic per run of lanes
    const int before = __shfl_up(best, 1);
    const bool head = lane == 0 || best != before;
    const uint64_t heads = __ballot(head), after = lane == 63 ? 0 : heads >> (lane + 1);
    if (head && best >= 0) atomicAdd(&wp[best], after ? __builtin_ctzll(after) + 1 : 64 - lane);
  }
  __syncthreads();
  if (threadIdx.x == 0 && count) base = atomicAdd(&far[0], count);
  __syncthreads();
  for (int q = threadIdx.x; q < count; q += 256) far[1 + base + q] = list[q];
}

// Second pass, over far; or, where positions lie outside [0, ng] or are NaN (at no distance: a cube that
// holds no other particle does not end the search), the whole search.  A test beside the select in the search
// loops cost k_pd_nearest 5 % (18 us at 200^3), a launch of its own 5 us.
__global__ __launch_bounds__(256) void k_pd_far(int* __restrict__ near, int* __restrict__ wp, const int* __restrict__ far,
                                                PdSearch P) {
  if (*P.out) {
    const unsigned ncell = (unsigned)P.ng * P.ng * P.ng;
    for (unsigned c = blockIdx.x * 256u + threadIdx.x; c < ncell; c += gridDim.x * 256u) {
      int best = -1;
      if (P.end[c] <= P.start[c]) best = pd_search<false, true>(P, c, 1);
      near[c] = best;
      if (best >= 0) atomicAdd(&wp[best], 1);
    }
    return;
  }
  const int count = far[0];
  for (int q = blockIdx.x * 256 + threadIdx.x; q < count; q += gridDim.x * 256) {
    const unsigned c = (unsigned)far[1 + q];
    int r0 = P.ng > 2 ? 2 : 1;
    if (2 * PD_NEAR < P.ng) {
      const int rw = pd_row_words(P.ng);
      const unsigned row = c / (unsigned)P.ng;
      const int i = (int)(c - row * P.ng);
#pragma unroll
      for (int r = PD_NEAR; r >= 2; --r) {
        const int x0 = i - r + 32;
        const unsigned* w = P.near + (r - 1) * P.nwords + (int)row * rw + (x0 >> 5);
        const unsigned any = (unsigned)((((uint64_t)w[1] << 32) | w[0]) >> ((unsigned)x0 & 31u)) & ((2u << (2 * r)) - 1u);
        if (!any && r0 == 2) r0 = r + 1;
      }
    }
    const int best = pd_search<false>(P, c, r0);
    near[c] = best;
    if (best >= 0) atomicAdd(&wp[best], 1);
  }
}

// Density of every cell (haloden.f90:170-181): a non-empty cell sums 1/wp of its particles in
// increasing index order; an empty cell holds 1/wp of the particle that filled it.
__global__ void k_pd_density(float* __restrict__ den, const int* __restrict__ near, const int* __restrict__ wp,
                             const int* __restrict__ start, const int* __restrict__ end, const int* __restrict__ order,
                             i64 ncell) {
  const i64 c = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  float s = 0.f;
  if (near[c] >= 0) s = s + 1.f / (float)wp[near[c]];
  else
    for (int q = start[c]; q < end[c]; ++q) s = s + 1.f / (float)wp[order[q]];
  den[c] = s;
}

// den = real(den, 8) / sum * float(ng)**3 (haloden.f90:187)
__global__ void k_pd_normalise(float* __restrict__ den, const double* __restrict__ sum, float ng3, i64 ncell) {
  const i64 c = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  den[c] = (float)((double)den[c] / sum[0] * (double)ng3);
}

}  // namespace mmh
