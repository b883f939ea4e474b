// Device kernels of the automatic-k callers (emeans-cluster/src/auto.rs and
// metrics.rs), which train and score many small models on data bound once:
//
//  k_row_chain     one chain per row over its columns: kmeans_pp (auto.rs:
//                  401-455) raises every row's best cosine to the picks so far
//                  by the latest pick (the dot in the reference's order:
//                  rounded products added in sequence from zero, no fma), and
//                  internal_scores takes each row's f64 sum of squares;
//  k_sum64         internal_scores' cluster sums (metrics.rs:123-131): f64
//                  sums of each cluster's rows in row order, a chain per
//                  (cluster, column);
//  k_iscore_terms  each row's silhouette, objective and Davies-Bouldin distance
//                  terms in the reference's f64 order (metrics.rs:158-184).
// Each row's dots with the cluster sums (rounded to f32) are launch_dots'.

#include <algorithm>

#include "emh_internal.h"

namespace emh {
namespace {

// A wave takes PR rows: PPH columns of them (16 KB) come to LDS by one burst
// of DMA copies, then lane r runs row r's chain from there (the other lanes
// repeat it: a wave's instructions cost the same); nine such blocks fit a CU.
// Bound by the memory's latency and, from some ten thousand rows, by its
// bandwidth. A thread a row with tiles of 32 columns (256 rows a block) waited
// out the memory's latency once a tile on a fifth of the chip: a pick over
// 12,000 x 768 took 252 us and takes 14, over 60,000 x 1,024 350 and 50
// (4.9 TB/s), over 300,000 x 64 46 and 17. With 768 columns a pass (three
// blocks a CU) the second took 100 us.
// LDS slots are 16 bytes, columns 4u .. 4u + 3:
//  rows of a pass or more (RM): a copy takes 1 KB of one row, slot (r, u) at
//    r * PRS + u (odd stride: the lanes' reads spread over the banks);
//  shorter ones: a copy takes 4 slots of each row, at u * PR + r (whole copies
//    of one row would be mostly padding: 26 us instead of 17 at d = 64);
//  d % 4 != 0 or unaligned rows (V = 1): the same slots by 4-byte lanes.
constexpr int PR = 16, PPH = 256, PU = PPH / 4, PRS = PU + 1;

template <int V, bool PP, bool RM>
__global__ __launch_bounds__(64) void k_row_chain(const float* __restrict__ x, size_t n, int d,
                                                  size_t last, float* __restrict__ best,
                                                  double* __restrict__ xx) {
  typedef float v4f __attribute__((ext_vector_type(4)));
  extern __shared__ __attribute__((aligned(16))) v4f lds[];
  v4f* const qs = lds;  // PP: the pick's columns
  v4f* const xs = lds + (PP ? (min(PU, (d + 3) / 4) + 63) / 64 * 64 : 0);
  const int lane = threadIdx.x, r = lane % PR;
  const float* const q = x + last * (size_t)d;
  const size_t ngr = (n + PR - 1) / PR;
  for (size_t g = blockIdx.x; g < ngr; g += gridDim.x) {
    const size_t mine = g * PR + (V == 4 ? r : lane / 4);  // the row this lane copies from
    const float* const src = x + (mine < n ? mine : n - 1) * (size_t)d;
    float s = 0.0f;
    double sq = 0.0;
    for (int t0 = 0; t0 < d; t0 += PPH) {
      const int m = min(PPH, d - t0), nu = (m + 3) / 4;
      if (RM) {  // (past the last row the last one again)
        const int col = min(t0 + 4 * lane, d - 4);
#pragma unroll
        for (int a = 0; a < PR; a++) {
          const size_t row = g * PR + a < n ? g * PR + a : n - 1;
          __builtin_amdgcn_global_load_lds(x + row * (size_t)d + col, &xs[a * PRS], 16, 0, 0);
        }
        if (PP) __builtin_amdgcn_global_load_lds(q + col, qs, 16, 0, 0);
      } else if (V == 4) {  // d % 4 == 0
        for (int i = 0; i < (nu + 3) / 4; i++)
          __builtin_amdgcn_global_load_lds(src + min(t0 + 4 * (4 * i + lane / PR), d - 4),
                                           &xs[i * 64], 16, 0, 0);
        if (PP)
          for (int i = 0; i < (nu + 63) / 64; i++)
            __builtin_amdgcn_global_load_lds(q + min(t0 + 4 * (64 * i + lane), d - 4),
                                             &qs[i * 64], 16, 0, 0);
      } else {
        for (int i = 0; i < nu; i++)
          __builtin_amdgcn_global_load_lds(src + min(t0 + 4 * i + (lane & 3), d - 1), &xs[i * PR],
                                           4, 0, 0);
        if (PP)
          for (int i = 0; i < (m + 63) / 64; i++)
            __builtin_amdgcn_global_load_lds(q + min(t0 + 64 * i + lane, d - 1), &qs[i * 16], 4,
                                             0, 0);
      }
      __syncthreads();  // waits for the copies
      auto step = [&](float v, float c) __attribute__((always_inline)) {
        if (PP) {
          const float p = v * c;
          s = s + p;
        } else {
          const double p = (double)v * (double)v;
          sq = sq + p;
        }
      };
      const int nf = m / 4;
#pragma unroll 8
      for (int u = 0; u < nf; u++) {
        const v4f v = xs[RM ? r * PRS + u : u * PR + r], c = PP ? qs[u] : v;
        step(v.x, c.x);
        step(v.y, c.y);
        step(v.z, c.z);
        step(v.w, c.w);
      }
      if (V == 1 && nf < nu) {  // the last m % 4 columns
        const v4f v = xs[nf * PR + r], c = PP ? qs[nf] : v;
        step(v.x, c.x);
        if (m % 4 > 1) step(v.y, c.y);
        if (m % 4 > 2) step(v.z, c.z);
      }
      __syncthreads();  // the next copies overwrite these slots
    }
    const size_t row = g * PR + r;
    if (lane >= PR || row >= n) continue;
    if (PP) {
      if (s > best[row]) best[row] = s;
    } else {
      xx[row] = sq;
    }
  }
}

template <bool PP>
void row_chain(emh_ctx* c, const float* x, size_t n, size_t d, size_t last, float* best,
               double* xx) {
  if (n == 0) return;
  const bool v4 = d % 4 == 0 && ((uintptr_t)x & 15) == 0, rm = v4 && d >= PPH;
  const size_t nu = std::min<size_t>(PU, (d + 3) / 4);
  const size_t lds =
      ((PP ? (nu + 63) / 64 * 64 : 0) + (rm ? (size_t)PRS : (nu + 3) / 4 * 4) * PR) * 16;
  const unsigned g = (unsigned)std::min<size_t>((n + PR - 1) / PR, (size_t)32 * c->cus);
  auto kern = rm ? k_row_chain<4, PP, true>
                 : v4 ? k_row_chain<4, PP, false> : k_row_chain<1, PP, false>;
  hipLaunchKernelGGL(kern, dim3(g), dim3(64), lds, c->stream, x, n, (int)d, last, best, xx);
  EMH_HIP(hipGetLastError());
}

// Thread per (cluster s, column t): sums[s][t] = the f64 sum of column t over
// the rows rid[start[s] .. start[s + 1]) in order; sq is filled later. Bound by
// the memory's latency along each chain, so many loads go ahead of the adds (8,
// and none while they are added: 190 us at 12,000 x 768 with 5 clusters; two
// groups of 32 in turn: 106 us).
constexpr int SU = 32;

__global__ __launch_bounds__(256) void k_sum64(const float* __restrict__ x, int d,
                                               const uint32_t* __restrict__ rid,
                                               const uint32_t* __restrict__ start, int ke,
                                               double* __restrict__ sums) {
  const int s = blockIdx.y;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (s >= ke || t >= d) return;
  const uint32_t a = start[s], b = start[s + 1];
  double acc = 0.0;
  const float* const col = x + t;
  auto ids = [&](uint32_t (&r)[SU], uint32_t i) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < SU; q++) r[q] = rid[min(i + q, b - 1)];
  };
  auto load = [&](float (&v)[SU], const uint32_t (&r)[SU]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < SU; q++) v[q] = col[(size_t)r[q] * d];
  };
  auto add = [&](const float (&v)[SU]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < SU; q++) acc += (double)v[q];
  };
  uint32_t i = a;
  if (b - a >= SU) {  // groups of SU rows: one added, one loading, one's ids loading
    const uint32_t end = a + (b - a) / SU * SU;
    uint32_t r[SU];
    float u[SU], v[SU];
    ids(r, a);
    load(u, r);
    ids(r, a + SU);
    for (; i + SU < end; i += 2 * SU) {
      load(v, r);
      ids(r, i + 2 * SU);
      add(u);
      load(u, r);
      ids(r, i + 3 * SU);
      add(v);
    }
    if (i < end) {  // an odd number of groups: the last one is in u
      add(u);
      i += SU;
    }
  }
  for (; i < b; i++) acc += (double)col[(size_t)rid[i] * d];
  sums[(size_t)s * d + t] = acc;
}

// Per row: the silhouette, objective and distance-to-own-mean terms of
// metrics.rs:158-184 from the row's dots g[row][0 .. ke) with the live
// cluster sums (slot own = the row's cluster), f64 throughout.
__global__ __launch_bounds__(256) void k_iscore_terms(
    size_t n, int ke, const float* __restrict__ g, const double* __restrict__ xx,
    const uint32_t* __restrict__ own_of, const double* __restrict__ size,
    const double* __restrict__ sq, double* __restrict__ sil, double* __restrict__ obj,
    double* __restrict__ dist) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int own = (int)own_of[i];
  const float* row = g + i * (size_t)ke;
  const double na = size[own];
  const double dot_own = (double)row[own];
  dist[i] = sqrt(fmax(xx[i] - 2.0 * dot_own / na + sq[own] / (na * na), 0.0));
  const double cos_c = dot_own / fmax(sqrt(sq[own]), 1e-30);
  obj[i] = 2.0 - 2.0 * cos_c;
  double s = 0.0;
  if (!(ke < 2 || na < 2.0)) {
    const double a = 1.0 - (dot_own - xx[i]) / (na - 1.0);
    double b = INFINITY;
    for (int q = 0; q < ke; q++)
      if (q != own) b = fmin(b, 1.0 - (double)row[q] / size[q]);
    const double m = fmax(a, b);
    s = m > 0.0 ? (b - a) / m : 0.0;
  }
  sil[i] = s;
}

}  // namespace

void launch_pp_best(emh_ctx* c, const float* x, size_t n, size_t d, size_t last, float* best) {
  row_chain<true>(c, x, n, d, last, best, nullptr);
}

void launch_sum64(emh_ctx* c, const float* x, size_t d, const uint32_t* rid,
                  const uint32_t* start, size_t ke, double* sums) {
  hipLaunchKernelGGL(k_sum64, dim3((unsigned)((d + 255) / 256), (unsigned)ke), dim3(256), 0,
                     c->stream, x, (int)d, rid, start, (int)ke, sums);
  EMH_HIP(hipGetLastError());
}

void launch_row_dots(emh_ctx* c, const float* x, size_t n, size_t d, const float* sums32,
                     size_t ke, float* g, double* xx) {
  launch_dots(c, x, n, d, sums32, ke, g);
  if (xx && ke > 0) row_chain<false>(c, x, n, d, 0, nullptr, xx);
}

void launch_iscore_terms(emh_ctx* c, size_t n, size_t ke, const float* g, const double* xx,
                         const uint32_t* own, const double* size, const double* sq, double* sil,
                         double* obj, double* dist) {
  hipLaunchKernelGGL(k_iscore_terms, grid1(n, 256), dim3(256), 0, c->stream, n, (int)ke, g, xx,
                     own, size, sq, sil, obj, dist);
  EMH_HIP(hipGetLastError());
}

}  // namespace emh
