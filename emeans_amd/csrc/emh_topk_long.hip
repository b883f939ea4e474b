// Exact top-k for more neighbours than the screen's lists hold (kk above
// KMAX = 16, up to KLONG). Device::topk (core/mod.rs:114-124) serves
// kk <= GPU_KMAX in the reference; larger k runs its CPU search (knn.rs:42,
// core/src/knn.rs:53-107). Here both stay on the GPU, with that search's
// results:
//
//  - k_dots: the exact dots of a block of queries against every data row,
//    each the sequential f32 fma chain over the d dimensions (the float order
//    of every other score in this library), into scratch;
//  - or, where queries and data rows make it pay, the same dots on the MFMA
//    within a bound (k_screen5's SCORES), from which k_select_screened lists
//    every row that can be among the kk best and computes those rows' chains
//    alone; queries that it cannot settle go through the next two;
//  - k_select_long: one workgroup per query keeps the kk best data rows by a
//    radix select over the scores (larger score first, the lower id among
//    equal scores: the rows the reference keeps by replacing its worst entry
//    only on a strictly larger score while ids increase, knn.rs:82-96), then
//    sorts them by score descending in IEEE total order, then id ascending
//    (knn.rs:97-99). NaN and -inf scores are never kept (no score is larger
//    than the -inf a slot starts with); exclude_self skips j == i; missing
//    entries are id 0xFFFFFFFF, score -inf.

#include <algorithm>

#include "emh_select.h"

namespace emh {
namespace {

// S[i ldS + j] = chain over t < d of q[q0 + i][t] * x[j][t], i < qb, j < n.
// A block computes BM queries against BN data rows, a thread TM x TN chains
// (TM, TN / 4 groups of four consecutive columns, so that LDS reads are 16
// bytes and a row's stores are contiguous): with 8 x 8 the fmas of a
// dimension (64 a thread) take twice the time of its four LDS reads, where
// 4 x 4 was bound by the reads (1,000 x 50,000 x 384: 1.26 ms). Slabs of DK
// dimensions are double-buffered: the next one's loads are in flight while the
// present one's fmas run. Few queries take narrow tiles (bound by the reads of
// the data, and by what is padded).
constexpr int DK = 16;

// LIST: of queries list[1 .. list[0]] (rows of S too) instead, at most qb.
template <int BM, int BN, int TM, int TN, bool LIST>
__global__ __launch_bounds__(256) void k_dots(const float* __restrict__ q, size_t q0, int qb,
                                              const float* __restrict__ x, int n, int d,
                                              float* __restrict__ S, size_t ldS,
                                              const uint32_t* __restrict__ list) {
  static_assert((BM / TM) * (BN / TN) == 256, "threads");
  constexpr int QP = BM + 4, XP = BN + 4;  // padded: the transposed stores spread over the banks
  constexpr int NTX = BN / TN;             // threads along the data rows
  constexpr int VT = TN < 4 ? TN : 4;      // columns per group
  constexpr int GN = TN / VT;              // groups, BN / GN columns apart
  constexpr int LQ = (BM * DK / 4 + 255) / 256, LX = (BN * DK / 4 + 255) / 256;  // float4 loads
  __shared__ __attribute__((aligned(16))) float Qs[2][DK][QP];
  __shared__ __attribute__((aligned(16))) float Xs[2][DK][XP];
  const int tid = threadIdx.x, tx = tid % NTX, ty = tid / NTX;
  const int j0 = blockIdx.x * BN, i0 = blockIdx.y * BM;
  if (LIST) {
    qb = min(qb, (int)list[0]);
    if (i0 >= qb) return;
  }
  auto qrow = [&](int i) { return LIST ? (int)list[1 + i] : i; };
  // Loader: float4 e of an operand's slab is row e / 4, dimensions 4 (e % 4) .. + 3.
  float qr[LQ][4], xr[LX][4];
  auto load = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < LQ; u++) {
      const int e = u * 256 + tid, r = e >> 2, t = t0 + 4 * (e & 3);
      const float* p = q + (q0 + (size_t)qrow(min(i0 + min(r, BM - 1), qb - 1))) * (size_t)d;
#pragma unroll
      for (int c = 0; c < 4; c++) qr[u][c] = t + c < d ? p[t + c] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < LX; u++) {
      const int e = u * 256 + tid, r = e >> 2, t = t0 + 4 * (e & 3);
      const float* p = x + (size_t)min(j0 + min(r, BN - 1), n - 1) * (size_t)d;
#pragma unroll
      for (int c = 0; c < 4; c++) xr[u][c] = t + c < d ? p[t + c] : 0.f;
    }
  };
  auto store = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < LQ; u++) {
      const int e = u * 256 + tid, r = e >> 2, t = 4 * (e & 3);
      if (r < BM)
#pragma unroll
        for (int c = 0; c < 4; c++) Qs[b][t + c][r] = qr[u][c];
    }
#pragma unroll
    for (int u = 0; u < LX; u++) {
      const int e = u * 256 + tid, r = e >> 2, t = 4 * (e & 3);
      if (r < BN)
#pragma unroll
        for (int c = 0; c < 4; c++) Xs[b][t + c][r] = xr[u][c];
    }
  };
  float acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) acc[a][b] = 0.f;
  auto dim = [&](int b, int t) __attribute__((always_inline)) {
    float qv[TM], xv[TN];
#pragma unroll
    for (int a = 0; a < TM; a++) qv[a] = Qs[b][t][ty * TM + a];
#pragma unroll
    for (int g = 0; g < GN; g++)
#pragma unroll
      for (int c = 0; c < VT; c++) xv[g * VT + c] = Xs[b][t][g * (BN / GN) + tx * VT + c];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int c = 0; c < TN; c++) acc[a][c] = fmaf(qv[a], xv[c], acc[a][c]);
  };
  load(0);
  store(0);
  __syncthreads();
  for (int t0 = 0, b = 0; t0 < d; t0 += DK, b ^= 1) {
    const bool more = t0 + DK < d;
    if (more) load(t0 + DK);
    const int tn = min(DK, d - t0);  // dimensions past d never enter a chain
    if (tn == DK) {
#pragma unroll
      for (int t = 0; t < DK; t++) dim(b, t);
    } else {
      for (int t = 0; t < tn; t++) dim(b, t);
    }
    if (more) store(b ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < TM; a++) {
    const int i = i0 + ty * TM + a;
    if (i >= qb) break;
    float* o = S + (size_t)qrow(i) * ldS;
#pragma unroll
    for (int g = 0; g < GN; g++)
#pragma unroll
      for (int c = 0; c < VT; c++) {
        const int j = j0 + g * (BN / GN) + tx * VT + c;
        if (j < n) o[j] = acc[a][g * VT + c];
      }
  }
}

template <int BM, int BN, int TM, int TN>
void dots(emh_ctx* c, const float* q, size_t q0, size_t nb, const float* data, size_t n, size_t d,
          float* S, size_t ldS, const uint32_t* list = nullptr) {
  const dim3 g((unsigned)((n + BN - 1) / BN), (unsigned)((nb + BM - 1) / BM));
  if (list)
    hipLaunchKernelGGL((k_dots<BM, BN, TM, TN, true>), g, dim3(256), 0, c->stream, q, q0, (int)nb,
                       data, (int)n, (int)d, S, ldS, list);
  else
    hipLaunchKernelGGL((k_dots<BM, BN, TM, TN, false>), g, dim3(256), 0, c->stream, q, q0, (int)nb,
                       data, (int)n, (int)d, S, ldS, list);
  EMH_HIP(hipGetLastError());
}

// Ascending unsigned image of a float's IEEE total order.
__device__ __forceinline__ uint32_t ord_total(float v) {
  const uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_ord(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}
// The selection's key: 0 for a score that is never kept (NaN, -inf, the
// query itself), else the ascending image of its IEEE value (-0 == +0:
// adding +0 turns -0 into +0). Every kept key is above ord_total(-inf) > 0.
__device__ __forceinline__ uint32_t sel_key(float v, bool skip) {
  if (skip || !(v > -INFINITY)) return 0u;
  return ord_total(v + 0.0f);
}

constexpr int NT = 1024;  // threads per selecting workgroup
constexpr int NW = NT / 64;

// Block-wide exclusive prefix of one flag per thread, and the block's total.
__device__ __forceinline__ int block_rank(bool f, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long b = __ballot(f);
  const int below = __popcll(b & ((1ull << lane) - 1ull));
  if (lane == 0) wsum[w] = __popcll(b);
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int v = 0; v < NW; v++) {
    const int c = wsum[v];
    before += v < w ? c : 0;
    total += c;
  }
  __syncthreads();
  return before + below;
}

// Bitonic sort of sk[0 .. cnt) (P slots, the rest filled), ascending.
template <int P, int T = NT>
__device__ __forceinline__ void sort_keys(unsigned long long* sk, uint32_t cnt) {
  const int tid = threadIdx.x;
  // (A power of two that holds them: short lists skip the wide stages.)
  int m = 2;
  while (m < (int)cnt) m <<= 1;
  for (int s = tid; s < m; s += T)
    if ((uint32_t)s >= cnt) sk[s] = ~0ull;
  __syncthreads();
  for (int size = 2; size <= m; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = tid; t < m / 2; t += T) {
        const int lo = 2 * t - (t & (stride - 1));
        const int hi = lo + stride;
        const bool up = (lo & size) == 0;
        const unsigned long long a = sk[lo], b = sk[hi];
        if ((a > b) == up) {
          sk[lo] = b;
          sk[hi] = a;
        }
      }
      __syncthreads();
    }
  }
}

// The largest x that kk of the threads' values `mine` are not below (0: fewer
// than kk are above 0).
__device__ __forceinline__ uint32_t kth_of_threads(uint32_t mine, int kk) {
  uint32_t x = 0u;
  for (int b = 31; b >= 0; b--)
    if (__syncthreads_count(mine >= (x | (1u << b))) >= kk) x |= 1u << b;
  return x;
}

// sk[0 .. got) = (~key, id) of listed scores, any order: sorted, cut to the kk
// best, and those given their own order (IEEE total order, then id) as keys.
// Returns how many.
template <int P, int T = NT>
__device__ __forceinline__ uint32_t best_of_listed(unsigned long long* sk, uint32_t got, int kk,
                                                   const float* row) {
  sort_keys<P, T>(sk, got);
  const uint32_t cnt = min(got, (uint32_t)kk);
  for (uint32_t s = threadIdx.x; s < cnt; s += T) {
    const uint32_t j = (uint32_t)sk[s];
    sk[s] = ((unsigned long long)(~ord_total(row[j])) << 32) | (unsigned long long)j;
  }
  __syncthreads();
  return cnt;
}

// The sorted result of a query.
template <int T = NT>
__device__ __forceinline__ void put_result(const unsigned long long* sk, uint32_t cnt, size_t qi,
                                           int kk, uint32_t* __restrict__ ids,
                                           float* __restrict__ sims) {
  for (int t = threadIdx.x; t < kk; t += T) {
    const size_t o = qi * (size_t)kk + t;
    if ((uint32_t)t < cnt) {
      const unsigned long long e = sk[t];
      ids[o] = (uint32_t)e;
      sims[o] = from_ord(~(uint32_t)(e >> 32));
    } else {
      ids[o] = NONE;
      sims[o] = -INFINITY;
    }
  }
}

// Workgroup i: the kk best data rows of query q0 + i from its screen scores
// S[i ldS ..], each within bound[i] = E of its exact chain. kk of the scores
// are not below the kk-th largest x of the threads' maxima (two a thread), so kk exact ones
// are not below x - E, and a row whose score is below x - 2E is not among the
// kk best: the others, listed in sk, get their exact chains (into S) and the
// selection takes it from there. A query with a bound that is not a small
// number (NaN; 1e32 keeps every chain finite), with fewer than kk candidates
// or more than KLONG goes to list[1 + list[0]++]. kk <= ST.
//
// Bound by its two reads of the scores and the latency of the listed rows'
// loads: a lane runs one candidate's chain, eight loads ahead, the candidates
// spread over the waves. 1,000 x 50,000 x 384, k = 100, whole calls: 929 us
// with every chain computed (k_dots' share is bound by the VALU at 48
// TFLOP/s), 362 us with the screen's scores, 266 us since the workgroup has 512
// threads (four a CU, so that one's loads cover another's chains: 1,024 of
// them made two waves of two a CU), one wave finds x by ballots and short lists
// are ranked instead of sorted (this kernel: 249 -> 147 us).
constexpr int ST = 512;  // threads of k_select_screened
template <bool VEC4>
__global__ __launch_bounds__(ST) void k_select_screened(
    float* __restrict__ S, size_t ldS, int n, int d, const float* __restrict__ q, size_t q0,
    const float* __restrict__ x, const float* __restrict__ bound, int kk, int exclude_self,
    uint32_t* __restrict__ ids, float* __restrict__ sims, uint32_t* __restrict__ list) {
  constexpr int P = KLONG;  // (32 KB: four workgroups a CU all the same)
  __shared__ unsigned long long sk[P];
  __shared__ uint32_t sh_n, sh_x;
  uint32_t* mx = (uint32_t*)sk;  // the 2 ST maxima, until the list starts
  const int tid = threadIdx.x;
  const size_t qi = q0 + blockIdx.x;
  float* row = S + (size_t)blockIdx.x * ldS;
  const float E = bound[blockIdx.x];
  auto give_up = [&]() {
    if (tid == 0) list[1 + atomicAdd(&list[0], 1u)] = blockIdx.x;
  };
  if (!(E < 1e32f)) {  // (uniform)
    give_up();
    return;
  }
  // Scores four at a time (a row starts at a multiple of 16 bytes and its
  // padding up to ldS is readable).
  auto load4 = [&](int j, uint32_t (&k4)[4]) __attribute__((always_inline)) {
    const float4 v = *reinterpret_cast<const float4*>(row + j);
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int t = 0; t < 4; t++)
      k4[t] = j + t < n ? sel_key(e[t], exclude_self && (size_t)(j + t) == qi) : 0u;
  };
  uint32_t mine[2] = {0u, 0u};
  for (int j0 = 4 * tid; j0 < n; j0 += 32 * ST) {
#pragma unroll
    for (int u = 0; u < 8; u++) {
      uint32_t k4[4];
      if (j0 + 4 * u * ST < n) {
        load4(j0 + 4 * u * ST, k4);
        mine[u & 1] = max(max(mine[u & 1], max(k4[0], k4[1])), max(k4[2], k4[3]));
      }
    }
  }
  mx[tid] = mine[0];
  mx[ST + tid] = mine[1];
  if (tid == 0) sh_n = 0u;
  __syncthreads();
  if (tid < 64) {  // the largest x that kk maxima are not below, by ballots of one wave
    uint32_t v[2 * ST / 64];
#pragma unroll
    for (int i = 0; i < 2 * ST / 64; i++) v[i] = mx[64 * i + tid];
    uint32_t xk = 0u;
    for (int b = 31; b >= 0; b--) {
      const uint32_t t = xk | (1u << b);
      int c = 0;
#pragma unroll
      for (int i = 0; i < 2 * ST / 64; i++) c += __popcll(__ballot(v[i] >= t));
      if (c >= kk) xk = t;
    }
    if (tid == 0) sh_x = xk;
  }
  __syncthreads();
  const uint32_t xk = sh_x;
  if (xk == 0u) {
    give_up();
    return;
  }
  const float xv = from_ord(xk);
  const float lim = xv - 2.0157f * E - fabsf(xv) * 4.7683716e-07f - 1e-42f;
  const uint32_t lk = sel_key(lim, false);  // (lim is finite)
  for (int j0 = 4 * tid; j0 < n; j0 += 32 * ST) {
#pragma unroll
    for (int u = 0; u < 8; u++) {
      uint32_t k4[4];
      const int j = j0 + 4 * u * ST;
      if (j < n) {
        load4(j, k4);
#pragma unroll
        for (int t = 0; t < 4; t++)
          if (k4[t] >= lk) {
            const uint32_t at = atomicAdd(&sh_n, 1u);
            if (at < (uint32_t)P) sk[at] = (unsigned long long)(uint32_t)(j + t);
          }
      }
    }
  }
  __syncthreads();
  const uint32_t got = sh_n;
  if (got > (uint32_t)P || got < (uint32_t)kk) {
    give_up();
    return;
  }
  const float* qr = q + qi * (size_t)d;
  for (uint32_t s = (uint32_t)((tid & 63) * (ST / 64) + (tid >> 6)); s < got; s += ST) {
    const uint32_t j = (uint32_t)sk[s];
    const float* p = x + (size_t)j * (size_t)d;
    float acc = 0.f;
    int t = 0;
    for (; t + 32 <= d; t += 32) {
      float v[32];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        if (VEC4) {
          const float4 f = *reinterpret_cast<const float4*>(p + t + 4 * e);
          v[4 * e] = f.x;
          v[4 * e + 1] = f.y;
          v[4 * e + 2] = f.z;
          v[4 * e + 3] = f.w;
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++) v[4 * e + c] = p[t + 4 * e + c];
        }
      }
#pragma unroll
      for (int e = 0; e < 32; e++) acc = fmaf(qr[t + e], v[e], acc);
    }
    for (; t < d; t++) acc = fmaf(qr[t], p[t], acc);
    row[j] = acc;
    // Key first (-0 and +0 alike, as the selection compares them), then id.
    sk[s] = ((unsigned long long)(~sel_key(acc, false)) << 32) | (unsigned long long)j;
  }
  __syncthreads();
  if (got > (uint32_t)P / 4) {
    const uint32_t cnt = best_of_listed<P, ST>(sk, got, kk, row);
    sort_keys<P, ST>(sk, cnt);
    put_result<ST>(sk, cnt, qi, kk, ids, sims);
    return;
  }
  // Few: each key's rank by comparing it with all (110 of them: 28 stages of
  // the bitonic sort, with a barrier each, otherwise); then the kk best in
  // their own order (IEEE total order, then id) the same way.
  unsigned long long* best = sk + P / 2;
  for (uint32_t s = tid; s < got; s += ST) {
    const unsigned long long k = sk[s];
    uint32_t r = 0;
    for (uint32_t i = 0; i < got; i++) r += sk[i] < k ? 1u : 0u;
    if (r < (uint32_t)kk)
      best[r] = ((unsigned long long)(~ord_total(row[(uint32_t)k])) << 32) | (uint32_t)k;
  }
  __syncthreads();
  for (int s = tid; s < kk; s += ST) {
    const unsigned long long k = best[s];
    uint32_t r = 0;
    for (int i = 0; i < kk; i++) r += best[i] < k ? 1u : 0u;
    const size_t o = qi * (size_t)kk + r;
    ids[o] = (uint32_t)k;
    sims[o] = from_ord(~(uint32_t)(k >> 32));
  }
}

// Workgroup i: the kk best data rows of query q0 + i from its scores
// S[i ldS ..], written to ids / sims row q0 + i. P (a power of two >= kk)
// slots of sort keys in LDS. With list, i = list[1 + workgroup] for the first
// list[0] of them.
template <int P>
__global__ __launch_bounds__(NT) void k_select_long(const float* __restrict__ S, size_t ldS,
                                                    int n, size_t q0, int kk, int exclude_self,
                                                    uint32_t* __restrict__ ids,
                                                    float* __restrict__ sims,
                                                    const uint32_t* __restrict__ list) {
  if (list && blockIdx.x >= list[0]) return;
  __shared__ unsigned long long sk[P];
  __shared__ uint32_t hist[2048];
  __shared__ int wsum[NW];
  __shared__ uint32_t sh_prefix, sh_rem, sh_all;
  const int tid = threadIdx.x;
  const size_t bi = list ? list[1 + blockIdx.x] : blockIdx.x;
  const size_t qi = q0 + bi;
  const float* row = S + bi * ldS;
  auto key_at = [&](int j) { return sel_key(row[j], exclude_self && (size_t)j == qi); };

  uint32_t cnt = 0;
  bool listed = false;
  if (kk <= NT / 2) {
    // The kk-th largest of the threads' own maxima is at most the kk-th
    // largest key: the keys not below it are few (about -NT ln(1 - kk / NT) of
    // them in no particular order), so one more pass lists them all. Two reads
    // of the row and no histogram, whose atomics meet in a few bins (1,000
    // rows of 50,000: 593 us with the three radix passes).
    uint32_t mine = 0u;
    for (int j0 = tid; j0 < n; j0 += 8 * NT) {
      uint32_t k8[8];
#pragma unroll
      for (int u = 0; u < 8; u++) k8[u] = j0 + u * NT < n ? key_at(j0 + u * NT) : 0u;
#pragma unroll
      for (int u = 0; u < 8; u++) mine = max(mine, k8[u]);
    }
    const uint32_t x = kth_of_threads(mine, kk);
    if (tid == 0) sh_all = 0u;
    __syncthreads();
    for (int j0 = tid; j0 < n; j0 += 8 * NT) {
      uint32_t k8[8];
#pragma unroll
      for (int u = 0; u < 8; u++) k8[u] = j0 + u * NT < n ? key_at(j0 + u * NT) : 0u;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        if (k8[u] == 0u || k8[u] < x) continue;
        const int j = j0 + u * NT;
        const uint32_t at = atomicAdd(&sh_all, 1u);
        // Key first (-0 and +0 alike, as the selection compares them), then id.
        if (at < (uint32_t)P) sk[at] = ((unsigned long long)(~k8[u]) << 32) | (uint32_t)j;
      }
    }
    __syncthreads();
    const uint32_t got = sh_all;
    __syncthreads();
    listed = got <= (uint32_t)P;
    if (listed) cnt = best_of_listed<P>(sk, got, kk, row);
  }
  if (!listed) {
  // Radix select of the kk-th largest key: digits of 11, 11 and 10 bits.
  uint32_t prefix = 0, pmask = 0;
  uint32_t rem = (uint32_t)kk;
  bool all = false;  // fewer kept scores than kk: every one is taken
  for (int pass = 0; pass < 3 && !all; pass++) {
    const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
    const int nb = pass == 2 ? 1024 : 2048;
    for (int b = tid; b < nb; b += NT) hist[b] = 0u;
    __syncthreads();
    for (int j = tid; j < n; j += NT) {
      const uint32_t k = key_at(j);
      if (k != 0u && (k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & (nb - 1)], 1u);
    }
    __syncthreads();
    if (tid < 64) {
      // Lane l sums bins from the top: segment [nb - (l + 1) s, nb - l s).
      const int s = nb / 64;
      const int hi = nb - tid * s;
      uint32_t seg = 0;
      for (int b = hi - 1; b >= hi - s; b--) seg += hist[b];
      uint32_t incl = seg;  // inclusive prefix over lanes 0 .. tid (top bins first)
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o, 64);
        if (tid >= o) incl += t;
      }
      const uint32_t total = __shfl(incl, 63, 64);
      if (pass == 0 && total <= rem) {
        if (tid == 0) sh_all = 1u;
      } else {
        const uint32_t excl = incl - seg;
        if (excl < rem && rem <= incl) {  // the digit is in this lane's segment
          uint32_t above = excl;
          for (int b = hi - 1; b >= hi - s; b--) {
            const uint32_t c = hist[b];
            if (above + c >= rem) {
              sh_prefix = prefix | ((uint32_t)b << shift);
              sh_rem = rem - above;
              break;
            }
            above += c;
          }
        }
        if (tid == 0) sh_all = 0u;
      }
    }
    __syncthreads();
    all = sh_all != 0u;
    if (!all) {
      prefix = sh_prefix;
      rem = sh_rem;
      pmask |= (uint32_t)(nb - 1) << shift;
    }
    __syncthreads();
  }
  // Keys above T = prefix are all kept (kk - rem of them); of the keys equal
  // to T, the rem with the lowest ids. With `all`, every kept key.
  const uint32_t T = prefix;
  const uint32_t n_gt = all ? 0u : (uint32_t)kk - rem, need = all ? 0u : rem;
  uint32_t got_gt = 0, got_eq = 0;
  for (int j0 = 0; j0 < n; j0 += NT) {
    const int j = j0 + tid;
    const uint32_t k = j < n ? key_at(j) : 0u;
    const bool gt = all ? k != 0u : k > T;
    const bool eq = !all && k != 0u && k == T;
    int tot_gt, tot_eq;
    const int rg = block_rank(gt, wsum, tot_gt);
    const int re = block_rank(eq, wsum, tot_eq);
    const float v = j < n ? row[j] : 0.f;
    const unsigned long long sortkey =
        ((unsigned long long)(~ord_total(v)) << 32) | (unsigned long long)(uint32_t)j;
    if (gt) sk[got_gt + rg] = sortkey;
    if (eq && got_eq + re < need) sk[n_gt + got_eq + re] = sortkey;
    got_gt += tot_gt;
    got_eq += tot_eq;
  }
  cnt = all ? got_gt : (uint32_t)kk;
  }
  sort_keys<P>(sk, cnt);
  put_result<NT>(sk, cnt, qi, kk, ids, sims);
}

template <int P>
void select_long(emh_ctx* c, unsigned blocks, const float* S, size_t ldS, size_t n, size_t q0,
                 size_t kk, bool exclude_self, uint32_t* ids, float* sims,
                 const uint32_t* list = nullptr) {
  hipLaunchKernelGGL(k_select_long<P>, dim3(blocks), dim3(NT), 0, c->stream, S, ldS, (int)n, q0,
                     (int)kk, exclude_self ? 1 : 0, ids, sims, list);
  EMH_HIP(hipGetLastError());
}

void select_screened(emh_ctx* c, unsigned blocks, float* S, size_t ldS, size_t n, size_t d,
                     const float* q, size_t q0, const float* data, const float* bound, size_t kk,
                     bool exclude_self, uint32_t* ids, float* sims, uint32_t* list) {
  auto kern = d % 4 == 0 ? k_select_screened<true> : k_select_screened<false>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(ST), 0, c->stream, S, ldS, (int)n, (int)d, q, q0,
                     data, bound, (int)kk, exclude_self ? 1 : 0, ids, sims, list);
  EMH_HIP(hipGetLastError());
}

// Whether the screened selection takes a call. Splitting the data into lines,
// the scores' launch and the (mostly empty) launches over the list cost about
// 45 us, and the chains of the listed rows grow with kk and not with n: below
// 10^9 products (us, direct / screened: 20,000 x 64 by 256 queries, k = 100: 70
// / 75; 8,192 x 768 by 64: 106 / 104; above: 20,000 x 64 by 1,000: 212 / 179),
// with fewer than 32 rows a neighbour (8,192 x 768 by 1,000, k = 500: 388 /
// 471; 20,000 x 384, k = 500: 497 / 371) and for fewer than 16 queries (which
// read the data once, with nothing written) the direct dots stay.
bool long_screened(emh_ctx* c, size_t m, size_t n, size_t d, size_t kk) {
  return c->screen != SCREEN_OFF && c->screen != SCREEN_F32 && kk <= ST && d >= 32 &&
         d <= 16384 && m >= 16 && m < (1u << 25) && n >= 32 * kk && n < (1u << 25) &&
         (double)m * (double)n * (double)d >= 1e9;
}

}  // namespace

// Tiles by the columns there are: 16 for a handful (four chains a thread, more
// blocks), 64, or 128 x 128 when such tiles make two blocks a CU (20,000 x 768
// by 100: 32 x 128 tiles 175 us, 128 x 128 194; a thread a row 4,260). The clusters of the automatic-k sweeps
// are 2 to 40: 12,000 x 768 rows against 20 took 1,374 us with a thread a row and
// 64 chains each, 63 us here.
void launch_dots(emh_ctx* c, const float* a, size_t m, size_t d, const float* b, size_t nb,
                 float* out) {
  EMH_ENSURE(d > 0 && d < (1u << 31), "dots: shape too large");
  // (grid.y, and the int arithmetic on columns, stay in range.)
  const size_t rows = size_t(1) << 21, cols = size_t(1) << 24;
  for (size_t i0 = 0; i0 < m; i0 += rows)
    for (size_t j0 = 0; j0 < nb; j0 += cols) {
      const size_t mi = std::min(rows, m - i0), nj = std::min(cols, nb - j0);
      const float* bj = b + j0 * d;
      float* o = out + i0 * nb + j0;
      if (nj <= 16)
        dots<64, 16, 4, 1>(c, a, i0, mi, bj, nj, d, o, nb);
      else if (nj <= 64)
        dots<64, 64, 4, 4>(c, a, i0, mi, bj, nj, d, o, nb);
      else if ((mi + 127) / 128 * ((nj + 127) / 128) < 2 * (size_t)c->cus)
        dots<32, 128, 4, 4>(c, a, i0, mi, bj, nj, d, o, nb);
      else
        dots<128, 128, 8, 8>(c, a, i0, mi, bj, nj, d, o, nb);
    }
}

void launch_topk_long(emh_ctx* c, const float* q, size_t m, const float* data, size_t n,
                      size_t d, size_t kk, bool exclude_self, uint32_t* ids, float* sims) {
  EMH_ENSURE(kk >= 1 && kk <= KLONG, "topk: kk = %zu outside 1..%d", kk, KLONG);
  EMH_ENSURE(m < (1u << 31) && n < (1u << 31) && d < (1u << 31), "topk: shape too large");
  if (m == 0) return;
  // Scores of a block of queries against all data rows: about 1 GiB of
  // scratch, at least one 128-query tile.
  constexpr size_t DT = 128;
  const size_t ldS = std::max<size_t>((n + 3) & ~size_t(3), 4);
  const size_t budget = size_t(1) << 30;
  size_t qb = std::max<size_t>(budget / (ldS * 4) / DT * DT, DT);
  qb = std::min(std::min(qb, size_t(65535) * DT), m);  // grid.y of k_dots within 65535
  float* S = (float*)c->klong.get(qb * ldS * 4);
  const bool screened = long_screened(c, m, n, d, kk);
  Split5 sp{};
  uint32_t* list = nullptr;
  float* bound = nullptr;
  if (screened) {
    list = (uint32_t*)c->fblist.get((qb + 1) * 4);
    bound = (float*)c->xnorm.get(2 * qb * 4);
    split5(c, q, m, data, n, d, list, 1, &sp);
  }
  for (size_t q0 = 0; q0 < m; q0 += qb) {
    const size_t nb = std::min(qb, m - q0);
    if (screened) {
      if (q0 > 0) launch_fill_u32(c, list, 1, 0);
      launch_scores5(c, sp, q0, nb, S, ldS, bound);
      select_screened(c, (unsigned)nb, S, ldS, n, d, q, q0, data, bound, kk, exclude_self, ids,
                      sims, list);
    }
    // (Screened: what is left in the list, by the same kernels.)
    if (n > 0) {
      // Tiles by the queries there are; the wide one also needs data rows for
      // two blocks a CU.
      const size_t wide = (nb + 127) / 128 * ((n + 127) / 128);
      if (nb <= 8)
        dots<8, 256, 4, 2>(c, q, q0, nb, data, n, d, S, ldS, list);
      else if (nb <= 64 || wide < 2 * (size_t)c->cus)
        dots<32, 128, 4, 4>(c, q, q0, nb, data, n, d, S, ldS, list);
      else
        dots<128, 128, 8, 8>(c, q, q0, nb, data, n, d, S, ldS, list);
    }
    const unsigned blocks = (unsigned)nb;
    if (kk <= 128)
      select_long<1024>(c, blocks, S, ldS, n, q0, kk, exclude_self, ids, sims, list);
    else
      select_long<KLONG>(c, blocks, S, ldS, n, q0, kk, exclude_self, ids, sims, list);
  }
}

}  // namespace emh
