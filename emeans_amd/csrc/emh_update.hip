// The update of one small training batch (up to USB positions) in one launch:
// scatter_add (core/cpu.rs:118-143, scatter_rows 337-375) and the EMA step
// (cpu.rs:389-432), for labels the batch's top-1 call tallied. The separate
// path places every position in a cluster-sorted order (k_place_scan), adds
// the sums (k_sums) and moves the centroids (k_ema): three launches whose
// few, small workgroups spend their time waiting on memory, which on small
// fits and those of the automatic-k sweeps (64- to 1,024-row batches, a hundred
// steps per fit) is most of a step. Here the workgroup of cluster j
//   - reads the batch's labels and row ids (every position at once: a batch
//     is at most USB) and keeps the positions with label j, in order, by
//     ballots: the cluster's rows in selection order;
//   - adds them in that order from +0 (a thread a column), as k_sums;
//   - moves the centroid from the sums in registers, as k_ema: the position,
//     then either the squared norm (one lane adds the rounded squares in
//     order) with the split row and the bound's maxima, or the spherical
//     readout (v / max|v| over its sqrt of the in-order sum of squares);
//   - updates the mass and the epoch's count, and clears its count and the
//     tally's chunk histograms for the next batch.
// Every add and rounding is the separate path's, so the bits are the same.
// No workgroup reads what another writes.

#include "emh_halves.h"
#include "emh_internal.h"

namespace emh {
namespace {

constexpr int UT = 1024;               // most threads per workgroup (d <= UT)
constexpr int USB = UPDATE_SMALL_BATCH;  // most positions per batch
constexpr uint32_t NOROW = 0xffffffffu;
static_assert(USB % 64 == 0 && UPDATE_SMALL_MAX_D <= UT, "shape");

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The mass half of the EMA step (as k_ema and k_mass_preview compute it).
__device__ __forceinline__ float ema_mass(float u, uint32_t cnt, float alpha, float decay,
                                          int replace, float* weight) {
  if (!replace) u = u * decay;
  *weight = 0.0f;
  if (cnt > 0) {
    const float count = (float)cnt;
    const float retained = replace ? 0.0f : u;
    const float step = alpha * count;
    const float mass = retained + step;
    *weight = step / mass;
    u = mass;
  }
  return u;
}

// One element of a moved row: sum s of its n = count rows, old value p.
__device__ __forceinline__ float ema_value(float s, float p, float count, float weight) {
  const float mean = s / count;
  if (weight == 1.0f) return mean;
  const float diff = mean - p;
  const float inc = weight * diff;
  return p + inc;
}

// s0 + v[0] + ... + v[len - 1] in order (one lane; v 16-byte aligned LDS), two
// groups of 16 values' reads alternating with the adds (as k_ema's chain).
__device__ __forceinline__ float ordered_sum(const float* v, int len) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef const float __attribute__((address_space(3)))* lf;
  typedef const f4 __attribute__((address_space(3)))* lf4;
  uint32_t base = (uint32_t)(uintptr_t)v;
  asm volatile("" : "+v"(base));
  const lf lv = (lf)(uintptr_t)base;
  auto load = [&](f4 (&g)[4], int t) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) g[u] = *(lf4)(lv + t + 4 * u);
  };
  auto add = [](float s, const f4 (&g)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      s = s + g[u].x;
      s = s + g[u].y;
      s = s + g[u].z;
      s = s + g[u].w;
    }
    return s;
  };
  float s = 0.0f;
  const int len16 = len & ~15;
  int t = 0;
  if (len16 > 0) {
    f4 a[4], b[4];
    load(a, 0);
    for (; t + 32 <= len16; t += 32) {
      load(b, t + 16);
      s = add(s, a);
      load(a, min(t + 32, len16 - 16));  // the last step reloads a group it has
      s = add(s, b);
    }
    if (t < len16) {
      s = add(s, a);
      t += 16;
    }
  }
  for (; t < len; t++) s = s + lv[t];
  return s;
}

// Cluster j's own group of the bound's maxima.
__device__ __forceinline__ void put_part(const CentsOut& o, size_t j, float norm) {
  const uint32_t m = __float_as_uint(norm);
  uint4 g = make_uint4(m, m, 0u, m);
  if (o.scale) {
    const float2 v = o.norm2[j];
    g.x = __float_as_uint(v.x);
    g.z = __float_as_uint(v.y);
  }
  reinterpret_cast<uint4*>(o.part)[j] = g;
}

template <int NB>
struct SmallLds {
  uint32_t lst[64 * NB];             // the cluster's rows in order
  float sq[UPDATE_SMALL_MAX_D];      // rounded squares of the new row (or of the readout's)
  float nv[UPDATE_SMALL_MAX_D];      // the new row, for its split
  float wmax[UT / 64];               // readout: each wave's max |v|
  uint32_t cnt;
  float weight, rnorm, dif, res;
};

// Cluster j = blockIdx.x, a thread per column in whole waves; a batch of at
// most 64 NB positions. Bound by the memory's latency and, where a cluster has
// hundreds of long rows, by what one CU can fetch: the rows are added in order,
// so two groups of USU of them are in flight in turn (a thread per four columns
// had the registers for one group: 15.2 us for 1,052 x 64 with 32 clusters,
// 11.8 now; 512 x 768 with 5 clusters 27 either way). The separate launches
// take 7.5 + 11 + 4.8 us and 7.3 + 13.7 + 10.0 there, and two more gaps between
// launches.
constexpr int USU = 32;
template <int NB>
__global__ __launch_bounds__(UT) void k_update_small(
    const float* __restrict__ x, size_t nx, size_t d, const uint32_t* __restrict__ ids,
    size_t lo, size_t hi, const uint32_t* __restrict__ labels, size_t k,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ zero_words, size_t nzero,
    float* __restrict__ acc, float* __restrict__ pos, float* __restrict__ usage, float alpha,
    float decay, int replace, float* __restrict__ norms, const CentsOut co,
    float* __restrict__ readout, uint32_t* __restrict__ tally, uint32_t* __restrict__ small) {
  __shared__ __attribute__((aligned(16))) SmallLds<NB> L;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = (int)(blockDim.x >> 6);
  const size_t j = blockIdx.x;
  const bool own = tid < (int)d;  // this thread has a column
  const size_t at = j * d + tid;
  const int n = (int)(hi - lo);
  // The next batch's tally starts from zero; the screen's words too.
  for (size_t i = (size_t)blockIdx.x * blockDim.x + tid; i < nzero;
       i += (size_t)gridDim.x * blockDim.x)
    zero_words[i] = 0;
  if (blockIdx.x == 0 && tid < 3) small[tid] = 0;
  if (tid == 0) {
    const uint32_t cnt = counts[j];
    counts[j] = 0;  // read above by this thread only
    tally[j] += cnt;
    float wgt;
    usage[j] = ema_mass(usage[j], cnt, alpha, decay, replace, &wgt);
    L.cnt = cnt;
    L.weight = wgt;
  }
  // The batch's labels and row ids, every position at once (wave 0).
  uint32_t lab[NB], rw[NB];
  if (w == 0) {
#pragma unroll
    for (int u = 0; u < NB; u++) {
      const int i = 64 * u + lane;
      const size_t p = lo + (size_t)i;
      lab[u] = i < n ? labels[p] : NOROW;
      rw[u] = i < n ? (ids ? ids[p] : (uint32_t)p) : NOROW;
    }
  }
  __syncthreads();
  const uint32_t cnt = L.cnt;
  if (cnt == 0) {  // the row stays; so do its norm, halves and readout
    if (tid == 0 && co.part) put_part(co, j, norms[j]);
    return;
  }
  const float p = own ? pos[at] : 0.0f;
  if (w == 0) {
    uint32_t r = 0;
    bool bad = false;  // a row id past the data adds nothing; reported at the next read
#pragma unroll
    for (int u = 0; u < NB; u++) {
      const bool m = lab[u] == (uint32_t)j;
      const uint64_t b = __ballot(m);
      if (m) {
        const uint32_t i = r + lanes_below(b);
        const bool ok = (size_t)rw[u] < nx;
        bad |= !ok;
        if (i < 64u * NB) L.lst[i] = ok ? rw[u] : NOROW;
      }
      r += (uint32_t)__popcll(b);
    }
    if (bad) small[SW_BAD_ID] = 1;
  }
  __syncthreads();
  // The rows in order from +0 (as k_sums).
  const uint32_t nr = min(cnt, 64u * NB);
  float s = 0.0f, v = 0.0f;
  float tmx = 0.0f;  // readout: max |v| of this thread's values (fold from 0, fmaxf)
  if (own) {
    const float* const col = x + tid;
    // Past the list its last row again, never added; a bad row reads row 0 and
    // adds +0 (s is never -0, so this adds nothing).
    auto load = [&](float (&g)[USU], uint32_t q) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < USU; u++) {
        const uint32_t r = __builtin_amdgcn_readfirstlane(L.lst[min(q + u, nr - 1)]);
        g[u] = col[(size_t)(r != NOROW ? r : 0u) * d];
        g[u] = r != NOROW ? g[u] : 0.0f;
      }
    };
    auto add = [&](const float (&g)[USU], uint32_t q) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < USU; u++)
        if (q + u < nr) s = s + g[u];
    };
    float a[USU], b[USU];
    load(a, 0);
    for (uint32_t q = 0; q < nr; q += 2 * USU) {
      if (q + USU < nr) load(b, q + USU);
      add(a, q);
      if (q + 2 * USU < nr) load(a, q + 2 * USU);
      if (q + USU < nr) add(b, q + USU);
    }
    if (acc) acc[at] = acc[at] + s;
    v = ema_value(s, p, (float)cnt, L.weight);
    pos[at] = v;
    if (norms)
      L.sq[tid] = v * v;
    else if (readout)
      tmx = fmaxf(tmx, fabsf(v));
  }
  // The split row, with the zero columns of the last slab.
  if (co.cs) {
    if (tid == 0) L.dif = L.res = 0.0f;
    L.nv[tid] = v;
    __syncthreads();
    if (tid < (int)(((d + 31) & ~(size_t)31) / 4)) {
      const int t = 4 * tid;
      const float4 q = t < (int)d ? *reinterpret_cast<const float4*>(L.nv + t)
                                  : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const float2 r = put_quad(co, k, j, (size_t)t, q);  // zeros past d
      if (co.scale) add_quad(r, &L.dif, &L.res);  // in any order: the bound allows for it
    }
  }
  if (norms) {
    __syncthreads();
    if (tid == 0) {
      const float nrm = ordered_sum(L.sq, (int)d);
      norms[j] = nrm;
      if (co.part) {
        if (co.scale) co.norm2[j] = make_float2(L.dif, L.res);
        put_part(co, j, nrm);
      }
    }
    return;
  }
  if (!readout) return;
  // The spherical readout (faiss normalize_into, as k_normalize_rows): v /
  // max|v|, then / sqrt of the in-order sum of the squares.
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) tmx = fmaxf(tmx, __shfl_xor(tmx, o, 64));
  if (lane == 0) L.wmax[w] = tmx;
  __syncthreads();
  float mx = L.wmax[0];
  for (int i = 1; i < nw; i++) mx = fmaxf(mx, L.wmax[i]);
  const float s1 = mx > 0.0f ? mx : 1.0f;
  const float qv = v / s1;
  if (own) L.sq[tid] = qv * qv;
  __syncthreads();
  if (tid == 0) L.rnorm = sqrtf(ordered_sum(L.sq, (int)d));
  __syncthreads();
  const float nv = L.rnorm;
  const float s2 = nv > 0.0f ? nv : 1.0f;
  if (own) readout[at] = qv / s2;
}

}  // namespace

bool update_small(size_t n, size_t d, bool spherical) {
  return n > 0 && n <= (size_t)USB && d % 4 == 0 && d <= UPDATE_SMALL_MAX_D &&
         (!spherical || d <= EMA_READOUT_MAX_D);
}

void launch_update_small(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids,
                         size_t lo, size_t hi, const uint32_t* labels, size_t k, uint32_t* counts,
                         uint32_t* tcnt, size_t ntcnt, float* acc, float* pos, float* usage,
                         float alpha, float decay, int replace, float* norms, const CentsOut& co,
                         float* readout, uint32_t* tally) {
  const size_t n = hi > lo ? hi - lo : 0;
  EMH_ENSURE(update_small(n, d, readout != nullptr) && tally && (norms != nullptr) != (readout != nullptr) &&
                 (!co.cs || (norms && co.part)),
             "update: shape outside the small-batch path");
  if (k == 0) return;
  const unsigned threads = (unsigned)std::max<size_t>(64, (d + 63) / 64 * 64);
  auto kern = n <= 256 ? k_update_small<4> : k_update_small<USB / 64>;
  hipLaunchKernelGGL(kern, dim3((unsigned)k), dim3(threads), 0, c->stream, x, nx, d, ids,
                     lo, hi, labels, k, counts, tcnt, tcnt ? ntcnt : 0, acc, pos, usage, alpha,
                     decay, replace, norms, co, readout, tally, c->small);
  EMH_HIP(hipGetLastError());
}

}  // namespace emh
