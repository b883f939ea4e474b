// The one-pass screen's instantiations (k_screen5) and the kernels that
// prepare its operands: the scales (k_scales) and the fp16 lines (k_lines).
#include <algorithm>

#include "emh_screen5.h"

namespace emh {
namespace {

// Block b (b = 0: a, 1: b): the power of two that brings the largest element of
// up to `rows` whole rows, spread over the selection, to 2^7 .. 2^8, and its
// inverse, into out; no finer than 2^(8 - emin). Whole rows, so that a column
// in larger units than the others is always seen (runs of 64 elements a fixed
// step apart could miss the same columns of every row); rows of the selection,
// because the others may hold anything. 8 bits of fp16's range are left above
// the sample and 21 normal ones below; elements beyond that cost their row the
// exact scan (a centroid's or a data row's: every row of the call). Also clears
// `clear` (nclear words). A thread a column: latency-bound, its loads in flight
// together.
constexpr int SCALE_LOADS = 32;
__global__ __launch_bounds__(1024) void k_scales(const ScaleIn a, const ScaleIn b, int d, int rows,
                                                 uint32_t* __restrict__ clear, int nclear) {
  const ScaleIn in = blockIdx.x ? b : a;
  __shared__ const float* rp[SCALE_ROWS_READ];
  __shared__ float wm[16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if (blockIdx.x == 0 && tid < nclear) clear[tid] = 0u;
  const int nr = (int)min((size_t)rows, in.n);
  if (tid < nr) {
    // Row i of n: in the i-th of nr equal stretches, at a place in it that
    // follows no period (multiples of the golden ratio).
    const uint64_t f = ((uint64_t)tid << 16) + (((uint64_t)tid + 1) * 40503u & 65535u);
    const size_t at = in.lo + (in.n <= (size_t)rows ? (size_t)tid
                                                    : (size_t)((f * in.n >> 16) / (uint64_t)nr));
    const size_t id = in.ids ? (size_t)in.ids[at] : at;
    rp[tid] = in.p + (id < in.nx ? id : 0) * (size_t)d;
  }
  __syncthreads();
  float m = 0.f;
  for (int t = tid; t < d; t += 1024)
    for (int i0 = 0; i0 < nr; i0 += SCALE_LOADS) {
      float v[SCALE_LOADS];
#pragma unroll
      for (int u = 0; u < SCALE_LOADS; u++) v[u] = rp[min(i0 + u, nr - 1)][t];
#pragma unroll
      for (int u = 0; u < SCALE_LOADS; u++) {
        const float e = fabsf(v[u]);
        m = e < INFINITY ? fmaxf(m, e) : m;  // NaN and infinities say nothing of the scale
      }
    }
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) wm[w] = m;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < 16; i++) m = fmaxf(m, wm[i]);
    int e = 8;  // zeros: scale 1
    if (m > 0.f) frexpf(m, &e);  // m in [2^(e - 1), 2^e)
    e = max(max(-50, in.emin), min(e, 60));  // two inverse scales' product stays a normal f32
    in.out[0] = ldexpf(1.0f, 8 - e);
    in.out[1] = ldexpf(1.0f, e - 8);
  }
}

// Rows ids[lo + g] (lo + g without ids; an id >= nx reads row 0) for g < n as
// fp16 lines in out (emh_lines.h, scale[0]), in selection order; norm[g] =
// (|x|^2, the residual), f32 sums in any order. With part: block b writes the
// largest |x|^2 of its rows, with cnorm the largest cnorm[g], and the largest
// residual (f32 bits; a NaN wins) to part[4 b .. 4 b + 2].
// Block b takes rows 8 b .. 8 b + 7, two per wave. HBM-bound: a wave reads a
// row in 256-dimension segments, 16 contiguous bytes per lane, and eight lanes
// fill one 64-byte line; the wave's two rows share a cache line in each slab.
template <bool VEC4>
__global__ __launch_bounds__(256) void k_lines(const float* __restrict__ x, size_t nx, int d,
                                               const uint32_t* __restrict__ ids, size_t lo,
                                               size_t n, const float* __restrict__ scale,
                                               char* __restrict__ out, float2* __restrict__ norm,
                                               const float* __restrict__ cnorm,
                                               uint32_t* __restrict__ part) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int d32 = (d + LINE_DIMS - 1) / LINE_DIMS, nseg = (d32 + 7) >> 3;
  const int js = lane >> 3, q = lane & 7;
  const float s = scale[0];
  size_t g[2];
  bool valid[2];
  const float* xr[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    g[i] = (size_t)blockIdx.x * 8 + 2 * w + i;
    valid[i] = g[i] < n;
    size_t id = 0;
    if (valid[i]) {
      id = ids ? (size_t)ids[lo + g[i]] : lo + g[i];
      if (id >= nx) id = 0;
    }
    xr[i] = x + id * (size_t)d;
  }
  float sq[2] = {0.f, 0.f}, rs[2] = {0.f, 0.f};
#pragma unroll 3
  for (int sg = 0; sg < nseg; sg++) {
    const int j = 8 * sg + js;
    if (j >= d32) break;
    const int col = LINE_DIMS * j + 4 * q;
    float4 v[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (VEC4) {
        v[i] = col < d ? *reinterpret_cast<const float4*>(xr[i] + col) : make_float4(0.f, 0.f, 0.f, 0.f);
      } else {
        v[i].x = col < d ? xr[i][col] : 0.f;
        v[i].y = col + 1 < d ? xr[i][col + 1] : 0.f;
        v[i].z = col + 2 < d ? xr[i][col + 2] : 0.f;
        v[i].w = col + 3 < d ? xr[i][col + 3] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      sq[i] = fmaf(v[i].x, v[i].x, sq[i]);
      sq[i] = fmaf(v[i].y, v[i].y, sq[i]);
      sq[i] = fmaf(v[i].z, v[i].z, sq[i]);
      sq[i] = fmaf(v[i].w, v[i].w, sq[i]);
      const uint2 hv = line_quad(v[i], s, rs[i]);
      if (valid[i])
        *reinterpret_cast<uint2*>(out + ((size_t)j * n + g[i]) * LINE_BYTES + 8 * q) = hv;
    }
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      sq[i] += __shfl_xor(sq[i], m, 64);
      rs[i] += __shfl_xor(rs[i], m, 64);
    }
    if (valid[i] && lane == 0) norm[g[i]] = make_float2(sq[i], rs[i]);
  }
  if (part) {
    uint32_t ma = 0u, mb = 0u, mc = 0u;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (valid[i]) {
        ma = max(ma, __float_as_uint(sq[i]));
        if (cnorm) mb = max(mb, __float_as_uint(cnorm[g[i]]));
        mc = max(mc, __float_as_uint(rs[i]));
      }
    }
    __shared__ uint32_t red[3][4];
    if (lane == 0) {
      red[0][w] = ma;
      red[1][w] = mb;
      red[2][w] = mc;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      const uint32_t* r = red[threadIdx.x];
      part[4 * blockIdx.x + threadIdx.x] = max(max(r[0], r[1]), max(r[2], r[3]));
    }
  }
}

// out[0 .. 2] = the maxima of part[4 i .. 4 i + 2] over i < nparts.
__global__ __launch_bounds__(1024) void k_part_max4(const uint32_t* __restrict__ part,
                                                    size_t nparts, uint32_t* __restrict__ out) {
  constexpr int B = 8;
  __shared__ uint32_t wm[3][16];
  const int tid = threadIdx.x;
  uint32_t ma = 0u, mb = 0u, mc = 0u;
  for (size_t i0 = 0; i0 < nparts; i0 += 1024 * B) {
    uint4 v[B];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const size_t i = i0 + 1024 * (size_t)u + tid;
      v[u] = i < nparts ? reinterpret_cast<const uint4*>(part)[i] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < B; u++) {
      ma = max(ma, v[u].x);
      mb = max(mb, v[u].y);
      mc = max(mc, v[u].z);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    ma = max(ma, (uint32_t)__shfl_xor((int)ma, o, 64));
    mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
    mc = max(mc, (uint32_t)__shfl_xor((int)mc, o, 64));
  }
  if ((tid & 63) == 0) {
    wm[0][tid >> 6] = ma;
    wm[1][tid >> 6] = mb;
    wm[2][tid >> 6] = mc;
  }
  __syncthreads();
  if (tid < 3) {
    uint32_t m = 0u;
    for (int i = 0; i < 16; i++) m = max(m, wm[tid][i]);
    out[tid] = m;
  }
}

template <int KIND, bool ONE>
void launch5(emh_ctx* c, unsigned blocks, const Args5& a) {
  hipLaunchKernelGGL((k_screen5<KIND, ONE>), dim3(blocks), dim3(512), 0, c->stream, a);
  EMH_HIP(hipGetLastError());
}

}  // namespace

void launch_scales(emh_ctx* c, size_t d, const ScaleIn& a, const ScaleIn* b, uint32_t* clear,
                   int nclear) {
  EMH_ENSURE(a.n > 0 && a.nx > 0 && (!b || (b->n > 0 && b->nx > 0)), "scales: no rows");
  hipLaunchKernelGGL(k_scales, dim3(b ? 2 : 1), dim3(1024), 0, c->stream, a, b ? *b : a, (int)d,
                     d <= 2048 ? SCALE_ROWS_READ : SCALE_ROWS_READ / 4, clear, nclear);
  EMH_HIP(hipGetLastError());
}

void launch_lines(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids, size_t lo,
                  size_t n, const float* scale, void* out, float2* norm, const float* cnorm,
                  uint32_t* part) {
  if (n == 0) return;
  EMH_ENSURE(d >= 1 && n < (1u << 31), "lines: shape out of range");
  auto kern = d % 4 == 0 ? k_lines<true> : k_lines<false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)lines_blocks(n)), dim3(256), 0, c->stream, x, nx, (int)d,
                     ids, lo, n, scale, (char*)out, norm, cnorm, part);
  EMH_HIP(hipGetLastError());
}

void launch_part_max4(emh_ctx* c, const uint32_t* part, size_t nparts, uint32_t* out) {
  hipLaunchKernelGGL(k_part_max4, dim3(1), dim3(1024), 0, c->stream, part, nparts, out);
  EMH_HIP(hipGetLastError());
}

void launch_screen5(emh_ctx* c, const Lines5& l, bool ip) {
  // The kernel addresses a slab's rows with 32-bit byte offsets (64 per row).
  EMH_ENSURE(l.nx < (1u << 25) && l.k < (1u << 25), "screen: more than 2^25 rows or centroids");
  EMH_ENSURE(l.tpp >= 1 && l.parts >= 1 && (l.parts - 1) * l.tpp < l.ntiles &&
                 l.parts * l.tpp >= l.ntiles,
             "screen: parts");
  const bool one = l.tpp == 1;
  Args5 a{};
  a.xs = (const char*)l.xs;
  a.xslab = l.xslab;
  a.xn = l.xn;
  a.nx = l.nx;
  a.ids = l.ids;
  a.cs = (const char*)l.cs;
  a.cslab = l.k * (size_t)LINE_BYTES;
  a.cnorm = l.cnorm;
  a.k = (int)l.k;
  a.d = (int)l.d;
  a.kk = 1;
  a.tpp = l.tpp;
  a.parts = l.parts;
  a.ntiles = l.ntiles;
  a.bstride = l.n;
  a.part = l.part;
  a.nparts = l.nparts;
  a.sx = l.sx;
  a.sc = l.sc;
  // Parts of several tiles keep logs (128 KB a block): launches of at most
  // four blocks a CU bound them to 128 MB.
  const int row_tiles = (int)((l.n + T5 - 1) / T5);
  const int step = one ? row_tiles : std::max(1, 4 * std::max(c->cus, 1) / l.parts);
  if (!one)
    a.log = (Cand*)c->log5.get((size_t)std::min(step, row_tiles) * l.parts * 512 * LOG5_TOP1 *
                               sizeof(Cand));
  for (int r = 0; r < row_tiles; r += step) {
    const size_t q0 = (size_t)r * T5, q1 = std::min((size_t)(r + step) * T5, l.n);
    a.lo = l.lo + q0;
    a.nrows = (int)(q1 - q0);
    a.cand = l.cand + q0 * l.parts * L5;
    a.ncand = l.ncand + q0 * l.parts;
    a.bound = l.bound + q0;
    const unsigned blocks = (unsigned)((q1 - q0 + T5 - 1) / T5 * l.parts);
    if (one)
      ip ? launch5<TOP1_IP, true>(c, blocks, a) : launch5<TOP1_L2, true>(c, blocks, a);
    else
      ip ? launch5<TOP1_IP, false>(c, blocks, a) : launch5<TOP1_L2, false>(c, blocks, a);
  }
}

bool screen5_knn_fits(emh_ctx* c, size_t m, size_t n, size_t d) {
  // (fp16 one-pass in every mode but SCREEN_OFF and SCREEN_F32)
  return c->screen != SCREEN_OFF && c->screen != SCREEN_F32 && d >= 32 && m >= 256 && n >= 512 &&
         m < (1u << 25) && n < (1u << 25);
}

void split5(emh_ctx* c, const float* q, size_t m, const float* data, size_t n, size_t d,
            uint32_t* clear, int nclear, Split5* s) {
  // The data's lines once (with their norms, residuals and the maxima of
  // both); the queries' too, unless they are the data.
  const bool same = q == data && m == n;
  float* sc = c->scales + 2 * SCALE_CENTS;
  float* sx = same ? sc : c->scales + 2 * SCALE_ROWS;
  const ScaleIn is{data, n, nullptr, 0, n, sc, -50}, iq{q, m, nullptr, 0, m, sx, -50};
  launch_scales(c, d, is, same ? nullptr : &iq, clear, nclear);
  void* xs = c->csplit.get(lines_bytes(n, d));
  float2* xn = (float2*)c->csplit_norm.get(n * 8);
  // Past PART_MAX_ONCE partials, one workgroup reduces them ahead of the
  // screen, whose every block would otherwise read them all.
  const size_t hb = lines_blocks(n);
  uint32_t* part = (uint32_t*)c->csplit_part.get((hb + 1) * 16);
  launch_lines(c, data, n, d, nullptr, 0, n, sc, xs, xn, nullptr, part);
  s->part = part;
  s->nparts = (int)hb;
  if (hb > PART_MAX_ONCE) {
    launch_part_max4(c, part, hb, part + 4 * hb);
    s->part = part + 4 * hb;
    s->nparts = 1;
  }
  s->cs = s->xs = xs;
  s->xn = xn;
  if (!same) {
    void* qw = c->xsplit.get(lines_bytes(m, d));
    float2* qnw = (float2*)c->xsplit_norm.get(m * 8);
    launch_lines(c, q, m, d, nullptr, 0, m, sx, qw, qnw, nullptr, nullptr);
    s->xs = qw;
    s->xn = qnw;
  }
  s->sx = sx;
  s->sc = sc;
  s->m = m;
  s->n = n;
  s->d = d;
}

int screen5_knn(emh_ctx* c, const float* q, size_t m, const float* data, size_t n, size_t d,
                size_t kk, bool exclude_self, Cand** cand_out, float** bound_out) {
  Split5 s;
  split5(c, q, m, data, n, d, c->small, 3, &s);
  const int row_tiles = (int)((m + T5 - 1) / T5);
  const int ntiles = (int)((n + T5 - 1) / T5);
  // Parts (data-tile ranges) where they fill waves of blocks better: up to
  // MAX_PARTS5, so that a few query tiles still fill the chip (2,000 queries
  // against 100,000 x 512: 8 parts gave 64 blocks, 0.94 ms; 31 take 0.45).
  int parts = parts5(row_tiles, ntiles, std::max(c->cus, 1), MAX_PARTS5, 2.0);
  const int tpp = (ntiles + parts - 1) / parts;
  Cand* cand = (Cand*)c->cand.get((size_t)parts * m * LK * sizeof(Cand));
  float* bound = (float*)c->xnorm.get(2 * m * 4);
  // A launch's threads each keep a log (1 MB a block): launches of whole waves
  // of blocks, at most four.
  const int wave = std::max(1, std::max(c->cus, 1) / parts);
  const int rt_step = 4 * wave;
  Cand* log = (Cand*)c->log5.get((size_t)std::min(rt_step, row_tiles) * parts * 512 * LOG5_KNN *
                                 sizeof(Cand));
  Args5 a{};
  a.xslab = m * (size_t)LINE_BYTES;
  a.cs = (const char*)s.cs;
  a.cslab = n * (size_t)LINE_BYTES;
  a.k = (int)n;
  a.d = (int)d;
  a.kk = (int)kk;
  a.tpp = tpp;
  a.parts = parts;
  a.ntiles = ntiles;
  a.log = log;
  a.bstride = m;
  a.part = s.part;
  a.nparts = s.nparts;
  a.sx = s.sx;
  a.sc = s.sc;
  ProfScope prof(c, EMH_PROF_SCREEN, 2.0 * (double)m * (double)n * (double)d,
                 prof_take(c, EMH_PROF_SCREEN));
  a.xs = (const char*)s.xs;
  a.xn = s.xn;
  a.nx = m;
  for (int r = 0; r < row_tiles; r += rt_step) {
    const size_t q0 = (size_t)r * T5, q1 = std::min((size_t)(r + rt_step) * T5, m);
    a.lo = q0;
    a.nrows = (int)(q1 - q0);
    a.cand = cand + q0 * parts * LK;
    a.bound = bound + q0;
    const unsigned blocks = (unsigned)((q1 - q0 + T5 - 1) / T5 * parts);
    if (exclude_self)
      launch5<KNN_SELF, false>(c, blocks, a);
    else
      launch5<KNN, false>(c, blocks, a);
  }
  *cand_out = cand;
  *bound_out = bound;
  return parts;
}

void launch_scores5(emh_ctx* c, const Split5& s, size_t q0, size_t nb, float* scores, size_t ldS,
                    float* bound) {
  EMH_ENSURE(s.m < (1u << 25) && s.n < (1u << 25) && ldS % 4 == 0 && ldS >= s.n && q0 + nb <= s.m,
             "scores: shape out of range");
  const int row_tiles = (int)((nb + T5 - 1) / T5), ntiles = (int)((s.n + T5 - 1) / T5);
  const int parts0 = parts5(row_tiles, ntiles, std::max(c->cus, 1), 1024, 0.5);
  Args5 a{};
  a.xs = (const char*)s.xs;
  a.xslab = s.m * (size_t)LINE_BYTES;
  a.xn = s.xn;
  a.nx = s.m;
  a.lo = q0;
  a.nrows = (int)nb;
  a.cs = (const char*)s.cs;
  a.cslab = s.n * (size_t)LINE_BYTES;
  a.k = (int)s.n;
  a.d = (int)s.d;
  a.kk = 1;
  a.tpp = (ntiles + parts0 - 1) / parts0;
  a.parts = (ntiles + a.tpp - 1) / a.tpp;
  a.ntiles = ntiles;
  a.bound = bound;
  a.bstride = nb;
  a.part = s.part;
  a.nparts = s.nparts;
  a.sx = s.sx;
  a.sc = s.sc;
  a.scores = scores;
  a.ldS = ldS;
  launch5<SCORES, false>(c, (unsigned)(row_tiles * a.parts), a);
}

}  // namespace emh
