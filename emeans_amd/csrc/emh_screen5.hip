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
// exact scan (a centroid's or a data row's: every row of the call). With
// in.mean: the rows' mean and the scale of the differences, where the mean
// holds a quarter of the rows' squares or more (the mean of 32 rows without one
// holds a 32nd, and would only add to them); else zeros. Also clears `clear`
// (nclear words). A thread a column: latency-bound, its loads in flight
// together.
__global__ __launch_bounds__(1024) void k_scales(const ScaleIn a, const ScaleIn b, int d, int rows,
                                                 uint32_t* __restrict__ clear, int nclear) {
  constexpr int R = SCALE_ROWS_READ;
  const int NT = (int)blockDim.x;
  const ScaleIn in = blockIdx.x ? b : a;
  __shared__ const float* rp[R];
  __shared__ float4 wr[16];
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
  // Largest element and difference; squares of the rows and of the mean.
  float mv = 0.f, mc = 0.f, sv = 0.f, sm = 0.f;
  const float inv = 1.0f / (float)nr;
  for (int t = tid; t < d; t += NT) {
    float v[R];
#pragma unroll
    for (int u = 0; u < R; u++) v[u] = rp[min(u, nr - 1)][t];
    float m = 0.f;
#pragma unroll
    for (int u = 0; u < R; u++) {
      // NaN and infinities say nothing; past the rows read: not counted.
      v[u] = u < nr && fabsf(v[u]) < INFINITY ? v[u] : 0.f;
      mv = fmaxf(mv, fabsf(v[u]));
      sv = fmaf(v[u], v[u], sv);
      m = fmaf(v[u], inv, m);
    }
    if (in.mean) {
#pragma unroll
      for (int u = 0; u < R; u++) mc = u < nr ? fmaxf(mc, fabsf(v[u] - m)) : mc;
      sm = fmaf(m, m, sm);
      in.mean[t] = m;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    mv = fmaxf(mv, __shfl_xor(mv, o, 64));
    mc = fmaxf(mc, __shfl_xor(mc, o, 64));
    sv += __shfl_xor(sv, o, 64);
    sm += __shfl_xor(sm, o, 64);
  }
  if (lane == 0) wr[w] = make_float4(mv, mc, sv, sm);
  __syncthreads();
  mv = mc = sv = sm = 0.f;
  for (int i = 0; i < NT / 64; i++) {
    const float4 o = wr[i];
    mv = fmaxf(mv, o.x);
    mc = fmaxf(mc, o.y);
    sv += o.z;
    sm += o.w;
  }
  const bool use = in.mean && sv < INFINITY && sm > 0.f && 4.0f * (float)nr * sm >= sv;
  if (in.mean) {
    for (int t = (use ? d : 0) + tid; t < (int)mean_flag(d); t += NT) in.mean[t] = 0.f;
    if (tid == 0) in.mean[mean_flag(d)] = use ? 1.f : 0.f;
  }
  if (tid == 0) {
    int e = 8;  // zeros: scale 1
    const float m = use ? mc : mv;
    if (m > 0.f) frexpf(m, &e);  // m in [2^(e - 1), 2^e)
    if (use) {  // (rows that all but agree: any other row as long as they are stays in range)
      int ev;
      frexpf(mv, &ev);
      e = m > 0.f ? max(e, ev - 6) : ev - 6;
    }
    e = max(max(-50, in.emin), min(e, 60));  // two inverse scales' product stays a normal f32
    in.out[0] = ldexpf(1.0f, 8 - e);
    in.out[1] = ldexpf(1.0f, e - 8);
  }
}

// Rows ids[lo + g] (lo + g without ids; an id >= nx reads row 0) for g < n,
// less `mean` when given, as fp16 lines (emh_lines.h) in o.out, in selection
// order; o.norm[g] = (their squares, the residual), f32 sums in any order. With
// BOTH, the rows themselves as lines in p, too, unless the mean is all zeros
// (they would be the same: the screen reads o's instead). With part: block b writes the
// largest square of its rows, with cnorm the largest cnorm[g], the largest
// residual and the largest |x|^2 (f32 bits; a NaN wins) to part[4 b ..].
// Block b takes rows 8 b .. 8 b + 7, two per wave. HBM-bound: a wave reads a
// row in 256-dimension segments, 16 contiguous bytes per lane, and eight lanes
// fill one 64-byte line; the wave's two rows share a cache line in each slab.
constexpr int NARROW_U = 4;
template <bool VEC4, bool MEAN, bool BOTH>
__global__ __launch_bounds__(256) void k_lines(const float* __restrict__ x, size_t nx, int d,
                                               const uint32_t* __restrict__ ids, size_t lo,
                                               size_t n, const LinesOut o, const LinesOut p,
                                               const float* __restrict__ mean,
                                               const float* __restrict__ cnorm,
                                               uint32_t* __restrict__ part) {
  static_assert(MEAN || !BOTH, "two lines of a row only where they differ");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int d32 = (d + LINE_DIMS - 1) / LINE_DIMS, nseg = (d32 + 7) >> 3;
  const int js = lane >> 3, q = lane & 7;
  const float s = o.scale[0], sp = BOTH ? p.scale[0] : 0.f;
  const bool both = BOTH && mean[mean_flag(d)] != 0.f;
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
  auto square = [](float4 v, float a) __attribute__((always_inline)) {
    return fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, fmaf(v.x, v.x, a))));
  };
  // Squares and residuals: the lines' (sv, rv), the rows' (sx, rx with BOTH).
  float sv[2] = {0.f, 0.f}, rv[2] = {0.f, 0.f}, sx[2] = {0.f, 0.f}, rx[2] = {0.f, 0.f};
#pragma unroll 3
  for (int sg = 0; sg < nseg; sg++) {
    const int j = 8 * sg + js;
    if (j >= d32) break;
    const int col = LINE_DIMS * j + 4 * q;
    float4 v[2], m = make_float4(0.f, 0.f, 0.f, 0.f);
    if (MEAN) m = *reinterpret_cast<const float4*>(mean + col);
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
      const size_t at = ((size_t)j * n + g[i]) * LINE_BYTES + 8 * q;
      if (MEAN) {
        sx[i] = square(v[i], sx[i]);
        if (both) {
          const uint2 hv = line_quad(v[i], sp, rx[i]);
          if (valid[i]) *reinterpret_cast<uint2*>((char*)p.out + at) = hv;
        }
        v[i] = make_float4(v[i].x - m.x, v[i].y - m.y, v[i].z - m.z, v[i].w - m.w);
      }
      sv[i] = square(v[i], sv[i]);
      const uint2 hv = line_quad(v[i], s, rv[i]);
      if (valid[i]) *reinterpret_cast<uint2*>((char*)o.out + at) = hv;
    }
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) {
      sv[i] += __shfl_xor(sv[i], k, 64);
      rv[i] += __shfl_xor(rv[i], k, 64);
      if (MEAN) sx[i] += __shfl_xor(sx[i], k, 64);
      if (both) rx[i] += __shfl_xor(rx[i], k, 64);
    }
    if (!MEAN) sx[i] = sv[i];
    if (valid[i] && lane == 0) {
      o.norm[g[i]] = make_float2(sv[i], rv[i]);
      if (both) p.norm[g[i]] = make_float2(sx[i], rx[i]);
    }
  }
  if (part) {
    uint32_t mx[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (valid[i]) {
        mx[0] = max(mx[0], __float_as_uint(sv[i]));
        if (cnorm) mx[1] = max(mx[1], __float_as_uint(cnorm[g[i]]));
        mx[2] = max(mx[2], __float_as_uint(rv[i]));
        mx[3] = max(mx[3], __float_as_uint(sx[i]));
      }
    }
    __shared__ uint32_t red[4][4];
    if (lane == 0) {
#pragma unroll
      for (int e = 0; e < 4; e++) red[e][w] = mx[e];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
      const uint32_t* r = red[threadIdx.x];
      part[4 * blockIdx.x + threadIdx.x] = max(max(r[0], r[1]), max(r[2], r[3]));
    }
  }
}

// k_lines of rows of at most 32 P dimensions (P = 1, 2 or 4), without mean and
// part: 8 P lanes hold a row, so that no lane idles, and a thread has four
// rows' loads in flight (65,536 x 32: 15.3 us with a wave a row, 5.5 here).
template <bool VEC4, int P>
__global__ __launch_bounds__(256) void k_lines_narrow(const float* __restrict__ x, size_t nx, int d,
                                                      const uint32_t* __restrict__ ids, size_t lo,
                                                      size_t n, const LinesOut o) {
  constexpr int G = 8 * P, RW = 64 / G, U = NARROW_U;  // lanes per row; rows per wave and step
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = (lane % G) >> 3, col = 4 * (lane % G);
  const size_t g0 = ((size_t)blockIdx.x * 4 + w) * (U * RW) + lane / G;
  const float s = o.scale[0];
  float4 v[U];
#pragma unroll
  for (int i = 0; i < U; i++) {
    const size_t g = g0 + (size_t)(i * RW);
    size_t id = 0;
    if (g < n) {
      id = ids ? (size_t)ids[lo + g] : lo + g;
      if (id >= nx) id = 0;
    }
    const float* r = x + id * (size_t)d;
    if (VEC4) {
      v[i] = col < d ? *reinterpret_cast<const float4*>(r + col) : make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
      v[i].x = col < d ? r[col] : 0.f;
      v[i].y = col + 1 < d ? r[col + 1] : 0.f;
      v[i].z = col + 2 < d ? r[col + 2] : 0.f;
      v[i].w = col + 3 < d ? r[col + 3] : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < U; i++) {
    const size_t g = g0 + (size_t)(i * RW);
    float sq = fmaf(v[i].w, v[i].w, fmaf(v[i].z, v[i].z, fmaf(v[i].y, v[i].y, v[i].x * v[i].x)));
    float rs = 0.f;
    const uint2 h = line_quad(v[i], s, rs);
    if (g < n && LINE_DIMS * j < d)
      *reinterpret_cast<uint2*>((char*)o.out + ((size_t)j * n + g) * LINE_BYTES + 8 * (lane & 7)) = h;
#pragma unroll
    for (int m = G / 2; m > 0; m >>= 1) {
      sq += __shfl_xor(sq, m, 64);
      rs += __shfl_xor(rs, m, 64);
    }
    if (g < n && lane % G == 0) o.norm[g] = make_float2(sq, rs);
  }
}

// out[0 .. 3] = the maxima of part[4 i .. 4 i + 3] over i < nparts.
__global__ __launch_bounds__(1024) void k_part_max4(const uint32_t* __restrict__ part,
                                                    size_t nparts, uint32_t* __restrict__ out) {
  constexpr int B = 8;
  __shared__ uint32_t wm[4][16];
  const int tid = threadIdx.x;
  uint32_t m[4] = {0u, 0u, 0u, 0u};
  for (size_t i0 = 0; i0 < nparts; i0 += 1024 * B) {
    uint4 v[B];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const size_t i = i0 + 1024 * (size_t)u + tid;
      v[u] = i < nparts ? reinterpret_cast<const uint4*>(part)[i] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < B; u++) {
      m[0] = max(m[0], v[u].x);
      m[1] = max(m[1], v[u].y);
      m[2] = max(m[2], v[u].z);
      m[3] = max(m[3], v[u].w);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    for (int o = 32; o > 0; o >>= 1) m[e] = max(m[e], (uint32_t)__shfl_xor((int)m[e], o, 64));
    if ((tid & 63) == 0) wm[e][tid >> 6] = m[e];
  }
  __syncthreads();
  if (tid < 4) {
    uint32_t r = 0u;
    for (int i = 0; i < 16; i++) r = max(r, wm[tid][i]);
    out[tid] = r;
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
  const unsigned nt = (unsigned)std::min<size_t>((d + 63) / 64 * 64, 1024);  // a column each
  hipLaunchKernelGGL(k_scales, dim3(b ? 2 : 1), dim3(nt), 0, c->stream, a, b ? *b : a, (int)d,
                     d <= 2048 ? SCALE_ROWS_READ : SCALE_ROWS_READ / 2, clear, nclear);
  EMH_HIP(hipGetLastError());
}

void launch_lines(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids, size_t lo,
                  size_t n, const LinesOut& o, const float* cnorm, uint32_t* part,
                  const float* mean, const LinesOut* also) {
  if (n == 0) return;
  EMH_ENSURE(d >= 1 && n < (1u << 31) && (mean || !also), "lines: shape out of range");
  if (d <= 128 && !mean && !part) {
    const int p = d <= 32 ? 1 : d <= 64 ? 2 : 4;
    auto kern = d % 4 == 0 ? (p == 1   ? k_lines_narrow<true, 1>
                              : p == 2 ? k_lines_narrow<true, 2>
                                       : k_lines_narrow<true, 4>)
                           : (p == 1   ? k_lines_narrow<false, 1>
                              : p == 2 ? k_lines_narrow<false, 2>
                                       : k_lines_narrow<false, 4>);
    const size_t rows = (size_t)(4 * NARROW_U * 8 / p);  // per block
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + rows - 1) / rows)), dim3(256), 0, c->stream, x,
                       nx, (int)d, ids, lo, n, o);
    EMH_HIP(hipGetLastError());
    return;
  }
  auto kern = d % 4 == 0 ? (also   ? k_lines<true, true, true>
                            : mean ? k_lines<true, true, false>
                                   : k_lines<true, false, false>)
                         : (also   ? k_lines<false, true, true>
                            : mean ? k_lines<false, true, false>
                                   : k_lines<false, false, false>);
  hipLaunchKernelGGL(kern, dim3((unsigned)lines_blocks(n)), dim3(256), 0, c->stream, x, nx, (int)d,
                     ids, lo, n, o, also ? *also : o, mean, cnorm, part);
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
  // The data's lines less their mean (with their norms, residuals and the
  // maxima of both), and the queries' as they are: of the same rows, in one
  // pass over them.
  const bool same = q == data && m == n;
  float* sc = c->scales + 2 * SCALE_CENTS;
  float* sx = c->scales + 2 * SCALE_ROWS;
  float* mean = (float*)c->cmean.get(mean_floats(d) * 4);
  const ScaleIn is{data, n, nullptr, 0, n, sc, -50, mean}, iq{q, m, nullptr, 0, m, sx, -50};
  launch_scales(c, d, is, &iq, clear, nclear);
  const LinesOut xo{sc, c->csplit.get(lines_bytes(n, d)), (float2*)c->csplit_norm.get(n * 8)};
  const LinesOut qo{sx, c->xsplit.get(lines_bytes(m, d)), (float2*)c->xsplit_norm.get(m * 8)};
  // Past PART_MAX_ONCE partials, one workgroup reduces them ahead of the
  // screen, whose every block would otherwise read them all.
  const size_t hb = lines_blocks(n);
  uint32_t* part = (uint32_t*)c->csplit_part.get((hb + 1) * 16);
  launch_lines(c, data, n, d, nullptr, 0, n, xo, nullptr, part, mean, same ? &qo : nullptr);
  s->part = part;
  s->nparts = (int)hb;
  if (hb > PART_MAX_ONCE) {
    launch_part_max4(c, part, hb, part + 4 * hb);
    s->part = part + 4 * hb;
    s->nparts = 1;
  }
  if (!same) launch_lines(c, q, m, d, nullptr, 0, m, qo);
  s->cs = xo.out;
  s->xs = qo.out;
  s->xn = qo.norm;
  s->mean = mean;
  s->same = nullptr;
  if (same) {
    s->same = mean + mean_flag(d);
    s->cn = xo.norm;
  }
  s->sx = sx;
  s->sc = sc;
  s->m = m;
  s->n = n;
  s->d = d;
}

int screen5_knn(emh_ctx* c, const float* q, size_t m, const float* data, size_t n, size_t d,
                size_t kk, bool exclude_self, Cand** cand_out, int* L_out, float** bound_out,
                const float** mean_out) {
  Split5 s;
  split5(c, q, m, data, n, d, c->small, 3, &s);
  const int row_tiles = (int)((m + T5 - 1) / T5);
  const int ntiles = (int)((n + T5 - 1) / T5);
  // Parts (data-tile ranges) where they fill waves of blocks better: up to
  // MAX_PARTS5, so that a few query tiles still fill the chip (2,000 queries
  // against 100,000 x 512: 8 parts gave 64 blocks, 0.94 ms; 31 take 0.45).
  int parts = parts5(row_tiles, ntiles, std::max(c->cus, 1), MAX_PARTS5, 2.0);
  const int tpp = (ntiles + parts - 1) / parts;
  // Lists of 24 leave room for the near-ties of at most 12 neighbours: among
  // 1,000,000 unit rows with a common mean (d = 32) 10 queue 2,557 rows (160 ms),
  // 16 queued 311,078 (732 ms; 171 with lists of 40, 99 rows). Where both hold
  // everything 40 entries cost 1%.
  const int L = kk > (size_t)LK_KK ? LK5 : LK;
  Cand* cand = (Cand*)c->cand.get((size_t)parts * m * L * sizeof(Cand));
  float* bound = (float*)c->xnorm.get(2 * m * 4);
  // A launch's threads each keep a log (1 MB a block): launches of whole waves
  // of blocks, at most four: 1 GB on 256 CUs, kept with the context. One wave a
  // launch (256 MB) takes 8% longer at 180,000 x 256 and 5% at 108,000 x 256,
  // whose waves' ends then wait for one another (500,000 x 384: 1% less).
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
  a.L = L;
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
  a.same = s.same;
  a.cn = s.cn;
  a.nx = m;
  for (int r = 0; r < row_tiles; r += rt_step) {
    const size_t q0 = (size_t)r * T5, q1 = std::min((size_t)(r + rt_step) * T5, m);
    a.lo = q0;
    a.nrows = (int)(q1 - q0);
    a.cand = cand + q0 * parts * L;
    a.bound = bound + q0;
    const unsigned blocks = (unsigned)((q1 - q0 + T5 - 1) / T5 * parts);
    if (exclude_self)
      launch5<KNN_SELF, false>(c, blocks, a);
    else
      launch5<KNN, false>(c, blocks, a);
  }
  *cand_out = cand;
  *L_out = L;
  *bound_out = bound;
  *mean_out = s.mean;
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
  a.same = s.same;
  a.cn = s.cn;
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
