// The exact scans behind the MFMA screen (emh_screen.hip) and its check
// (emh_rescore.hip), for the rows the check could not settle:
//
//  k_exact1    top-1: the rows' scan over all centroids, split into
//              (4 rows x 64 centroids) items; the block that completes a row
//              group's last item reduces the group's rows (one launch). For
//              a selection without the screen, and queued rows when d % 4 != 0;
//  k_queued1   top-1 for the rows the check queues (d % 4 == 0): short
//              (4 rows x 16 centroids) items, one burst of DMA copies and one
//              chain per lane each, the winners folded by 64-bit atomics; long
//              queues in tiles of 128 x 128;
//  k_small1    top-1 for a small direct selection against at most 64
//              centroids (d % 4 == 0): a block holds all of them and its rows,
//              so a row's winner is found inside a wave;
//  k_exactk    top-k: tiles of queued queries x data rows, the kk best kept on
//              the way.
//
// Float order (the reference CPU backend, assign/fused.rs + assign.rs):
// dot = fma chain over t = 0..d-1 from +0; L2 key = cnorm[j] - 2 dot (two
// roundings); |x|^2 = sequential sum of rounded squares; score = dot (IP) or
// max(|x|^2 + key, 0) (L2); ties to the lower id; a key that is NaN or +inf
// never wins, and a row where nothing wins gets label 0 and the initial score.

#include <algorithm>

#include "emh_select.h"

namespace emh {
namespace {

constexpr int WAVE = 64;

// ------------------------------------------------------------- exact top-1
// Item = (group of RG rows, chunk of CJ centroids): one wave, lane = centroid,
// RG chains per lane. The dimensions go in tiles of TD: a tile of the chunk's
// centroids and the group's rows is loaded into registers (every load of the
// tile in flight at once) while the previous tile is consumed from LDS.
constexpr int CJ = 64, RG = 4, TD = 64, TDP = TD + 4;
constexpr int CL4 = CJ * TD / 4 / WAVE;  // float4 loads per lane per tile (centroids)
constexpr int XL4 = RG * TD / 4 / WAVE;  // float4 loads per lane per tile (rows)

// Columns col..col+3 of a row, zero past d. Branch-free: every load is issued
// (at a clamped column) and the zeros are selected afterwards, so a tile's
// loads stay in flight together instead of each waiting on a branch.
template <bool VEC4>
__device__ __forceinline__ float4 load_tile4(const float* row, int col, int d, bool valid = true) {
  if (VEC4) {  // d % 4 == 0: col < d implies col + 4 <= d
    const float4 v = *reinterpret_cast<const float4*>(row + min(col, d - 4));
    const bool in = valid && col < d;
    return make_float4(in ? v.x : 0.f, in ? v.y : 0.f, in ? v.z : 0.f, in ? v.w : 0.f);
  }
  float e[4];
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const float v = row[min(col + u, d - 1)];
    e[u] = valid && col + u < d ? v : 0.f;
  }
  return make_float4(e[0], e[1], e[2], e[3]);
}

// The end of row group g (rows g*RG ...): each row's smallest chunk minimum
// (lower id on ties; a row where nothing wins gets label 0 and the initial
// score) and, for L2, its |x|^2 as a sequential sum of rounded squares: the
// wave stages the group's squares in LDS (sq, RG rows of SEG floats per pass)
// and lane r adds row r's in order. One wave.
constexpr int SEG = CJ * TDP / RG;
__device__ __attribute__((noinline)) void finish_group(const float* __restrict__ x, size_t nx, int d,
                             const uint32_t* __restrict__ ids, size_t lo,
                             const uint32_t* __restrict__ list, uint32_t* __restrict__ small,
                             int nch, int ip, const Cand* __restrict__ partial, int g, int nrows,
                             float* sq, uint32_t* __restrict__ labels,
                             float* __restrict__ scores) {
  const int lane = threadIdx.x;
  float mybest = INFINITY;  // lane r < RG: row r's best key and id
  uint32_t mybid = NONE;
  size_t myp = 0;
  const float* xr[RG];
  bool ok[RG];
#pragma unroll
  for (int r = 0; r < RG; r++) {
    const int f = g * RG + r;
    ok[r] = false;
    xr[r] = x;
    if (f >= nrows) continue;  // uniform
    const size_t p = list ? (size_t)list[f] : lo + (size_t)f;
    const size_t xid = ids ? (size_t)ids[p] : p;
    if (xid >= nx) {
      if (lane == 0) small[SW_BAD_ID] = 1;
      continue;
    }
    ok[r] = true;
    xr[r] = x + xid * (size_t)d;
    float best = INFINITY;
    uint32_t bid = NONE;
    for (int q = lane; q < nch; q += WAVE) {
      const Cand c = partial[(size_t)f * nch + q];
      if (c.id != NONE && (c.key < best || (c.key == best && c.id < bid))) {
        best = c.key;
        bid = c.id;
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const float b2 = __shfl_xor(best, o, WAVE);
      const uint32_t i2 = __shfl_xor(bid, o, WAVE);
      if (i2 != NONE && (b2 < best || (b2 == best && i2 < bid))) {
        best = b2;
        bid = i2;
      }
    }
    if (lane == r) {
      mybest = best;
      mybid = bid;
      myp = p;
    }
  }
  float xn = 0.f;
  if (!ip) {
    for (int t0 = 0; t0 < d; t0 += SEG) {
      const int tl = min(SEG, d - t0);
#pragma unroll
      for (int r = 0; r < RG; r++) {
        if (!ok[r]) continue;  // uniform
        for (int i0 = 0; i0 < tl; i0 += WAVE * 8) {
          float v[8];
#pragma unroll
          for (int u = 0; u < 8; u++) {
            const int i = i0 + lane + WAVE * u;
            v[u] = i < tl ? xr[r][t0 + i] : 0.f;
          }
#pragma unroll
          for (int u = 0; u < 8; u++) {
            const int i = i0 + lane + WAVE * u;
            if (i < tl) sq[r * SEG + i] = v[u] * v[u];
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane < RG && ok[lane]) {  // in order, 16 LDS reads in flight
        const float* row = sq + lane * SEG;
        int i = 0;
        for (; i + 16 <= tl; i += 16) {
          float v[16];
#pragma unroll
          for (int u = 0; u < 16; u++) v[u] = row[i + u];
#pragma unroll
          for (int u = 0; u < 16; u++) xn = xn + v[u];
        }
        for (; i < tl; i++) xn = xn + row[i];
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (lane < RG && ok[lane]) {
    if (mybid == NONE) {
      mybid = 0;
      mybest = INFINITY;
    }
    labels[myp] = mybid;
    scores[myp] = ip ? -mybest : fmaxf(xn + mybest, 0.0f);
  }
}

// One wave.
template <bool VEC4>
__device__ __forceinline__ void exact_items(
    const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids, size_t lo,
    int nrows, const uint32_t* __restrict__ list, uint32_t* __restrict__ small,
    const float* __restrict__ cents, const float* __restrict__ cnorm, int k, int ip,
    Cand* __restrict__ partial, uint32_t* __restrict__ tickets, uint32_t* __restrict__ labels,
    float* __restrict__ scores) {
  __shared__ __attribute__((aligned(16))) float ct[CJ * TDP];
  __shared__ __attribute__((aligned(16))) float xt[RG * TD];
  __shared__ uint32_t xid_s[RG];
  __shared__ int last_s;
  const int nch = (k + CJ - 1) / CJ;
  const int ngr = (nrows + RG - 1) / RG;
  const int ntd = (d + TD - 1) / TD;
  const int lane = threadIdx.x;
  const int c4 = lane % (TD / 4), r0 = lane / (TD / 4);  // this lane's float4 column, first row
  constexpr int RSTEP = WAVE / (TD / 4);                  // rows per load instruction
  for (int item = blockIdx.x; item < ngr * nch; item += gridDim.x) {
    const int g = item / nch, q = item - g * nch;
    if (lane < RG) {
      const int f = g * RG + lane;
      uint32_t xid = NONE;
      if (f < nrows) {
        const size_t p = list ? (size_t)list[f] : lo + (size_t)f;
        const size_t id = ids ? (size_t)ids[p] : p;
        xid = id < nx ? (uint32_t)id : NONE;
      }
      xid_s[lane] = xid;
    }
    __syncthreads();
    const float* xp[XL4];
    bool xv[XL4];
#pragma unroll
    for (int u = 0; u < XL4; u++) {
      const uint32_t xid = xid_s[r0 + RSTEP * u];
      xv[u] = xid != NONE;
      xp[u] = x + (size_t)(xv[u] ? xid : 0) * d;
    }
    float4 cr[CL4], xr[XL4];
    auto gload = [&](int t0) {
      const int col = t0 + 4 * c4;
#pragma unroll
      for (int u = 0; u < CL4; u++)
        cr[u] = load_tile4<VEC4>(cents + (size_t)min(q * CJ + r0 + RSTEP * u, k - 1) * d, col, d);
#pragma unroll
      for (int u = 0; u < XL4; u++)
        xr[u] = load_tile4<VEC4>(xp[u], col, d, xv[u]);  // xp[u] is row 0 when invalid
    };
    float acc[RG];
#pragma unroll
    for (int r = 0; r < RG; r++) acc[r] = 0.f;
    gload(0);
    for (int tile = 0; tile < ntd; tile++) {
#pragma unroll
      for (int u = 0; u < CL4; u++)
        *reinterpret_cast<float4*>(&ct[(r0 + RSTEP * u) * TDP + 4 * c4]) = cr[u];
#pragma unroll
      for (int u = 0; u < XL4; u++)
        *reinterpret_cast<float4*>(&xt[(r0 + RSTEP * u) * TD + 4 * c4]) = xr[u];
      __syncthreads();
      const int t0 = tile * TD;
      if (tile + 1 < ntd) gload(t0 + TD);
      const int tl = min(TD, d - t0);
      const float* crow = &ct[lane * TDP];
      int tt = 0;
#pragma unroll 4
      for (; tt + 4 <= tl; tt += 4) {
        const float4 cv = *reinterpret_cast<const float4*>(crow + tt);
#pragma unroll
        for (int r = 0; r < RG; r++) {
          const float4 v = *reinterpret_cast<const float4*>(&xt[r * TD + tt]);
          acc[r] = fmaf(v.x, cv.x, acc[r]);
          acc[r] = fmaf(v.y, cv.y, acc[r]);
          acc[r] = fmaf(v.z, cv.z, acc[r]);
          acc[r] = fmaf(v.w, cv.w, acc[r]);
        }
      }
      for (; tt < tl; tt++) {
        const float cv = crow[tt];
#pragma unroll
        for (int r = 0; r < RG; r++) acc[r] = fmaf(xt[r * TD + tt], cv, acc[r]);
      }
      __syncthreads();
    }
    const int j = q * CJ + lane;
#pragma unroll
    for (int r = 0; r < RG; r++) {
      float kx = INFINITY;
      uint32_t id = NONE;
      if (j < k && xid_s[r] != NONE) {
        if (ip) {
          kx = -acc[r];
        } else {
          float two = 2.0f * acc[r];
          kx = cnorm[j] - two;
        }
        id = (uint32_t)j;
        if (!(kx < INFINITY)) {  // NaN or +inf never wins
          kx = INFINITY;
          id = NONE;
        }
      }
      for (int o = 32; o > 0; o >>= 1) {
        float k2 = __shfl_xor(kx, o, WAVE);
        uint32_t i2 = __shfl_xor(id, o, WAVE);
        if (k2 < kx || (k2 == kx && i2 < id)) {
          kx = k2;
          id = i2;
        }
      }
      const int f = g * RG + r;
      if (lane == 0 && f < nrows) partial[(size_t)f * nch + q] = Cand{kx, id};
    }
    // The group's ticket: the block that completes its last chunk finishes it.
    if (lane == 0) {
      __threadfence();
      last_s = atomicAdd(&tickets[g], 1u) == (uint32_t)(nch - 1);
    }
    __syncthreads();
    if (last_s) {
      __threadfence();
      finish_group(x, nx, d, ids, lo, list, small, nch, ip, partial, g, nrows, ct, labels, scores);
      if (lane == 0) tickets[g] = 0;
    }
    __syncthreads();
  }
}

template <bool VEC4>
__global__ __launch_bounds__(64) void k_exact1(
    const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids, size_t lo,
    int n, uint32_t* __restrict__ small, const float* __restrict__ cents,
    const float* __restrict__ cnorm, int k, int ip, Cand* __restrict__ partial,
    uint32_t* __restrict__ tickets, uint32_t* __restrict__ labels, float* __restrict__ scores) {
  exact_items<VEC4>(x, nx, d, ids, lo, n, nullptr, small, cents, cnorm, k, ip, partial, tickets,
                    labels, scores);
}

// ------------------------------------------------- exact top-1, queued rows
// The check queues few rows (often one to eight per batch), so this scan is
// built for latency: many short items, each a single wave that copies its
// data to LDS in one burst and then runs one fma chain per lane.
//
// Item = (group of QR rows, chunk of QJ centroids), plus one norm item per
// group for L2. Lane (j = lane / QR, r = lane % QR) runs row r's chain against
// centroid j of the chunk. The dimensions go in phases of up to QPH: the
// phase's slice of the chunk's centroids and of the group's rows is copied to
// LDS by the DMA path (global_load_lds, 16 bytes per lane, all instructions in
// flight together), then the chains read it. LDS slots (16 bytes, 4 dims):
// centroids at u * QJ + j, rows at u * QR + r for dims 4u..4u+3 of the phase,
// so a read touches consecutive slots (no bank conflicts) and lanes sharing a
// centroid or a row read it by broadcast.
//
// Each item folds its chunk's winners into one 64-bit word per row with an
// atomic max of the complement of (ordered key << 32 | id << 1 | sign of a
// zero key): the smallest key wins, then the lower id (keys -0 and +0 are
// equal, as in the reference's comparison; the sign bit restores the winner's
// own zero), so the reduction is exact and independent of the item order. The
// item that takes a group's last ticket writes the group's labels and scores
// and leaves the words and the ticket at zero for the next launch.
constexpr int QR = 4, QJ = 16, QPH = 768;
constexpr int QU = QPH / 4;  // 4-dim slots per phase

__device__ __forceinline__ uint64_t pack_best(float key, uint32_t id) {
  uint32_t b = __float_as_uint(key), z = 0;
  if (key == 0.0f) {  // -0 and +0 compare equal: one code, the sign kept apart
    z = b >> 31;
    b = 0u;
  }
  const uint32_t o = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ~(((uint64_t)o << 32) | ((uint64_t)id << 1) | z);
}

__device__ __forceinline__ bool unpack_best(uint64_t w, float& key, uint32_t& id) {
  if (w == 0) return false;
  const uint64_t v = ~w;
  const uint32_t o = (uint32_t)(v >> 32);
  uint32_t b = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
  if (b == 0u && (v & 1u)) b = 0x80000000u;
  key = __uint_as_float(b);
  id = (uint32_t)((v >> 1) & 0x7fffffffu);
  return true;
}

// Four dimensions (16 bytes) of a lane's row into its slot of LDS (`slots` +
// the lane): by DMA where rows start at multiples of 16 bytes (AL), else
// through registers (a wrapped buffer may start at any float).
typedef float v4f __attribute__((ext_vector_type(4)));
template <bool AL>
__device__ __forceinline__ void slot_copy(const float* src, v4f* slots) {
  if (AL) {
    __builtin_amdgcn_global_load_lds(src, slots, 16, 0, 0);
  } else {
    v4f v = {src[0], src[1], src[2], src[3]};
    slots[threadIdx.x & 63] = v;
  }
}

// Long queues (more than MANY row-centroid pairs: rows crowded beyond what the
// screen's bound can tell apart) take tiles instead: 128 rows against 128
// centroids at a time, a thread 8 x 8 chains, slabs of MD dimensions
// double-buffered in LDS. Bound by the fmas. Item = (128 rows, a range of
// centroid tiles), its winners folded by the same words and tickets (one a row
// tile); the first item of a row tile also runs the rows' |x|^2 for L2.
// 65,536 rows against 1,024 centroids, d = 768, every row queued: 1.7 ms for the
// whole call; as short items, 27.8.
constexpr int MR = 128, MD = 16, MP = MR + 4;
constexpr uint64_t MANY = 1u << 20;

struct QueuedLds {
  float xs[2][MD][MP], cs[2][MD][MP];  // a slab of the rows, of the centroids
  uint32_t rid[MR];
  int last;
};

template <bool AL>
__device__ __forceinline__ void queued_tiles(
    QueuedLds& L, const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids,
    int nrows, const uint32_t* __restrict__ list, uint32_t* __restrict__ small,
    const float* __restrict__ cents, const float* __restrict__ cnorm, int k, int ip,
    unsigned long long* __restrict__ best, uint32_t* __restrict__ tickets,
    float* __restrict__ xnq, uint32_t* __restrict__ labels, float* __restrict__ scores,
    uint32_t* __restrict__ tcnt, uint32_t* __restrict__ tcounts, size_t tlo, size_t tstride) {
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int nrt = (nrows + MR - 1) / MR, nct = (k + MR - 1) / MR;
  const int want = min(nct, max(1, ((int)gridDim.x + nrt - 1) / nrt));
  const int tpp = (nct + want - 1) / want, parts = (nct + tpp - 1) / tpp;
  for (int item = blockIdx.x; item < nrt * parts; item += gridDim.x) {
    const int rt = item / parts, q = item - rt * parts;
    __syncthreads();  // the previous item is done with L
    if (tid < MR) {
      const int f = rt * MR + tid;
      uint32_t xid = NONE;
      if (f < nrows) {
        const size_t p = (size_t)list[f];
        const size_t id = ids ? (size_t)ids[p] : p;
        if (id < nx)
          xid = (uint32_t)id;
        else
          small[SW_BAD_ID] = 1;
      }
      L.rid[tid] = xid;
    }
    __syncthreads();
    // Loader: 16-byte piece e = 256 u + tid of a slab is row e / 4, dimensions
    // 4 (e % 4) .. + 3 (AL: d % 4 == 0, all of them in or all past d).
    const float* xr[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const uint32_t r = L.rid[(256 * u + tid) >> 2];
      xr[u] = x + (size_t)(r == NONE ? 0u : r) * d + 4 * (tid & 3);
    }
    v4f xv[2], cv[2];
    auto piece = [&](const float* p, int t) __attribute__((always_inline)) {
      v4f v = {0.f, 0.f, 0.f, 0.f};
      if (AL) {
        if (t < d) v = *reinterpret_cast<const v4f*>(p);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (t + e < d) v[e] = p[e];
      }
      return v;
    };
    auto load = [&](int ct, int t0) __attribute__((always_inline)) {
      const int t = t0 + 4 * (tid & 3);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        xv[u] = piece(xr[u] + t0, t);
        const int j = min(ct * MR + ((256 * u + tid) >> 2), k - 1);
        cv[u] = piece(cents + (size_t)j * d + t, t);
      }
    };
    auto store = [&](int b) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int r = (256 * u + tid) >> 2, t = 4 * (tid & 3);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          L.xs[b][t + e][r] = xv[u][e];
          L.cs[b][t + e][r] = cv[u][e];
        }
      }
    };
    float bk[8];
    uint32_t bi[8];
#pragma unroll
    for (int a = 0; a < 8; a++) {
      bk[a] = INFINITY;
      bi[a] = NONE;
    }
    float nrm = 0.f;
    const int c0 = q * tpp, c1 = min(nct, c0 + tpp);
    for (int ct = c0; ct < c1; ct++) {
      float acc[8][8];
#pragma unroll
      for (int a = 0; a < 8; a++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[a][e] = 0.f;
      auto dim = [&](int b, int t) __attribute__((always_inline)) {
        float xa[8], ca[8];
#pragma unroll
        for (int a = 0; a < 8; a++) xa[a] = L.xs[b][t][ty * 8 + a];
#pragma unroll
        for (int e = 0; e < 8; e++) ca[e] = L.cs[b][t][(e >> 2) * 64 + tx * 4 + (e & 3)];
#pragma unroll
        for (int a = 0; a < 8; a++)
#pragma unroll
          for (int e = 0; e < 8; e++) acc[a][e] = fmaf(xa[a], ca[e], acc[a][e]);
      };
      load(ct, 0);
      store(0);
      __syncthreads();
      for (int t0 = 0, b = 0; t0 < d; t0 += MD, b ^= 1) {
        const bool more = t0 + MD < d;
        if (more) load(ct, t0 + MD);
        const int tn = min(MD, d - t0);  // dimensions past d never enter a chain
        if (tn == MD) {
#pragma unroll
          for (int t = 0; t < MD; t++) dim(b, t);
        } else {
          for (int t = 0; t < tn; t++) dim(b, t);
        }
        if (!ip && q == 0 && ct == 0 && tid < MR)
          for (int t = 0; t < tn; t++) {
            const float v = L.xs[b][t][tid];
            nrm = nrm + v * v;
          }
        if (more) store(b ^ 1);
        __syncthreads();
      }
      // A thread's columns come in rising order: the lower id wins ties.
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int j = ct * MR + (e >> 2) * 64 + tx * 4 + (e & 3);
        if (j < k) {
          const float cn = ip ? 0.f : cnorm[j];
#pragma unroll
          for (int a = 0; a < 8; a++) {
            const float key = ip ? -acc[a][e] : cn - 2.0f * acc[a][e];
            if (key < bk[a]) {  // (NaN or +inf never)
              bk[a] = key;
              bi[a] = (uint32_t)j;
            }
          }
        }
      }
    }
#pragma unroll
    for (int a = 0; a < 8; a++) {
      uint64_t w = bi[a] == NONE ? 0ull : pack_best(bk[a], bi[a]);
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const uint64_t w2 = __shfl_xor(w, o, WAVE);
        w = w2 > w ? w2 : w;
      }
      const int f = rt * MR + ty * 8 + a;
      if (tx == 0 && w != 0 && f < nrows) atomicMax(&best[f], (unsigned long long)w);
    }
    const int f = rt * MR + tid;
    if (!ip && q == 0 && tid < MR && f < nrows)
      __hip_atomic_store(&xnq[f], nrm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence();
    __syncthreads();
    if (tid == 0) L.last = atomicAdd(&tickets[rt], 1u) == (uint32_t)(parts - 1);
    __syncthreads();
    if (!L.last) continue;
    __threadfence();
    if (tid < MR && f < nrows) {
      const unsigned long long w = atomicExch(&best[f], 0ull);
      if (L.rid[tid] != NONE) {
        float bkey = INFINITY;
        uint32_t bid = 0;  // nothing wins: label 0 and the initial score
        unpack_best(w, bkey, bid);
        const size_t p = (size_t)list[f];
        labels[p] = bid;
        scores[p] = ip ? -bkey
                       : fmaxf(__hip_atomic_load(&xnq[f], __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT) + bkey, 0.0f);
        if (tcnt) {
          atomicAdd(&tcnt[(size_t)bid * tstride + (p - tlo) / TALLY_CP], 1u);
          atomicAdd(&tcounts[bid], 1u);
        }
      }
    }
    if (tid == 0) tickets[rt] = 0;
  }
}

// Queued rows of any width (d % 4 != 0): short items as k_exact1's by the first
// wave, or, with `best`, tiles.
__global__ __launch_bounds__(256) void k_exact1_list(
    const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids, size_t lo,
    const uint32_t* __restrict__ list, uint32_t* __restrict__ small,
    const float* __restrict__ cents, const float* __restrict__ cnorm, int k, int ip,
    Cand* __restrict__ partial, uint32_t* __restrict__ tickets,
    unsigned long long* __restrict__ best, float* __restrict__ xnq, uint32_t* __restrict__ labels,
    float* __restrict__ scores) {
  __shared__ __attribute__((aligned(16))) QueuedLds tiles;
  const int nrows = (int)small[SW_FALLBACK_COUNT];
  if (blockIdx.x == 0 && threadIdx.x == 0) small[SW_FALLBACK_TOTAL] += (uint32_t)nrows;
  if (best && (uint64_t)nrows * (uint64_t)k > MANY) {
    queued_tiles<false>(tiles, x, nx, d, ids, nrows, list, small, cents, cnorm, k, ip, best,
                        tickets, xnq, labels, scores, nullptr, nullptr, 0, 0);
    return;
  }
  if (threadIdx.x >= WAVE) return;
  exact_items<false>(x, nx, d, ids, lo, nrows, list, small, cents, cnorm, k, ip, partial, tickets,
                     labels, scores);
}

// (Four waves; short items take the first alone.)
template <bool AL>
__global__ __launch_bounds__(256) void k_queued1(
    const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids, size_t lo,
    int n_direct, const uint32_t* __restrict__ list, uint32_t* __restrict__ small,
    const float* __restrict__ cents, const float* __restrict__ cnorm, int k, int ip,
    unsigned long long* __restrict__ best, uint32_t* __restrict__ tickets,
    float* __restrict__ xnq, uint32_t* __restrict__ labels, float* __restrict__ scores,
    uint32_t* __restrict__ tcnt, uint32_t* __restrict__ tcounts, size_t tlo, size_t tstride) {
  __shared__ __attribute__((aligned(16))) char lds[(QU * QJ + QU * QR) * sizeof(v4f)];
  static_assert(sizeof(QueuedLds) <= sizeof(lds), "tiles");
  v4f* const cs = reinterpret_cast<v4f*>(lds);
  v4f* const xs = cs + QU * QJ;
  __shared__ uint32_t xid_s[QR];
  // Queued rows (list: positions, count on the device), or a direct
  // selection of n_direct rows at positions lo, lo + 1, ...
  const int nrows = list ? (int)small[SW_FALLBACK_COUNT] : n_direct;
  if (list && blockIdx.x == 0 && threadIdx.x == 0) small[SW_FALLBACK_TOTAL] += (uint32_t)nrows;
  if (list && (uint64_t)nrows * (uint64_t)k > MANY) {
    queued_tiles<AL>(*reinterpret_cast<QueuedLds*>(lds), x, nx, d, ids, nrows, list, small, cents,
                     cnorm, k, ip, best, tickets, xnq, labels, scores, tcnt, tcounts, tlo,
                     tstride);
    return;
  }
  if (threadIdx.x >= WAVE) return;
  const int nch = (k + QJ - 1) / QJ;
  const int per = nch + (ip ? 0 : 1);  // items per group (the last one: |x|^2)
  const int ngr = (nrows + QR - 1) / QR;
  const int lane = threadIdx.x;
  const int j = lane / QR, r = lane % QR;
  for (int item = blockIdx.x; item < ngr * per; item += gridDim.x) {
    const int g = item / per, q = item - g * per;
    const bool norm = q == nch;
    if (lane < QR) {
      const int f = g * QR + lane;
      uint32_t xid = NONE;
      if (f < nrows) {
        const size_t p = list ? (size_t)list[f] : lo + (size_t)f;
        const size_t id = ids ? (size_t)ids[p] : p;
        if (id < nx)
          xid = (uint32_t)id;
        else
          small[SW_BAD_ID] = 1;
      }
      xid_s[lane] = xid;
    }
    __syncthreads();
    // This lane's DMA sources: rows (slot l of each row instruction covers
    // dims 4 * (16 i + l / QR) of row l % QR) and centroids (dims
    // 4 * (4 i + l / QJ) of centroid l % QJ).
    const uint32_t xr = xid_s[lane % QR];
    const float* xrow = x + (size_t)(xr == NONE ? 0u : xr) * d;
    const float* crow = cents + (size_t)min(q * QJ + lane % QJ, k - 1) * d;
    float acc = 0.f;
    for (int t0 = 0; t0 < d; t0 += QPH) {
      const int nu = min(QU, (d - t0) / 4);  // d % 4 == 0
      for (int i = 0; i < (nu + 15) / 16; i++) {
        const int col = min(t0 + 4 * (16 * i + lane / QR), d - 4);
        slot_copy<AL>(xrow + col, &xs[i * 64]);
      }
      if (!norm)
        for (int i = 0; i < (nu + 3) / 4; i++) {
          const int col = min(t0 + 4 * (4 * i + lane / QJ), d - 4);
          slot_copy<AL>(crow + col, &cs[i * 64]);
        }
      __syncthreads();  // waits for the copies
      if (norm) {  // |x|^2 of row r: sequential sum of rounded squares
#pragma unroll 8
        for (int u = 0; u < nu; u++) {
          const v4f v = xs[u * QR + r];
          acc = acc + v.x * v.x;
          acc = acc + v.y * v.y;
          acc = acc + v.z * v.z;
          acc = acc + v.w * v.w;
        }
      } else {
#pragma unroll 8
        for (int u = 0; u < nu; u++) {
          const v4f cv = cs[u * QJ + j];
          const v4f v = xs[u * QR + r];
          acc = fmaf(v.x, cv.x, acc);
          acc = fmaf(v.y, cv.y, acc);
          acc = fmaf(v.z, cv.z, acc);
          acc = fmaf(v.w, cv.w, acc);
        }
      }
      __syncthreads();  // the next phase's copies overwrite these slots
    }
    const int f = g * QR + r;
    const bool valid = f < nrows && xid_s[r] != NONE;
    if (norm) {
      if (j == 0 && valid) xnq[f] = acc;
    } else {
      const int cj = q * QJ + j;
      float kx = INFINITY;
      uint32_t id = NONE;
      if (valid && cj < k) {
        kx = ip ? -acc : cnorm[cj] - 2.0f * acc;
        id = (uint32_t)cj;
        if (!(kx < INFINITY)) id = NONE;  // NaN or +inf never wins
      }
      uint64_t w = id == NONE ? 0ull : pack_best(kx, id);
#pragma unroll
      for (int o = QR; o < WAVE; o <<= 1) {  // across the centroids of row r
        const uint64_t w2 = __shfl_xor(w, o, WAVE);
        w = w2 > w ? w2 : w;
      }
      if (j == 0 && w != 0) atomicMax(&best[f], (unsigned long long)w);
    }
    // The group's ticket: the item that completes it writes the rows.
    __shared__ int last_s;
    if (lane == 0) {
      __threadfence();
      last_s = atomicAdd(&tickets[g], 1u) == (uint32_t)(per - 1);
    }
    __syncthreads();
    if (last_s) {
      __threadfence();
      if (lane < QR && f < nrows) {
        const unsigned long long w = atomicExch(&best[f], 0ull);
        if (xid_s[r] != NONE) {
          float bk = INFINITY;
          uint32_t bid = 0;  // nothing wins: label 0 and the initial score
          unpack_best(w, bk, bid);
          const size_t p = list ? (size_t)list[f] : lo + (size_t)f;
          labels[p] = bid;
          scores[p] = ip ? -bk : fmaxf(xnq[f] + bk, 0.0f);
          if (tcnt) {  // the tally (few rows: one atomic each)
            atomicAdd(&tcnt[(size_t)bid * tstride + (p - tlo) / TALLY_CP], 1u);
            atomicAdd(&tcounts[bid], 1u);
          }
        }
      }
      if (lane == 0) tickets[g] = 0;
    }
    __syncthreads();
  }
}

// Whether rows of d % 4 == 0 floats at x and c start at multiples of 16 bytes.
bool aligned16(const float* x, const float* c) {
  return (((uintptr_t)x | (uintptr_t)c) & 15) == 0;
}

// ---------------------------------------- exact top-1, at most 64 centroids
// A block takes R = 256 / KP rows against all k <= KP centroids: four waves
// run one chain a lane (row idx / KP, centroid idx % KP), a fifth the rows'
// |x|^2 for L2. Bound by latency (an id, one burst of DMA copies, one chain of
// d fmas and the LDS reads of four such waves), so whole rows come at once
// where 128 KB of LDS hold them, in phases otherwise; LDS slots as in
// k_queued1. A row's candidates meet inside its wave: no atomics on words in
// memory, no tickets, no fences. k_queued1 took 17 us for 1,052 rows x 64
// against 32 centroids (526 items of a wave, their LDS sized for any d: two
// rounds); this takes 8.4. (One chain wave a block instead of four: 8.3 there,
// but 30 us instead of 19 for 1,024 x 768 against 20, where every block takes
// most of a CU's LDS.)
constexpr int S1_W = 4, S1_T = 64 * S1_W + 64, S1_LDS = 128 * 1024;

template <int KP, bool AL>
__global__ __launch_bounds__(S1_T) void k_small1(
    const float* __restrict__ x, size_t nx, int d, const uint32_t* __restrict__ ids, size_t lo,
    int nrows, uint32_t* __restrict__ small, const float* __restrict__ cents,
    const float* __restrict__ cnorm, int k, int ip, int pu, uint32_t* __restrict__ labels,
    float* __restrict__ scores, uint32_t* __restrict__ tcnt, uint32_t* __restrict__ tcounts,
    size_t tlo, size_t tstride) {
  constexpr int R = 64 * S1_W / KP;
  extern __shared__ __attribute__((aligned(16))) v4f lds[];
  __shared__ float xn_s[R];
  v4f* const cs = lds;                          // pu x KP slots (pu: a multiple of 4)
  v4f* const xs = lds + (size_t)pu * KP;        // pu x R slots, up to whole 64s
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int f0 = blockIdx.x * R;
  // This lane's copies: row l % R, centroid l % KP.
  const int fc = f0 + lane % R;
  size_t xc = 0;
  bool okc = false;
  if (fc < nrows) {
    const size_t p = lo + (size_t)fc;
    const size_t id = ids ? (size_t)ids[p] : p;
    okc = id < nx;
    if (okc)
      xc = id;
    else
      small[SW_BAD_ID] = 1;
  }
  const float* const crow = cents + (size_t)min(lane % KP, k - 1) * d;
  const float* const xrow = x + xc * (size_t)d;  // row 0 where there is none
  // This lane's chain: row r, centroid j (the last wave: row r's |x|^2).
  const bool norm = w == S1_W;
  const int idx = w * 64 + lane;
  const int r = norm ? lane % R : idx / KP, j = idx % KP;
  float acc = 0.0f;
  for (int t0 = 0; t0 < d; t0 += 4 * pu) {
    const int nu = min(pu, (d - t0) / 4);  // d % 4 == 0
    for (int i = w; i < (nu * KP + 63) / 64; i += S1_W + 1)
      slot_copy<AL>(crow + min(t0 + 4 * (i * (64 / KP) + lane / KP), d - 4), &cs[i * 64]);
    for (int i = w; i < (nu * R + 63) / 64; i += S1_W + 1)
      slot_copy<AL>(xrow + min(t0 + 4 * (i * (64 / R) + lane / R), d - 4), &xs[i * 64]);
    __syncthreads();  // waits for the copies
    if (!norm) {
#pragma unroll 8
      for (int u = 0; u < nu; u++) {
        const v4f cv = cs[u * KP + j], v = xs[u * R + r];
        acc = fmaf(v.x, cv.x, acc);
        acc = fmaf(v.y, cv.y, acc);
        acc = fmaf(v.z, cv.z, acc);
        acc = fmaf(v.w, cv.w, acc);
      }
    } else if (!ip) {
#pragma unroll 8
      for (int u = 0; u < nu; u++) {
        const v4f v = xs[u * R + r];
        acc = acc + v.x * v.x;
        acc = acc + v.y * v.y;
        acc = acc + v.z * v.z;
        acc = acc + v.w * v.w;
      }
    }
    __syncthreads();  // the next phase's copies overwrite these slots
  }
  if (norm && lane < R) xn_s[lane] = acc;
  __syncthreads();
  const uint64_t okm = __ballot(okc);  // bit r: the block's row r is there
  if (norm) return;
  uint64_t best = 0;
  if (j < k) {
    const float key = ip ? -acc : cnorm[j] - 2.0f * acc;
    if (key < INFINITY) best = pack_best(key, (uint32_t)j);  // NaN or +inf never wins
  }
#pragma unroll
  for (int o = 1; o < KP; o <<= 1) {
    const uint64_t b2 = __shfl_xor(best, o, WAVE);
    best = b2 > best ? b2 : best;
  }
  if (j == 0 && (okm >> r & 1)) {
    float bk = INFINITY;
    uint32_t bid = 0;  // nothing wins: label 0 and the initial score
    unpack_best(best, bk, bid);
    const size_t p = lo + (size_t)(f0 + r);
    labels[p] = bid;
    scores[p] = ip ? -bk : fmaxf(xn_s[r] + bk, 0.0f);
    if (tcnt) {
      atomicAdd(&tcnt[(size_t)bid * tstride + (p - tlo) / TALLY_CP], 1u);
      atomicAdd(&tcounts[bid], 1u);
    }
  }
}

template <int KP>
void small1(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids, size_t lo,
            size_t n, const float* cents, const float* cnorm, size_t k, bool ip, uint32_t* labels,
            float* scores, const LabelTally* tally) {
  constexpr int R = 64 * S1_W / KP;
  // 4-dim slots a phase: all of them where they fit.
  const size_t most = (S1_LDS - 1024) / ((KP + R) * 16) / 4 * 4;
  const size_t pu = std::min<size_t>((d / 4 + 3) / 4 * 4, most);
  const size_t slots = pu * KP + (pu * R + 63) / 64 * 64;
  auto kern = aligned16(x, cents) ? k_small1<KP, true> : k_small1<KP, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)((n + R - 1) / R)), dim3(S1_T), slots * 16, c->stream,
                     x, nx, (int)d, ids, lo, (int)n, c->small, cents, cnorm, (int)k,
                     ip ? 1 : 0, (int)pu, labels, scores, tally ? tally->cnt : nullptr,
                     tally ? tally->counts : nullptr, tally ? tally->lo : 0,
                     tally ? tally->stride : 0);
  EMH_HIP(hipGetLastError());
}

// ------------------------------------------------------------- exact top-k
// Items of KQ queued queries x a range (part) of the data rows, few enough parts
// that the items fill the chip. A tile is KQ queries x KT data rows, a thread 4
// x 4 chains, slabs of KD dimensions in LDS with the next one in registers (bound
// by the fmas, the LDS reads that feed them and the loads' latency). A query keeps
// its kk best in LDS, behind them the rows of the last tiles that beat the kk-th
// of those it had (data rows come in rising order, so an equal score never does);
// when a tile may not fit any more, one wave keeps the kk best of the query's
// entries. With several parts, each leaves its kk best in memory and the last to
// finish picks from those of all parts. 20,000 queued queries of 128 dimensions
// against as many rows: 4.5 ms for the whole call; with slabs of 16 dimensions
// double-buffered 5.9; a workgroup a query, a data row a thread, 170.
constexpr int KQ = 32, KT = 128, KD = 32, KB = 160, KPARTS = 64;
constexpr int KQP = KQ + 4, KTP = KT + 4;

// The kk best (larger score, then lower id; NaN and -inf never came in) of the
// `cnt` <= KB entries at v, id, in any order, to their front; returns how many,
// and in kth the kk-th score (-inf: fewer). One wave: the kk-th key bit by bit by
// ballots (ranks by comparing all with all took five times as long), and among
// equal keys the last id kept the same way.
__device__ __forceinline__ int keep_best(float* v, uint32_t* id, int cnt, int kk, float& kth) {
  constexpr int E = (KB + 63) / 64;
  const int lane = threadIdx.x & 63;
  kth = -INFINITY;
  if (cnt < kk) return cnt;  // (uniform)
  float mv[E];
  uint32_t mi[E], key[E];  // key: ascending image of the score, -0 as +0; 0: no entry
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int i = e * 64 + lane;
    mv[e] = i < cnt ? v[i] : 0.f;
    mi[e] = i < cnt ? id[i] : 0u;
    const uint32_t u = __float_as_uint(mv[e] + 0.0f);
    key[e] = i < cnt ? ((u & 0x80000000u) ? ~u : (u | 0x80000000u)) : 0u;
  }
  uint32_t x = 0u;
  for (int b = 31; b >= 0; b--) {
    const uint32_t t = x | (1u << b);
    int c = 0;
#pragma unroll
    for (int e = 0; e < E; e++) c += __popcll(__ballot(key[e] >= t));
    if (c >= kk) x = t;
  }
  int above = 0, equal = 0;
#pragma unroll
  for (int e = 0; e < E; e++) {
    above += __popcll(__ballot(key[e] > x));
    equal += __popcll(__ballot(key[e] == x));
  }
  uint32_t y = 0xffffffffu;  // the last id kept of the equal ones
  if (above + equal > kk) {
    y = 0u;
    for (int b = 31; b >= 0; b--) {
      const uint32_t t = y | ((1u << b) - 1u);
      int c = 0;
#pragma unroll
      for (int e = 0; e < E; e++) c += __popcll(__ballot(key[e] == x && mi[e] <= t));
      if (above + c < kk) y |= 1u << b;
    }
  }
  __builtin_amdgcn_wave_barrier();  // (the wave's reads come before its writes)
  int at = 0;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const bool keep = key[e] > x || (key[e] == x && mi[e] <= y);
    const unsigned long long m = __ballot(keep);
    if (keep) {
      const int i = at + (int)__builtin_amdgcn_mbcnt_hi(
                             (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      v[i] = mv[e];
      id[i] = mi[e];
    }
    at += __popcll(m);
  }
  __builtin_amdgcn_wave_barrier();
  kth = __uint_as_float((x & 0x80000000u) ? (x & 0x7fffffffu) : ~x);
  return kk;
}

__global__ __launch_bounds__(256) void k_exactk(const float* __restrict__ q, int d,
                                                const float* __restrict__ data, int n, int kk,
                                                int exclude_self, const uint32_t* __restrict__ list,
                                                uint32_t* __restrict__ small,
                                                uint32_t* __restrict__ ids_out,
                                                float* __restrict__ sims_out,
                                                Cand* __restrict__ plist,
                                                uint32_t* __restrict__ tickets) {
  __shared__ __attribute__((aligned(16))) float Qs[KD][KQP];
  __shared__ __attribute__((aligned(16))) float Xs[KD][KTP];
  __shared__ __attribute__((aligned(16))) float bv[KQ][KB];
  __shared__ __attribute__((aligned(16))) uint32_t bi[KQ][KB];
  __shared__ float thr[KQ];  // the kk-th best, -inf while there are fewer
  __shared__ int cnt[KQ];
  __shared__ uint32_t qid[KQ];
  __shared__ int last;
  const int nrows = (int)small[SW_FALLBACK_COUNT];
  if (blockIdx.x == 0 && threadIdx.x == 0) small[SW_FALLBACK_TOTAL] += (uint32_t)nrows;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int tx = tid & 31, ty = tid >> 5;
  const int nqt = (nrows + KQ - 1) / KQ, ntile = (n + KT - 1) / KT;
  if (nqt == 0) return;
  const int want = max(1, min(min(ntile, KPARTS), ((int)gridDim.x + nqt - 1) / nqt));
  const int tpp = (ntile + want - 1) / want, parts = ntile > 0 ? (ntile + tpp - 1) / tpp : 1;
  for (int item = blockIdx.x; item < nqt * parts; item += gridDim.x) {
    const int qt = item / parts, part = item - qt * parts;
    const int rows = min(KQ, nrows - qt * KQ);
    __syncthreads();  // the previous item is done with LDS
    if (tid < KQ) {
      qid[tid] = list[qt * KQ + min(tid, rows - 1)];
      thr[tid] = -INFINITY;
      cnt[tid] = 0;
    }
    __syncthreads();
    // Loader: a thread takes dimensions 4 (tid % 8) .. + 3 of query tid / 8 and
    // of the data rows tid / 8 + 32 u (a slab is a whole line of a row).
    const int pr = tid >> 3, pt = 4 * (tid & 7);
    const float* const qrow = q + (size_t)qid[pr] * d;
    float qv[4], xv[4][4];
    auto load = [&](int j0, int t0) __attribute__((always_inline)) {
      const int t = t0 + pt;
#pragma unroll
      for (int c = 0; c < 4; c++) qv[c] = t + c < d ? qrow[t + c] : 0.f;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float* p = data + (size_t)min(j0 + 32 * u + pr, n - 1) * d;
#pragma unroll
        for (int c = 0; c < 4; c++) xv[u][c] = t + c < d ? p[t + c] : 0.f;
      }
    };
    auto store = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        Qs[pt + c][pr] = qv[c];
#pragma unroll
        for (int u = 0; u < 4; u++) Xs[pt + c][32 * u + pr] = xv[u][c];
      }
    };
    const int c0 = part * tpp, c1 = min(ntile, c0 + tpp);
    for (int ct = c0; ct < c1; ct++) {
      const int j0 = ct * KT;
      float acc[4][4];
#pragma unroll
      for (int a = 0; a < 4; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[a][e] = 0.f;
      auto dim = [&](int t) __attribute__((always_inline)) {
        float qa[4], xa[4];
#pragma unroll
        for (int a = 0; a < 4; a++) qa[a] = Qs[t][ty * 4 + a];
#pragma unroll
        for (int e = 0; e < 4; e++) xa[e] = Xs[t][tx * 4 + e];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[a][e] = fmaf(qa[a], xa[e], acc[a][e]);
      };
      if (ct == c0) load(j0, 0);
      for (int t0 = 0; t0 < d; t0 += KD) {
        store();
        __syncthreads();
        // The next slab (of the next tile, after the last) is on its way meanwhile.
        if (t0 + KD < d)
          load(j0, t0 + KD);
        else if (ct + 1 < c1)
          load(j0 + KT, 0);
        const int tn = min(KD, d - t0);  // dimensions past d never enter a chain
        if (tn == KD) {
#pragma unroll
          for (int t = 0; t < KD; t++) dim(t);
        } else {
          for (int t = 0; t < tn; t++) dim(t);
        }
        __syncthreads();
      }
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const int r = ty * 4 + a;
        const float lim = thr[r];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int j = j0 + tx * 4 + e;
          if (acc[a][e] > lim && j < n && !(exclude_self && (uint32_t)j == qid[r])) {
            const int at = atomicAdd(&cnt[r], 1);  // (at most KT a tile: there is room)
            bv[r][at] = acc[a][e];
            bi[r][at] = (uint32_t)j;
          }
        }
      }
      __syncthreads();
      for (int r = w; r < KQ; r += 4) {
        const int m = cnt[r];
        if (m <= KB - KT) continue;
        float kth;
        const int got = keep_best(bv[r], bi[r], m, kk, kth);
        if (lane == 0) {
          cnt[r] = got;
          thr[r] = kth;
        }
      }
      __syncthreads();
    }
    for (int r = w; r < KQ; r += 4) {
      float kth;
      const int got = keep_best(bv[r], bi[r], cnt[r], kk, kth);
      if (lane == 0) cnt[r] = got;
    }
    __syncthreads();
    if (parts > 1) {
      // (Agent-scope words: the ranking workgroup may be on another XCD.)
      unsigned long long* out = (unsigned long long*)plist + ((size_t)qt * parts + part) * KQ * kk;
      for (int i = tid; i < KQ * kk; i += 256) {
        const int r = i / kk, e = i - r * kk;
        const bool have = e < cnt[r];
        const unsigned long long word =
            ((unsigned long long)(have ? bi[r][e] : NONE) << 32) |
            __float_as_uint(have ? bv[r][e] : -INFINITY);
        __hip_atomic_store(&out[i], word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __threadfence();
      __syncthreads();
      if (tid == 0) last = atomicAdd(&tickets[qt], 1u) == (uint32_t)(parts - 1);
      __syncthreads();
      if (!last) continue;
      __threadfence();
      const unsigned long long* in = (const unsigned long long*)plist + (size_t)qt * parts * KQ * kk;
      for (int r = w; r < rows; r += 4) {
        int have = 0;
        for (int p0 = 0; p0 < parts; p0 += KT / KMAX) {  // eight parts' at a time
          const int np = min(KT / KMAX, parts - p0) * kk;
          int m = have;
          for (int i0 = 0; i0 < np; i0 += 64) {
            const int i = i0 + lane, p = i / kk, e = i - p * kk;
            unsigned long long word = (unsigned long long)NONE << 32;
            if (i < np)
              word = __hip_atomic_load(&in[((size_t)(p0 + p) * KQ + r) * kk + e], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            const bool ok = (uint32_t)(word >> 32) != NONE;
            const unsigned long long mask = __ballot(ok);
            if (ok) {
              const int at = m + (int)__builtin_amdgcn_mbcnt_hi(
                                     (uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
              bv[r][at] = __uint_as_float((uint32_t)word);
              bi[r][at] = (uint32_t)(word >> 32);
            }
            m += __popcll(mask);
          }
          __builtin_amdgcn_wave_barrier();
          float kth;
          have = keep_best(bv[r], bi[r], m, kk, kth);
        }
        if (lane == 0) cnt[r] = have;
      }
      if (tid == 0) tickets[qt] = 0;
      __syncthreads();
    }
    // Output order: IEEE total order descending (+0 before -0), then id.
    for (int r = w; r < rows; r += 4) {
      const int have = cnt[r];
      if (lane < kk) {
        const size_t o = (size_t)qid[r] * kk;
        if (lane < have) {
          auto ord = [](float f) {
            const uint32_t u = __float_as_uint(f);
            return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
          };
          const uint32_t mine = ord(bv[r][lane]), id = bi[r][lane];
          int at = 0;
          for (int e = 0; e < have; e++) {
            const uint32_t v = ord(bv[r][e]);
            at += v > mine || (v == mine && bi[r][e] < id) ? 1 : 0;
          }
          ids_out[o + at] = id;
          sims_out[o + at] = bv[r][lane];
        } else {
          ids_out[o + lane] = NONE;
          sims_out[o + lane] = -INFINITY;
        }
      }
    }
  }
}

}  // namespace

// The latency-bound scan's items for n rows against k centroids.
size_t queued_items(size_t n, size_t k, bool ip) {
  return ((n + QR - 1) / QR) * ((k + QJ - 1) / QJ + (ip ? 0 : 1));
}

size_t exact1_scratch_bytes(emh_ctx* c, size_t n, size_t d, size_t k, bool ip, bool list) {
  auto r = [](size_t b) { return (b + 255) & ~size_t(255); };
  if (!list && small_direct(c, n, d, k)) return 0;
  if ((list && d % 4 == 0) || (!list && queued_direct(c, n, d, k, ip))) {
    const size_t ngr = (n + QR - 1) / QR;
    return r(n * 8 + ngr * 4) + r(n * 4);
  }
  const size_t nch = (k + CJ - 1) / CJ, ngr = (n + RG - 1) / RG;
  return r(n * nch * sizeof(Cand)) + r(ngr * 4);
}

void launch_exact1(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids,
                   size_t lo, size_t n, const uint32_t* list, const float* cents,
                   const float* cnorm, size_t k, bool ip, uint32_t* labels, float* scores,
                   Arena* ar, const LabelTally* tally) {
  if (n == 0) return;
  EMH_ENSURE(!tally || (d % 4 == 0 && (list || queued_direct(c, n, d, k, ip))),
             "exact: a tally needs the queued-row scan");
  if (!list && small_direct(c, n, d, k)) {
    auto f = k <= 16 ? small1<16> : k <= 32 ? small1<32> : small1<64>;
    f(c, x, nx, d, ids, lo, n, cents, cnorm, k, ip, labels, scores, tally);
    return;
  }
  // Queued rows (few), or a small direct selection: the latency-bound scan.
  // (k_exact1's tiles each wait a memory round trip: ~30 us at any size up
  // to a few thousand rows.)
  if ((list && d % 4 == 0) || (!list && queued_direct(c, n, d, k, ip))) {
    const size_t ngr = (n + QR - 1) / QR;
    const size_t per = (k + QJ - 1) / QJ + (ip ? 0 : 1);
    // Self-cleaning: the best words, then the tickets, all left at zero (a
    // fixed block is cleared on every call instead).
    char* z;
    float* xnq;
    if (ar) {
      z = (char*)ar->take(n * 8 + ngr * 4);
      launch_fill_u32(c, (uint32_t*)z, n * 2 + ngr, 0);
      xnq = (float*)ar->take(n * 4);
    } else {
      z = (char*)c->tickets.get_zeroed(n * 8 + ngr * 4, c->stream);
      xnq = (float*)c->knn_tmp.get(n * 4);
    }
    const unsigned g = (unsigned)std::min<size_t>(ngr * per, (size_t)2 * c->cus);
    auto kern = aligned16(x, cents) ? k_queued1<true> : k_queued1<false>;
    hipLaunchKernelGGL(kern, dim3(g), dim3(256), 0, c->stream, x, nx, (int)d, ids, lo,
                       (int)n, list, c->small, cents, cnorm, (int)k, ip ? 1 : 0,
                       (unsigned long long*)z,
                       (uint32_t*)(z + n * 8), xnq, labels, scores,
                       tally ? tally->cnt : nullptr, tally ? tally->counts : nullptr,
                       tally ? tally->lo : 0, tally ? tally->stride : 0);
    EMH_HIP(hipGetLastError());
    return;
  }
  const size_t nch = (k + CJ - 1) / CJ;
  const size_t ngr = (n + RG - 1) / RG;
  Cand* partial;
  uint32_t* tickets;
  unsigned long long* best = nullptr;  // tiles: left at zero, as the tickets
  if (ar) {
    partial = (Cand*)ar->take(n * nch * sizeof(Cand));
    tickets = (uint32_t*)ar->take(ngr * 4);
    launch_fill_u32(c, tickets, ngr, 0);
  } else {
    partial = (Cand*)c->knn_tmp.get(n * nch * sizeof(Cand));
    best = (unsigned long long*)c->tickets.get_zeroed((list ? n * 8 : 0) + ngr * 4, c->stream);
    tickets = (uint32_t*)(best + (list ? n : 0));
  }
  // Queued rows: the count lives on the device, so the grid covers the worst
  // case. Queued rows are few: a grid of 2 blocks per CU covers them, and
  // blocks past the device-side count exit at once.
  const size_t items = ngr * nch;
  const unsigned g = (unsigned)std::min<size_t>(items, (size_t)(list ? 2 : 8) * c->cus);
  if (list) {  // (d % 4 != 0; the tiles' |x|^2 where the items' winners would be)
    hipLaunchKernelGGL(k_exact1_list, dim3(g), dim3(256), 0, c->stream, x, nx, (int)d, ids, lo,
                       list, c->small, cents, cnorm, (int)k, ip ? 1 : 0, partial, tickets, best,
                       (float*)partial, labels, scores);
  } else {
    auto kern = d % 4 == 0 ? k_exact1<true> : k_exact1<false>;
    hipLaunchKernelGGL(kern, dim3(g), dim3(64), 0, c->stream, x, nx, (int)d, ids, lo, (int)n,
                       c->small, cents, cnorm, (int)k, ip ? 1 : 0, partial, tickets, labels,
                       scores);
  }
  EMH_HIP(hipGetLastError());
}

void launch_exactk(emh_ctx* c, const float* q, size_t m, const float* data, size_t n, size_t d,
                   size_t kk, bool exclude_self, const uint32_t* fb, uint32_t* ids, float* sims) {
  if (m == 0) return;
  EMH_ENSURE(kk >= 1 && kk <= (size_t)KMAX, "exact: kk = %zu must be in 1..%d", kk, KMAX);
  const size_t g = 2 * (size_t)std::max(c->cus, 1);
  // Several parts only while the queries' tiles are fewer than the workgroups.
  const size_t lists = std::min(2 * g, (m + KQ - 1) / KQ * (size_t)KPARTS) * KQ * kk;
  Cand* plist = (Cand*)c->knn_tmp.get(lists * sizeof(Cand));
  uint32_t* tickets = (uint32_t*)c->tickets.get_zeroed((m + KQ - 1) / KQ * 4, c->stream);
  hipLaunchKernelGGL(k_exactk, dim3((unsigned)g), dim3(256), 0, c->stream, q, (int)d, data, (int)n,
                     (int)kk, exclude_self ? 1 : 0, fb, c->small, ids, sims, plist, tickets);
  EMH_HIP(hipGetLastError());
}

}  // namespace emh
