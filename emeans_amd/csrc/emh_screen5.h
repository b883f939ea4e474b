// The one-pass large-tile screen (k_screen5) over fp16 lines (emh_lines.h),
// for top-1 and top-k.
//
// The screen only has to name every row's possible winners; the check's exact
// chains decide. One fp16 MFMA per 16 dimensions (where the bf16 three-pass
// screens issue three) leaves an error bound, in units of |x||c - m|
// (emh_lines.h; theirs in |x||c|), of 1.6 times theirs at d = 1,024, 2.9 at 384,
// 6 at 64 and 10 at 32, because it rests on each row's measured rounding residual
// instead of the worst case, and the operands take half the bytes from HBM to
// LDS. Rows that the longer lists cannot settle all the same go to exact scans
// that take long queues in tiles (emh_verify.hip).
//
// Tile: 256 rows x 256 centroids (kNN: queries x data rows), 8 waves; wave w
// owns rows 64 (w % 4) .. + 64 and centroids 128 (w / 4) .. + 128, as 2 x 4
// blocks of 32 x 32 (the centroids as the MFMA's A, the rows as its B: a lane
// holds one row of each block, 16 columns in registers). Slabs of 32
// dimensions (two MFMA steps) stream into a four-stage LDS ring (32 KB a
// stage) by LDS DMA, with up to three slabs in flight: one pass of MFMAs
// leaves a slab a third of the time that the three-pass screens do, less than
// the latency of its loads.
#pragma once

#include <type_traits>

#include "emh_dma.h"
#include "emh_lines.h"
#include "emh_screen_kern.h"

namespace emh {
namespace {

constexpr int T5 = 256;                       // rows, and centroids, per tile
constexpr int S5_HALF = T5 * LINE_BYTES;      // one operand's slab: 16 KB
constexpr int S5_STAGE = 2 * S5_HALF;         // both: 32 KB
constexpr int NS5 = 4;                        // stages of the ring
constexpr int NN5 = 5;                        // tiles its steps and the present one may span

// A line's four 16-byte chunks (chunk c: dimensions 8 c .. 8 c + 7) are
// XOR-swizzled in LDS by swz5(row): a b128 operand read has lane l read row
// 32 y + l % 32 at chunk 2 kk + l / 32. Four rows fill the 64 banks; among 16
// consecutive rows the four with the same r % 4 have four different swizzles,
// and rows 4 apart differ in bit 1 while l / 32 flips bit 0, so sixteen
// consecutive lanes, and eight with their partners of the other half, hit
// sixteen different 16-byte groups.
__device__ __forceinline__ int swz5(int r) { return (((r >> 2) & 1) << 1) | ((r >> 3) & 1); }

// LDS by address (the ring's stage is a run-time value).
typedef const v8h __attribute__((address_space(3)))* lds8h;

// Maxima of part[4 i .. 4 i + 3] over i < nparts (f32 bits as u32: a NaN or
// negative value wins), in every lane of the wave; each lane's loads of a
// batch are issued together.
__device__ __forceinline__ void part_max4(const uint32_t* __restrict__ part, int nparts,
                                          uint32_t& ma, uint32_t& mb, uint32_t& mc, uint32_t& md) {
  constexpr int B = 8;
  const int lane = threadIdx.x & 63;
  ma = mb = mc = md = 0u;
  for (int i0 = 0; i0 < nparts; i0 += 64 * B) {
    uint4 v[B];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const int i = i0 + 64 * u + lane;
      v[u] = i < nparts ? reinterpret_cast<const uint4*>(part)[i] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < B; u++) {
      ma = max(ma, v[u].x);
      mb = max(mb, v[u].y);
      mc = max(mc, v[u].z);
      md = max(md, v[u].w);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    ma = max(ma, (uint32_t)__shfl_xor((int)ma, o, 64));
    mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
    mc = max(mc, (uint32_t)__shfl_xor((int)mc, o, 64));
    md = max(md, (uint32_t)__shfl_xor((int)md, o, 64));
  }
}

enum Kind5 : int {
  TOP1_IP = 0,   // top-1: key -dot
  TOP1_L2 = 1,   // top-1: key |c|^2 - 2 dot
  KNN = 2,       // top-k, key -dot
  KNN_SELF = 3,  // ... of the rows themselves, each row's own column left out
  SCORES = 4,    // no lists: every dot to memory (emh_topk_long.hip)
};
constexpr int KTH5 = KMAX;  // kNN: the smallest keys a thread keeps for its row's limit
constexpr int CAP5 = 12;    // slots of a row's append buffer (each of its two centroid waves)
constexpr int LOG5_TOP1 = 32, LOG5_KNN = 256;  // entries of a thread's log

struct Args5 {
  const char* xs;         // the rows' lines (slab stride xslab), row id of nx
  size_t xslab;
  const float2* xn;       // |x|^2 and the residual of every row
  size_t nx;
  const uint32_t* ids;    // position -> row id (or null: the position)
  size_t lo;
  int nrows;
  const char* cs;         // the centroids' lines (slab stride cslab)
  size_t cslab;
  const float* cnorm;     // L2: the centroids' given squared norms
  int k, d, kk;
  int L;                  // kNN: entries of a list, at most LK5 (top-1: L5)
  int tpp, parts, ntiles;
  Cand* cand;             // out: [row][part][L], see the end of k_screen5
  uint32_t* ncand;        // top-1: their lengths
  Cand* log;              // blocks x 512 x LOG5_* entries of scratch (parts of several tiles)
  float* bound;           // out: E of row r at r, its dot term at bstride + r
  size_t bstride;
  const uint32_t* part;   // the centroids' maxima (CentsOut)
  int nparts;
  const float* sx;        // scales: s, 1 / s
  const float* sc;
  const float* same;      // kNN: with *same == 0, the rows' lines, norms and scale are
  const float2* cn;       // the data's (norms cn)
  float* scores;          // SCORES: out, row r's dots at r ldS (a multiple of 4, >= k)
  size_t ldS;
};

// ONE: parts of one tile (its lists never leave LDS).
template <int KIND, bool ONE>
__global__ __launch_bounds__(512, 1) void k_screen5(const Args5 a_) {
  constexpr bool L2 = KIND == TOP1_L2, SELF = KIND == KNN_SELF;
  constexpr bool TOPK = KIND == KNN || KIND == KNN_SELF;
  constexpr bool LISTS = KIND != SCORES, TOP1 = LISTS && !TOPK;
  constexpr int NK = TOPK ? KTH5 : 1, CAP = CAP5;
  constexpr int LOG = TOPK ? LOG5_KNN : LOG5_TOP1;
  constexpr int WA = 4, WN = 2;  // centroid (A) and row (B) 32-blocks per wave
  constexpr int ND = 2;          // DMAs per operand per step per wave
  constexpr int PER = 2 * ND + (L2 ? 1 : 0);  // DMAs per step per wave
  __shared__ __attribute__((aligned(1024))) char ring[NS5 * S5_STAGE];
  __shared__ __attribute__((aligned(16))) float Ns[L2 ? NN5 : 1][L2 ? T5 : 4];  // tile norms, by tile % NN5
  // Append buffers: slot e of wave w's row r (0 .. 63) at (w CAP + e) 64 + r.
  __shared__ uint32_t buf[LISTS ? 8 * CAP * 64 : 1];
  // What the two centroid waves of a row publish for each other's limits
  // (see set_limit): a read that races a write takes either value, both valid.
  __shared__ float pub[2][TOPK ? 2 : 1][T5];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wr = w & 3, wc = w >> 2;
  const int li = lane & 31, h = lane >> 5;
  const int parts = a_.parts, k = a_.k, nrows = a_.nrows;
  const uint32_t wi = xcd_swizzle(blockIdx.x, gridDim.x);
  const int rt = (int)(wi / (uint32_t)parts), part = (int)(wi % (uint32_t)parts);
  const int t0 = part * a_.tpp;
  const int t1 = min(a_.ntiles, t0 + a_.tpp);
  if (t0 >= t1) return;
  const int row0 = rt * T5;
  const int d32 = (a_.d + LINE_DIMS - 1) / LINE_DIMS;

  // Loader: DMA j of wave w fills LDS rows 128 j + 16 w + lane / 4 of an
  // operand; a lane's 16 bytes land in slot lane % 4 of its row, which holds
  // chunk (lane % 4) ^ swz5(row). Rows past the selection (or with a bad id)
  // read data row 0, centroids past k whatever follows (the next slab's first
  // rows, or the padding that lines_bytes counts): neither is ever listed.
  const int lrow = w * 16 + (lane >> 2);
  const int lq = ((lane & 3) ^ swz5(lrow)) << 4;
  const uint32_t co = (uint32_t)(lrow * LINE_BYTES + lq);
  uint32_t xo[ND];  // byte offsets in a slab (fewer than 2^25 rows)
#pragma unroll
  for (int j = 0; j < ND; j++) {
    const int r = row0 + j * 128 + lrow;
    uint32_t id = 0;
    if (r < nrows) {
      const size_t p = a_.lo + (size_t)r;
      const size_t v = a_.ids ? (size_t)a_.ids[p] : p;
      id = v < a_.nx ? (uint32_t)v : 0u;
    }
    xo[j] = id * LINE_BYTES + lq;
  }
  // Load cursor (tile lt, slab lj, into stage ls): every step issues the DMAs
  // of the step NS5 later; past the last step they fetch the last tile again
  // into a stage nothing reads.
  int lt = t0, lj = 0;
  const int nsteps = (t1 - t0) * d32;
  const bool own = TOP1 || !a_.same || *a_.same != 0.f;
  const char* const xs0 = own ? a_.xs : a_.cs;
  const float2* const xn0 = own ? a_.xn : a_.cn;
  const float* const sx = own ? a_.sx : a_.sc;
  const uint32_t ring0 = lds_addr(ring);
  const uint32_t ldst = ring0 + (uint32_t)__builtin_amdgcn_readfirstlane(w) * 16 * LINE_BYTES;
  uint32_t ls = 0;                              // the load stage's offset in the ring
  const char *xp = xs0, *cp = a_.cs + (size_t)t0 * T5 * LINE_BYTES;  // slab lj of the rows, the tile
  auto dma_part = [&](int q) __attribute__((always_inline)) {
    const int j = q % ND;
    const uint32_t dst = ldst + ls + (q / ND) * S5_HALF + j * 128 * LINE_BYTES;
    if (q < ND) {
      dma16a(xp, xo[j], dst);
    } else {
      dma16a(cp + j * 128 * LINE_BYTES, co, dst);
      const int tl = min(lt, t1 - 1);
      if (L2 && q == 2 * ND - 1)  // 64 norms per wave (waves w and w + 4 alike)
        dma4(a_.cnorm + min(tl * T5 + wr * 64 + lane, k - 1), &Ns[L2 ? tl % NN5 : 0][L2 ? wr * 64 : 0]);
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    const bool wrap = ++lj == d32;
    lj = wrap ? 0 : lj;
    lt += wrap ? 1 : 0;
    xp = wrap ? xs0 : xp + a_.xslab;
    cp = wrap ? a_.cs + (size_t)min(lt, t1 - 1) * T5 * LINE_BYTES : cp + a_.cslab;
    ls = (ls + S5_STAGE) % (NS5 * S5_STAGE);
  };

  // Operand reads of MFMA step ks of the slab in stage st: every operand row
  // is li modulo 32, so the chunk's offset within its line is the same for
  // all, and MFMA step 1's is step 0's with bit 5 flipped.
  const uint32_t at0 = ring0 + (uint32_t)li * LINE_BYTES + (uint32_t)((h ^ swz5(li)) << 4);
  const uint32_t rat = at0 + wr * 64 * LINE_BYTES, cat = at0 + S5_HALF + wc * 128 * LINE_BYTES;
  struct Rows {
    v8h b[WN];
  };
  auto read_rows = [&](int st, int ks, Rows& o) __attribute__((always_inline)) {
    const uint32_t at = (rat + st * S5_STAGE) ^ (ks << 5);
#pragma unroll
    for (int y = 0; y < WN; y++) o.b[y] = *(lds8h)(uintptr_t)(at + y * 32 * LINE_BYTES);
  };
  v8h ca[WA];
  auto read_cent = [&](int st, int ks, int a) __attribute__((always_inline)) {
    const uint32_t at = (cat + st * S5_STAGE) ^ (ks << 5);
    ca[a] = *(lds8h)(uintptr_t)(at + a * 32 * LINE_BYTES);
  };

  // The bound E of the lane's rows (block y's row li): the check reads it
  // from bound[], and the fold keeps what lies within 2E' (E' >= E, with a
  // margin for the rounding of the sums that use it).
  float thr_q;  // 2E' of the row this lane keeps (block h's)
  const float f1 = sx[1] * a_.sc[1];  // accumulator -> dot, a power of two
  const float rf1 = sx[0] * a_.sc[0];  // its inverse
  {
    uint32_t ma, mb, mc, md;
    part_max4(a_.part, a_.nparts, ma, mb, mc, md);
    const int r = row0 + (tid & (T5 - 1));
    float2 xv = make_float2(0.f, 0.f);
    if (r < nrows) {
      const size_t p = a_.lo + (size_t)r;
      const size_t id = a_.ids ? (size_t)a_.ids[p] : p;
      xv = xn0[id < a_.nx ? id : 0];
    }
    float edot;
    const float E = screen_bound_lines(xv.x, xv.y, __uint_as_float(md), __uint_as_float(ma),
                                       __uint_as_float(mc), L2 ? __uint_as_float(mb) : 0.f,
                                       sx[1], a_.sc[1], a_.d, L2, &edot);
    thr_q = 2.0f * 1.0078125f * E;
    if (part == 0 && wc == 0 && r < nrows) {
      a_.bound[r] = E;
      a_.bound[a_.bstride + r] = edot;
    }
  }

  v16f acc[WA][WN];

  // ---- Candidates. The lane of half h keeps its wave's row 32 h + li: the
  // NK smallest keys of the wave's columns so far, in registers, and a log in
  // memory of every (key, id) that was within the row's limit when it came.
  //
  // Limit. The check settles a row when its candidates hold every key within
  // the row's kk-th smallest key plus 2E (top-1: kk = 1). That key is at most
  // this thread's kk-th, at most the other centroid wave's, at most the larger
  // of the two threads' ceil(kk / 2)-th keys (together they hold kk keys that
  // small), and at most the kk-th of any columns seen; all of these only
  // fall. So what the check needs was within the limit when it came. A log
  // that fills is swept of what has fallen out of the limit; when even that
  // does not make room (hundreds of near-ties) the row goes to the exact scan,
  // as it does with a NaN bound, under which nothing is kept.
  const int kk = TOPK ? a_.kk : 1, kh = (kk + 1) / 2;
  const int prow = tid & (T5 - 1);  // 64 wr + 32 h + li: the thread's row
  const bool live = thr_q == thr_q;
  float lkey[NK];
#pragma unroll
  for (int e = 0; e < NK; e++) lkey[e] = INFINITY;
  float kth = INFINITY, kha = INFINITY;  // this thread's kk-th and kh-th keys
  // Entry i of the thread's log (the block's base is uniform).
  Cand* const blog = a_.log + (size_t)blockIdx.x * 512 * LOG;
  auto mylog = [&](uint32_t i) __attribute__((always_inline))->Cand& { return blog[tid * LOG + i]; };
  uint32_t nlog = 0;
  bool spilt = false;  // the log (ONE: the buffer) did not hold everything
  // The largest key that may still matter, with room for the tags' 2^-16 on
  // both sides.
  auto limit_of = [&](float b) __attribute__((always_inline)) {
    return b + thr_q + fabsf(b) * 3.0517578125e-05f + 1e-42f;
  };
  // Gains: the accumulators hold dots in units of 1 / f1 (IP, kNN: key =
  // -f1 gain), or, once the fold has rewritten them, 2 dot - |c|^2 (L2: key =
  // -gain). gl: the least gains within the limits of the lane's two rows (its
  // own, and the partner lane's), or a hair less (f1 is a power of two; 2^-22
  // covers the product's rounding where it is subnormal).
  float gl[WN];
  auto set_limit = [&](float b) __attribute__((always_inline)) {
    const float lim = limit_of(b);
    float g = L2 ? -lim : -lim * rf1;
    if (!L2) g = g - fabsf(g) * 2.384185791015625e-07f - 1e-44f;
    // (Padding's -inf is never within it; a row that has spilt appends no more.)
    g = live && !spilt ? fmaxf(g, -3.4028235e38f) : __builtin_nanf("");
    const float gp = __shfl_xor(g, 32, 64);
    gl[0] = h == 0 ? g : gp;
    gl[1] = h == 1 ? g : gp;
  };
  auto published = [&]() __attribute__((always_inline)) {  // with the other wave's keys
    const float pk = __hip_atomic_load(&pub[wc ^ 1][0][prow], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
    if (!TOPK) return fminf(kth, pk);
    const float pa = __hip_atomic_load(&pub[wc ^ 1][TOPK ? 1 : 0][prow], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
    return fminf(fminf(kth, pk), fmaxf(kha, pa));
  };
  auto publish = [&]() __attribute__((always_inline)) {
    __hip_atomic_store(&pub[wc][0][prow], kth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (TOPK)
      __hip_atomic_store(&pub[wc][TOPK ? 1 : 0][prow], kha, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  uint32_t cnt[WN] = {0u, 0u};  // entries in the rows' append buffers (both lane halves agree)
  uint32_t* mybuf = buf + w * (CAP * 64);
  // Column 32 a + 8 (r / 4) + 4 half + r % 4 of the tag 64 half + 16 a + r.
  auto column = [](uint32_t v) __attribute__((always_inline)) {
    return ((v & 48u) << 1) + ((v & 12u) << 1) + ((v & 64u) >> 4) + (v & 3u);
  };
  // The buffered entries into the keys and the log.
  auto flush = [&](uint32_t base) __attribute__((always_inline)) {
    const uint32_t n = h ? cnt[1] : cnt[0];
    for (uint32_t i = 0; __ballot(i < n) != 0ull; i++) {
      const uint32_t v = mybuf[i * 64 + lane];
      const float key = i < n ? __uint_as_float(v) : INFINITY;
      insert_key<NK>(lkey, key);
      if (i < n) mylog(nlog++) = Cand{key, base + column(v)};
    }
    cnt[0] = cnt[1] = 0u;
    // The kk-th and kh-th keys are the largest of the first entries (a max
    // over masked entries, which needs no indexed read; the masks' bounds are
    // opaque, or they are all kept in registers through the loop).
    int nk = kk, nh = kh;
    asm volatile("" : "+s"(nk), "+s"(nh));
    kth = kha = lkey[0];
#pragma unroll
    for (int e = 1; e < NK; e++) {
      kth = fmaxf(kth, e < nk ? lkey[e] : -INFINITY);
      kha = fmaxf(kha, e < nh ? lkey[e] : -INFINITY);
    }
    if (__ballot(nlog > (uint32_t)(LOG - CAP)) != 0ull) {
      const float lim = limit_of(published());
      uint32_t m = 0;
      for (uint32_t i = 0; i < nlog; i++) {
        const Cand v = mylog(i);
        if (v.key <= lim) mylog(m++) = v;
      }
      if (m > (uint32_t)(LOG - 2 * CAP)) {
        spilt = true;
        m = LOG - 2 * CAP;
      }
      nlog = m;
    }
  };
  // A tile's accumulators into the lists. Per 32 x 32 block the largest gain
  // first; then, of the blocks where some lane's passes, the elements, each
  // lane appending those that pass, tagged with their column in the low 7 bits
  // (E allows for it), to its row's buffer in LDS, from which the row's thread
  // takes them: all rows of a wave insert at once, where an insert per element
  // would serve one.
  auto fold = [&](int tile) __attribute__((always_inline)) {
    const uint32_t base = (uint32_t)(tile * T5 + wc * 128);
    if (L2) {
      const float* ns = Ns[L2 ? tile % NN5 : 0];
#pragma unroll
      for (int a = 0; a < WA; a++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float4 n4 = *reinterpret_cast<const float4*>(ns + wc * 128 + a * 32 + 8 * q + 4 * h);
          const float nv[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int y = 0; y < WN; y++)
              acc[a][y][4 * q + e] = fmaf(2.0f * f1, acc[a][y][4 * q + e], -nv[e]);  // one rounding
        }
    }
    if ((tile + 1) * T5 > k) {  // the last tile: columns past k
      int left = k - (int)base - 4 * h;
      asm volatile("" : "+v"(left));  // (recomputed here, not kept through the loop)
#pragma unroll
      for (int a = 0; a < WA; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const bool in = a * 32 + 8 * (r >> 2) + (r & 3) < left;
#pragma unroll
          for (int y = 0; y < WN; y++) acc[a][y][r] = in ? acc[a][y][r] : -INFINITY;
        }
    }
    if (SELF && (size_t)tile * T5 == a_.lo + (size_t)row0) {  // the rows' own columns
      int own = wr * 64 + li - wc * 128 - 4 * h;
      asm volatile("" : "+v"(own));
#pragma unroll
      for (int a = 0; a < WA; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
#pragma unroll
          for (int y = 0; y < WN; y++)
            acc[a][y][r] = a * 32 + 8 * (r >> 2) + (r & 3) - y * 32 == own ? -INFINITY : acc[a][y][r];
        }
    }
    float mx[WA][WN];  // block maxima (fmaxf passes over NaN)
#pragma unroll
    for (int a = 0; a < WA; a++)
#pragma unroll
      for (int y = 0; y < WN; y++) {
        mx[a][y] = acc[a][y][0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx[a][y] = fmaxf(mx[a][y], acc[a][y][r]);
      }
    float b = published();
    if (!TOPK) {  // the wave's best key of this tile (both halves' columns)
      float t[WN];
#pragma unroll
      for (int y = 0; y < WN; y++) t[y] = fmaxf(fmaxf(mx[0][y], mx[1][y]), fmaxf(mx[2][y], mx[3][y]));
      const float own = h ? t[1] : t[0], give = h ? t[0] : t[1];
      const float best = fmaxf(own, __shfl_xor(give, 32, 64));
      const float key = L2 ? -best : -f1 * best;
      if (ONE) kth = key;
      b = fminf(b, key);
    } else if (tile == t0) {
      // The first tile: of each half's eight maxima over 8 elements, the kh-th
      // largest; the smaller of the two halves' has kk columns above it.
      int nh = kh;
      asm volatile("" : "+s"(nh));
      float t[WN];
#pragma unroll
      for (int y = 0; y < WN; y++) {
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] = INFINITY;
#pragma unroll
        for (int a = 0; a < WA; a++)
#pragma unroll
          for (int q = 0; q < 2; q++) {
            float m8 = acc[a][y][8 * q];
#pragma unroll
            for (int r = 1; r < 8; r++) m8 = fmaxf(m8, acc[a][y][8 * q + r]);
            insert_key<8>(s, -m8);
          }
        float v = s[0];
#pragma unroll
        for (int e = 1; e < 8; e++) v = fmaxf(v, e < nh ? s[e] : -INFINITY);
        t[y] = v;  // minus the kh-th largest
      }
      const float own = h ? t[1] : t[0], give = h ? t[0] : t[1];
      b = fminf(b, f1 * fmaxf(own, __shfl_xor(give, 32, 64)));
    }
    set_limit(b);
    // Pass 0 takes the whole tile. When a row's buffer overflowed, passes 1 ..
    // 16 start over with a quarter of a block each (8 columns of a row at most)
    // and the limits that the passes before left.
    for (int pass = 0;;) {
      bool over = false, any = false;
#pragma unroll
      for (int a = 0; a < WA; a++)
#pragma unroll
        for (int y = 0; y < WN; y++) {
          if (__ballot(mx[a][y] >= gl[y]) == 0ull) continue;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            if (!ONE && pass != 0 && pass != 4 * a + q + 1) continue;
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const int r = 4 * q + e;
              const unsigned long long m = __ballot(acc[a][y][r] >= gl[y]);
              if (m == 0ull) continue;
              any = true;
              // (Opaque, or the compiler computes every element's key and tag ahead
              // of the branch.)
              float v = acc[a][y][r];
              uint32_t half = 64u * h;
              asm volatile("" : "+v"(v), "+v"(half));
              const uint32_t p0 = ((uint32_t)m >> li) & 1u, p1 = ((uint32_t)(m >> 32) >> li) & 1u;
              const uint32_t slot = cnt[y] + (h ? p0 : 0u);
              if (v >= gl[y] && slot < (uint32_t)CAP) {
                const uint32_t key = __float_as_uint(L2 ? -v : -f1 * v);
                mybuf[slot * 64 + y * 32 + li] = (key & ~127u) | (uint32_t)(16 * a + r) | half;
              }
              cnt[y] += p0 + p1;
              over = over || cnt[y] > (uint32_t)CAP;
            }
          }
        }
      if (ONE) break;  // (its buffers go out as they are; an overflow shows in cnt)
      if (pass == 0 && __ballot(over) != 0ull) {
        cnt[0] = cnt[1] = 0u;
        pass = 1;
        continue;
      }
      if (any) {  // (wave-uniform)
        flush(base);
        set_limit(published());
      }
      if (pass == 0 || pass == 4 * WA) break;
      pass++;
    }
    publish();
  };

  // SCORES: a lane's four consecutive columns of its row are 16 bytes, and the
  // block's four such stores a row fill a 128-byte line in L2.
  auto store = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < WN; y++) {
      const int r = row0 + wr * 64 + y * 32 + li;
      if (r >= nrows) continue;
      float* o = a_.scores + (size_t)r * a_.ldS;
#pragma unroll
      for (int a = 0; a < WA; a++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const size_t col = (size_t)tile * T5 + wc * 128 + a * 32 + 8 * q + 4 * h;
          if (col < a_.ldS)
            *reinterpret_cast<float4*>(o + col) =
                make_float4(f1 * acc[a][y][4 * q], f1 * acc[a][y][4 * q + 1],
                            f1 * acc[a][y][4 * q + 2], f1 * acc[a][y][4 * q + 3]);
        }
    }
  };

  // Prologue: steps 0 .. NS5 - 1 into their stages; step 0's first operands.
  for (int i = tid; i < 2 * (TOPK ? 2 : 1) * T5; i += 512) (&pub[0][0][0])[i] = INFINITY;
#pragma unroll
  for (int s = 0; s < NS5; s++) {
#pragma unroll
    for (int q = 0; q < 2 * ND; q++) dma_part(q);
    advance();
  }
  wait_vm<(NS5 - 1) * PER>();  // step 0's DMAs are in (the others' stay in flight)
  __syncthreads();
  Rows r0, r1;
  read_rows(0, 0, r0);
#pragma unroll
  for (int a = 0; a < WA; a++) read_cent(0, 0, a);
  int ct = t0, cj = 0;  // compute cursor: tile and slab of the current step
  // A step: slab s in stage s % NS5. While the first MFMA step runs, each
  // centroid block's operands are replaced by the second's as soon as its
  // MFMAs are issued. Then the wave's DMAs of step s + 1 are in (those of s +
  // 2 and s + 3 may be in flight) and its reads of this stage done, and the
  // barrier makes that every wave's; the second MFMA step's groups read step
  // s + 1's first operands and issue the DMAs of step s + NS5 into this stage
  // (ls: the load cursor is NS5 steps ahead). After a tile's last step the
  // fold comes before those reads, which keeps their registers free for it.
  for (int s = 0, st = 0; s < nsteps; s++) {
    if (cj == 0) {
      // A tile's first MFMAs start its accumulators from +0.
      v16f z;
#pragma unroll
      for (int r = 0; r < 16; r++) z[r] = 0.f;
#pragma unroll
      for (int a = 0; a < WA; a++) {
#pragma unroll
        for (int y = 0; y < WN; y++)
          acc[a][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ca[a], r0.b[y], z, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (a == 0) read_rows(st, 1, r1);
        read_cent(st, 1, a);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int a = 0; a < WA; a++) {
#pragma unroll
        for (int y = 0; y < WN; y++)
          acc[a][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ca[a], r0.b[y], acc[a][y], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (a == 0) read_rows(st, 1, r1);
        read_cent(st, 1, a);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    wait_vm<(NS5 - 2) * PER>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    const bool last = cj + 1 == d32;
    const int nx = (st + 1) % NS5;
#pragma unroll
    for (int a = 0; a < WA; a++) {
#pragma unroll
      for (int y = 0; y < WN; y++)
        acc[a][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ca[a], r1.b[y], acc[a][y], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (!last) {
        if (a == 0) read_rows(nx, 0, r0);
        read_cent(nx, 0, a);
      }
      dma_part(a);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(2 * ND == WA, "one DMA per group of MFMAs");
    advance();
    st = nx;
    cj++;
    if (last) {
      if constexpr (LISTS)
        fold(ct);
      else
        store(ct);
      cj = 0;
      ++ct;
      read_rows(st, 0, r0);
#pragma unroll
      for (int a = 0; a < WA; a++) read_cent(st, 0, a);
    }
  }
  wait_vm<0>();  // the DMAs past the last step have landed (the output reuses the stages)
  if constexpr (!LISTS) return;

  // The rows' candidates: of the two threads' logs (ONE: buffers), what lies
  // within the final limit, into [row][part][L]. Top-1: the length and that
  // many entries, the best first; more than L, or a log that did not hold
  // everything: a length beyond L. kNN: in any order, the unused entries
  // {+inf, NONE}; more than L: L entries of -inf, which settle no row.
  const int L = TOPK ? a_.L : L5;
  constexpr int RS = (TOPK ? LK5 : L5) | 1, KS = NK | 1;  // LDS strides of a row's entries, and of a thread's keys
  float* OK = reinterpret_cast<float*>(ring);
  uint32_t* OI = reinterpret_cast<uint32_t*>(OK + T5 * RS);
  uint32_t* on = OI + T5 * RS;
  float* TK = reinterpret_cast<float*>(on + T5);
  static_assert((2 * T5 * RS + T5 + 512 * KS) * 4 <= NS5 * S5_STAGE, "output space");
  __syncthreads();  // every wave's DMAs are in and its keys published
  if (tid < T5) on[tid] = 0u;
  if (TOPK) {
#pragma unroll
    for (int e = 0; e < NK; e++) TK[tid * KS + e] = lkey[e];
  }
  __syncthreads();
  {
    // The limit from the row's exact kk-th key (the published ones bound it
    // by a key of rank kk .. 2 kk - 1, whose candidates may not fit the list).
    float b = TOPK ? INFINITY : published();
    if (TOPK) {
      const float *A = TK + prow * KS, *B = TK + (T5 + prow) * KS;
      for (int e = 0, i = 0; e < kk; e++) {  // i of A's and e - i of B's are the e smallest
        const float va = A[i], vb = B[e - i];
        b = fminf(va, vb);
        i += va <= vb ? 1 : 0;
      }
    }
    const float lim = limit_of(b);
    // A limit past the largest finite key: keys that overflowed may be within
    // it, and no entry says so.
    if (L2 && !(lim <= 3.4028235e38f)) spilt = true;
    auto keep = [&](float key, uint32_t id) __attribute__((always_inline)) {
      if (key <= lim) {
        const uint32_t e = atomicAdd(&on[prow], 1u);
        if (e < (uint32_t)L) {
          OK[prow * RS + e] = key;
          OI[prow * RS + e] = id;
        }
      }
    };
    if (ONE) {
      const uint32_t n = h ? cnt[1] : cnt[0];
      spilt = spilt || n > (uint32_t)CAP;
      for (uint32_t i = 0; i < min(n, (uint32_t)CAP); i++) {
        const uint32_t v = mybuf[i * 64 + lane];
        keep(__uint_as_float(v), (uint32_t)(t0 * T5 + wc * 128) + column(v));
      }
    } else {
      for (uint32_t i0 = 0; i0 < nlog; i0 += 8) {
        Cand v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = mylog(min(i0 + u, nlog - 1));
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (i0 + u < nlog) keep(v[u].key, v[u].id);
      }
    }
    if (spilt) atomicAdd(&on[prow], (uint32_t)(2 * L));
  }
  __syncthreads();
  if (TOPK) {  // eight lanes a row: 64 bytes of its list at a time
    for (int r = tid >> 3; r < min(T5, nrows - row0); r += 64) {
      Cand* out = a_.cand + ((size_t)(row0 + r) * parts + part) * L;
      const int n = (int)on[r];
      for (int e = tid & 7; e < L; e += 8)
        out[e] = n > L ? Cand{-INFINITY, 0u}
                 : e < n ? Cand{OK[r * RS + e], OI[r * RS + e]}
                         : Cand{INFINITY, NONE};
    }
  } else if (tid < T5 && row0 + tid < nrows) {
    const size_t at0 = (size_t)(row0 + tid) * parts + part;
    Cand* out = a_.cand + at0 * L;
    const uint32_t n = on[tid];
    const bool full = n > (uint32_t)L;
    a_.ncand[at0] = n;
    uint32_t best = 0;
    for (uint32_t e = 1; e < (full ? 0u : n); e++)
      best = OK[tid * RS + e] < OK[tid * RS + best] ? e : best;
    for (uint32_t e = 0; e < (full ? 0u : n); e++) {
      const uint32_t at = tid * RS + (e == 0 ? best : e == best ? 0u : e);
      out[e] = Cand{OK[at], OI[at]};
    }
  }
}

}  // namespace
}  // namespace emh
