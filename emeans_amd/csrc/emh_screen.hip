// Fused top-1 (Device::top1, core/mod.rs:97-112) and exact top-k
// (Device::topk, core/mod.rs:114-124) for gfx950: the MFMA screen and the
// orchestration of the check (emh_rescore.hip) and exact scans (emh_verify.hip).
//
// Exactness: the reference CPU backend (cpu-fused, assign/fused.rs) scores
// every (row, centroid) pair with one sequential f32 fma chain over the d
// dimensions. The screen computes the same dot products on the MFMA: in one
// fp16 pass over rows rounded ahead (k_screen5, whose bound rests on the
// measured residuals: screen_bound_lines, emh_lines.h), or, for small calls and
// the no-allocation entry, on the bf16 MFMA in three passes (x.c ~ xh.ch +
// xh.cl + xl.ch, the halves rounded to nearest even, f32 accumulation), whose
// scores differ from the chain's by about 2^-16 |x| |c| plus the
// accumulation's rounding. The path therefore has three stages:
//
//  1. screen (MFMA, the dense x . C^T contraction): per part (a range of
//     centroid tiles) each row keeps the L smallest screen keys (key = -dot
//     for IP, |c|^2 - 2 dot for L2) with their ids, in registers; the n x k
//     score matrix never leaves the CU.
//  2. check: bound the screen error E rigorously from |x| and max|c|. A
//     part's list holds every centroid of the part whose screen key is at
//     most best + 2E when the list is not full or its L-th key is above
//     best + 2E; with every part so, the centroids that can win are among
//     the lists' entries within best + 2E: re-score exactly those (at most
//     C1) with the fma chain and take the smallest exact key, lower id on
//     ties. Otherwise queue the row.
//  3. exact: the full fma-chain scan of the queued rows over all k centroids.
//
// The same stages with a longer list, merged over the parts, give the exact
// top-k of kNN.
//
// Bound of the bf16 screens (screen_bound, emh_select.h): the chain is within gamma_d sum|x_t c_t|
// of the exact dot (gamma_d = d u / (1 - d u), u = 2^-24) and sum|x_t c_t| <=
// |x| |c|; the screen adds the split's dropped and rounded parts
// (<= 3.05 * 2^-16 |x| |c|) and the MFMA chain's rounding (each MFMA within
// 16 u of its terms' magnitudes); L2 keys add the rounding of |c|^2 - 2 dot
// on both sides (one rounding in the screen's fma, two in the check's). E
// carries a 12.5% margin for its own rounding.

#include "emh_lines.h"
#include "emh_screen_kern.h"

namespace emh {
namespace {

// The 128 x 128 screens in the context's arithmetic (f32 in SCREEN_F32, else bf16).
void launch_screen_t1(emh_ctx* c, const ScreenArgs& a, bool ip) {
  if (c->screen == SCREEN_F32)
    launch_screen_t1_f32(c, a, ip);
  else
    launch_screen_t1_bf3(c, a, ip);
}
void launch_screen_kn(emh_ctx* c, const ScreenArgs& a, bool exclude_self) {
  if (c->screen == SCREEN_F32)
    exclude_self ? launch_screen_kn_f32_self(c, a) : launch_screen_kn_f32_any(c, a);
  else
    exclude_self ? launch_screen_kn_bf3_self(c, a) : launch_screen_kn_bf3_any(c, a);
}

int choose_parts(int row_tiles, int ntiles, int cus, int per_cu = 2) {
  // Enough blocks for per_cu per CU (all resident at once), never more parts
  // than tiles, and at most MAX_PARTS lists per row for the verify to merge.
  int want = (per_cu * cus + row_tiles - 1) / row_tiles;
  return std::max(1, std::min(std::min(want, ntiles), MAX_PARTS));
}

}  // namespace

namespace {
// The screen's launch geometry for n rows against k centroids. split: the
// call may take a split-operand screen (k >= 64, any d >= 32): the one-pass
// screen over fp16 lines (k_screen5; parts of one tile of 256 centroids while
// there are at most MAX_PARTS tiles, else of several) or, in SCREEN_F16 with
// at most MAX_PARTS tiles, the two-pass one (k_screen4). Otherwise (and for
// the no-allocation entry, which has no room to split a selection) the
// large-tile screen that splits its slabs itself (k_screen3, d % 4 == 0, k >=
// 64) or the 128 x 128 screens.
struct Top1Geom {
  bool screen, big, split;
  int row_tiles, ntiles, parts, tpp;
};
Top1Geom top1_geom(emh_ctx* c, size_t n, size_t d, size_t k, bool ip, bool split,
                   bool small_exact) {
  Top1Geom g{};
  // The screen for any k >= 2 with d >= 32: below that, and for k = 1, the
  // exact scan is as fast. (At small k the exact scan's items leave most
  // lanes idle: 900,000 rows against 40 centroids took 10x the screen's time.)
  // With small_exact, calls of at most c->exact_below exact items, or small
  // enough for the latency-bound scan, take the exact kernels too: one launch
  // beats the screen's three there.
  g.screen = c->screen && k >= 2 && d >= 32 &&
             !(small_exact && (exact_items(n, k) <= c->exact_below ||
                               queued_direct(c, n, d, k, ip)));
  if (!g.screen) return g;
  const int nt3 = (int)((k + TC3 - 1) / TC3);
  // (The split-operand screens address a slab's rows with 32-bit offsets: fewer than 2^25 rows.)
  // A selection that gives the large tiles fewer blocks than half the CUs (an
  // epoch's tail batch) takes the 128 x 128 screen, which splits its rows
  // itself: two launches less. Whole IP calls in us, one-pass / 128 x 128, d =
  // 64, 384, 1,024: 3,392 rows x 1,024 centroids (56 tiles) 38 / 29, 47 / 42, 68 /
  // 72; 16,384 x 128 (64 tiles) 39 / 29, 52 / 44, 82 / 75; 12,000 x 512 (94 tiles)
  // 40 / 34, 51 / 50, 78 / 83. Not past MAX_PARTS tiles of centroids, where the
  // 128 x 128 screen takes several a part: 2,545 x 3,000 (120 tiles) 49 / 47, 66 /
  // 85, 96 / 159; 600 x 10,000 66 / 106, 103 / 224, 169 / 461.
  const size_t blocks3 = (n + TR3 - 1) / TR3 * (size_t)nt3;
  const bool lines = c->screen != SCREEN_F16;  // the split-operand screen is the one-pass one
  const bool few = 2 * blocks3 < (size_t)c->cus && (nt3 <= MAX_PARTS || !lines);
  if (split && !few && c->screen != SCREEN_F32 && k >= 64 && (lines || nt3 <= MAX_PARTS) &&
      n < (1u << 25) && k < (1u << 25)) {
    g.big = g.split = true;
    g.row_tiles = (int)((n + TR3 - 1) / TR3);
    g.ntiles = nt3;
    g.parts = nt3 <= MAX_PARTS ? nt3 : parts5(g.row_tiles, nt3, c->cus, MAX_PARTS, 0.5);
    g.tpp = (g.ntiles + g.parts - 1) / g.parts;
    g.parts = (g.ntiles + g.tpp - 1) / g.tpp;
    return g;
  }
  // The large-tile bf16 screen (one 512-thread block per CU, 256-centroid
  // tiles) when d % 4 == 0 and k >= 64; smaller k fill a 128-centroid tile
  // better.
  g.big = c->screen != SCREEN_F32 && d % 4 == 0 && k >= 64 && !(split && few);
  const int TR = g.big ? TR3 : 128;
  g.row_tiles = (int)((n + TR - 1) / TR);
  g.ntiles = (int)((k + (g.big ? TC3 : TC) - 1) / (g.big ? TC3 : TC));
  g.parts = choose_parts(g.row_tiles, g.ntiles, c->cus, g.big ? 1 : 2);
  g.tpp = (g.ntiles + g.parts - 1) / g.parts;
  g.parts = (g.ntiles + g.tpp - 1) / g.tpp;
  return g;
}
}  // namespace

bool split_screen(emh_ctx* c, size_t n, size_t d, size_t k, bool ip) {
  return top1_geom(c, n, d, k, ip, true, true).split;
}
bool top1_screens(emh_ctx* c, size_t n, size_t d, size_t k, bool ip) {
  return top1_geom(c, n, d, k, ip, false, true).screen;
}
bool top1_tallies(emh_ctx* c, size_t n, size_t d, size_t k, bool ip) {
  // queued_direct holds for every smaller selection too (its items grow with n).
  return d % 4 == 0 && (top1_screens(c, n, d, k, ip) || queued_direct(c, n, d, k, ip));
}

SplitCents split_cents(emh_ctx* c, const float* cents, size_t d, size_t k, const float* cnorm,
                       const float* scale, const float* mean) {
  const LinesOut o{scale, c->csplit.get(lines_bytes(k, d)), (float2*)c->csplit_norm.get(k * 8)};
  const size_t nb = lines_blocks(k);
  uint32_t* pw = (uint32_t*)c->csplit_part.get((nb + 1) * 16);
  launch_lines(c, cents, k, d, nullptr, 0, k, o, cnorm, pw, mean);
  SplitCents s;
  s.cs = o.out;
  s.part = pw;
  s.nparts = (int)nb;
  s.scale = scale;
  s.mean = mean;
  if (nb > PART_MAX_ONCE) {
    launch_part_max4(c, pw, nb, pw + 4 * nb);
    s.part = pw + 4 * nb;
    s.nparts = 1;
  }
  return s;
}

size_t top1_scratch_bytes(emh_ctx* c, size_t n, size_t d, size_t k, bool ip) {
  const Top1Geom g = top1_geom(c, n, d, k, ip, false, true);
  if (!g.screen) return exact1_scratch_bytes(c, n, d, k, ip, false);
  auto r = [](size_t b) { return (b + 255) & ~size_t(255); };
  return r((size_t)g.parts * n * L1 * sizeof(Cand)) + 2 * r(n * 4) +
         exact1_scratch_bytes(c, n, d, k, ip, true);
}

namespace {
// The screen stage of a top-1 call: its lists, their parts, the rows' |x|^2
// (BOUND_LINES: their E), the check's queue and the arithmetic the check's
// bound must follow.
struct Top1Screen {
  Top1Geom g;
  Cand* cand = nullptr;
  uint32_t* ncand = nullptr;  // the lists' lengths (BOUND_LINES)
  uint32_t* fb = nullptr;
  float* xnorm = nullptr;
  BoundKind bound = BOUND_F32;
  int L = L1;  // entries per part list
  const float* mean = nullptr;  // BOUND_LINES: the keys are off by x.mean (L2: 2 x.mean)
};

// The one-pass screen's scales and the centroids' mean: the caller's, or this
// call's, in one launch that also clears the screen's words.
struct Frames {
  const float *sx, *sc, *mean;
};
Frames top1_frames(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids, size_t lo,
                   size_t n, const float* cents, size_t k, const SplitRows* pre,
                   const SplitCents* pc, bool& words_clear) {
  Frames f{pre ? pre->scale : nullptr, pc ? pc->scale : nullptr, pc ? pc->mean : nullptr};
  if (f.sx && f.sc) return f;
  float* wx = c->scales + 2 * SCALE_ROWS;
  float* wc = c->scales + 2 * SCALE_CENTS;
  float* mean = f.sc ? nullptr : (float*)c->cmean.get(mean_floats(d) * 4);
  const ScaleIn ix{x, nx, ids, lo, n, wx, -50}, ic{cents, k, nullptr, 0, k, wc, -50, mean};
  launch_scales(c, d, f.sx ? ic : ix, !f.sx && !f.sc ? &ic : nullptr, c->small,
                words_clear ? 0 : 3);
  words_clear = true;
  if (!f.sx) f.sx = wx;
  if (!f.sc) {
    f.sc = wc;
    f.mean = mean;
  }
  return f;
}

Top1Screen screen_top1(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids,
                       size_t lo, size_t n, const float* cents, const float* cnorm, size_t k,
                       bool ip, bool words_clear, Arena* ar, const SplitRows* pre,
                       const SplitCents* pc, bool small_exact) {
  Top1Screen s;
  s.g = top1_geom(c, n, d, k, ip, !ar, small_exact);
  if (!s.g.screen) return s;
  const Top1Geom& g = s.g;
  const bool f16 = g.split && c->screen == SCREEN_F16;
  const bool tagged = g.big && g.tpp == 1;
  s.bound = c->screen == SCREEN_F32 ? BOUND_F32
            : f16                   ? BOUND_F16_TAGGED
            : g.split               ? BOUND_LINES
            : tagged                ? BOUND_BF16_TAGGED
                                    : BOUND_BF16;
  s.L = f16 ? L1F : g.split ? L5 : g.big && !tagged ? L1S : L1;
  const size_t cbytes = (size_t)g.parts * n * s.L * sizeof(Cand);
  // (The one-pass screen's lists are followed by their lengths.)
  const size_t lbytes = g.split && !f16 ? (size_t)g.parts * n * 4 : 0;
  s.cand = (Cand*)(ar ? ar->take(cbytes) : c->cand.get(cbytes + lbytes));
  if (lbytes) s.ncand = (uint32_t*)((char*)s.cand + cbytes);
  s.fb = (uint32_t*)(ar ? ar->take(n * 4) : c->fblist.get(n * 4));
  const size_t nb = g.split && !f16 ? 2 * n * 4 : n * 4;  // E and its dot term, or |x|^2
  s.xnorm = (float*)(ar ? ar->take(nb) : c->xnorm.get(nb));
  // The words a screen starts from: fallback count, cmax2, cnmax (the maxima
  // filled by the screen or the split).
  auto clear_words = [&] {
    if (!words_clear) launch_fill_u32(c, c->small, 3, 0);
    words_clear = true;
  };
  const unsigned blocks = (unsigned)(g.row_tiles * g.parts);
  if (g.split) {
    EMH_ENSURE(!pre || pre->f16 == f16, "top1: rows split in the other format");
    EMH_ENSURE(!pc || pc->f16 == f16, "top1: centroids split in the other format");
  }
  if (g.split && !f16) {
    // The one-pass screen. What the caller did not bring: the scales, the
    // centroids' lines, then the selection's.
    const Frames f = top1_frames(c, x, nx, d, ids, lo, n, cents, k, pre, pc, words_clear);
    const float *sx = f.sx, *sc = f.sc;
    s.mean = f.mean;
    clear_words();
    Lines5 a{};
    if (pc && pc->cs) {
      a.cs = pc->cs;
      a.part = pc->part;
      a.nparts = pc->nparts;
    } else {
      const SplitCents own = split_cents(c, cents, d, k, ip ? nullptr : cnorm, sc, s.mean);
      a.cs = own.cs;
      a.part = own.part;
      a.nparts = own.nparts;
    }
    if (pre && pre->xs) {
      a.xs = pre->xs;
      a.xslab = pre->slab;
      a.xn = (const float2*)pre->xn;
      a.nx = pre->nx;
      a.ids = ids;
      a.lo = lo;
    } else {
      const LinesOut o{sx, c->xsplit.get(lines_bytes(n, d)), (float2*)c->xsplit_norm.get(n * 8)};
      launch_lines(c, x, nx, d, ids, lo, n, o);
      a.xs = o.out;
      a.xslab = n * LINE_BYTES;
      a.xn = o.norm;
      a.nx = n;
    }
    a.n = n;
    a.cnorm = cnorm;
    a.k = k;
    a.d = d;
    a.tpp = g.tpp;
    a.parts = g.parts;
    a.ntiles = g.ntiles;
    a.cand = s.cand;
    a.ncand = s.ncand;
    a.bound = s.xnorm;
    a.sx = sx;
    a.sc = sc;
    ProfScope prof(c, EMH_PROF_SCREEN, 2.0 * (double)n * (double)k * (double)d,
                   prof_take(c, EMH_PROF_SCREEN));
    launch_screen5(c, a, ip);
    return s;
  }
  clear_words();
  if (g.split) {
    // The two-pass screen: the centroids' halves and the bound's centroid
    // maxima (the caller's, split ahead, or split here), then the rows'
    // halves (the caller's, or this selection's).
    const void* cs;
    const uint32_t* part;
    int nparts;
    if (pc) {
      cs = pc->cs;
      part = pc->part;
      nparts = pc->nparts;
    } else {
      void* cw = c->csplit.get(halves_bytes(k, d));
      uint32_t* pw = (uint32_t*)c->csplit_part.get(halves_blocks(k) * 16);
      launch_halves(c, cents, k, d, nullptr, 0, k, cw, (float*)c->csplit_norm.get(k * 4),
                    ip ? nullptr : cnorm, pw);
      cs = cw;
      part = pw;
      nparts = (int)halves_blocks(k);
    }
    Screen4Args a{blocks, nullptr, 0,       nullptr, 0,       d,    nullptr, 0,
                  n,      cs,      k * 128, cnorm,   k,       1,    g.parts, g.ntiles,
                  s.cand, s.xnorm, part,    nparts};
    if (pre) {
      a.xs = pre->xs;
      a.xslab = pre->slab;
      a.xn = (const float*)pre->xn;
      a.nx = pre->nx;
      a.ids = ids;
      a.lo = lo;
    } else {
      void* xs = c->xsplit.get(halves_bytes(n, d));
      launch_halves(c, x, nx, d, ids, lo, n, xs, s.xnorm, nullptr, nullptr);
      a.xs = xs;
      a.xslab = n * 128;
      a.xn = s.xnorm;
      a.nx = n;
    }
    ProfScope prof(c, EMH_PROF_SCREEN, 2.0 * (double)n * (double)k * (double)d,
                   prof_take(c, EMH_PROF_SCREEN));
    launch_screen4(c, a, ip);
    return s;
  }
  ProfScope prof(c, EMH_PROF_SCREEN, 2.0 * (double)n * (double)k * (double)d,
                 !ar && prof_take(c, EMH_PROF_SCREEN));
  const ScreenArgs a{blocks, x, nx, d, ids, lo, n, cents, cnorm, k, g.tpp, g.parts, g.ntiles,
                     s.cand, s.xnorm};
  // One tile per part: tagged keys (the cheap fold); more: the sorted
  // insert, which skips most keys once the lists hold good ones.
  if (g.big)
    launch_screen3(c, a, ip, tagged);
  else
    launch_screen_t1(c, a, ip);
  return s;
}

}  // namespace

void launch_top1(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids, size_t lo,
                 size_t hi, const float* cents, const float* cnorm, size_t k, bool ip,
                 uint32_t* labels, float* scores, bool words_clear, Arena* ar,
                 const SplitRows* pre, const SplitCents* pc, const LabelTally* tally) {
  if (hi <= lo) return;
  const size_t n = hi - lo;
  EMH_ENSURE(d <= 16384, "top1: d = %zu above the supported 16384", d);
  EMH_ENSURE(n < (1u << 31) && k < (1u << 31), "top1: shape too large");
  // (Every kernel reads row 0 in place of a row whose id is out of range.)
  EMH_ENSURE(nx > 0, "top1: a selection of %zu rows over no data rows", n);
  // A tallying call takes the screen, or the latency-bound exact scan, which
  // tallies too; never k_exact1.
  const bool small_exact = !tally || queued_direct(c, n, d, k, ip);
  // Large selections on the one-pass screen go a piece at a time (a multiple of
  // the tally's chunks), which bounds the copy of the rows as lines and their
  // lists (1,056 bytes a row at eight parts); scales and centroids once.
  constexpr size_t PIECE = size_t(1) << 20;
  static_assert(PIECE % TALLY_CP == 0, "a piece starts a tally chunk");
  if (n > PIECE && !ar && c->screen != SCREEN_F16 &&
      top1_geom(c, PIECE, d, k, ip, true, small_exact).split) {
    const Frames f = top1_frames(c, x, nx, d, ids, lo, n, cents, k, pre, pc, words_clear);
    SplitRows pr = pre ? *pre : SplitRows{};
    pr.scale = f.sx;
    const SplitCents cc = pc && pc->cs ? *pc
                                       : split_cents(c, cents, d, k, ip ? nullptr : cnorm, f.sc,
                                                     f.mean);
    for (size_t b = lo; b < hi; b += PIECE) {
      launch_top1(c, x, nx, d, ids, b, std::min(b + PIECE, hi), cents, cnorm, k, ip, labels, scores,
                  words_clear, nullptr, &pr, &cc, tally);
      words_clear = false;
    }
    return;
  }
  const Top1Screen s = screen_top1(c, x, nx, d, ids, lo, n, cents, cnorm, k, ip, words_clear, ar,
                                   pre, pc, small_exact);
  EMH_ENSURE(!tally || (d % 4 == 0 && (s.g.screen || queued_direct(c, n, d, k, ip))),
             "top1: labels are tallied only by the screen or the queued-row scan, d %% 4 == 0");
  if (!s.g.screen) {
    launch_exact1(c, x, nx, d, ids, lo, n, nullptr, cents, cnorm, k, ip, labels, scores, ar,
                  tally);
    return;
  }
  launch_verify1(c, x, nx, d, ids, lo, n, cents, cnorm, k, ip, s.cand, s.g.parts, s.xnorm, labels,
                 scores, s.fb, s.bound, tally, s.L, s.ncand);
  launch_exact1(c, x, nx, d, ids, lo, n, s.fb, cents, cnorm, k, ip, labels, scores, ar, tally);
}

void screen_margin_top1(emh_ctx* c, const float* x, size_t nx, size_t d, const uint32_t* ids,
                        size_t lo, size_t hi, const float* cents, const float* cnorm, size_t k,
                        bool ip, emh_screen_report* out) {
  *out = emh_screen_report{};
  if (hi <= lo) return;
  const size_t n = hi - lo;
  EMH_ENSURE(d <= 16384 && n < (1u << 31) && k < (1u << 31), "top1: shape too large");
  EMH_ENSURE(nx > 0, "top1: a selection of %zu rows over no data rows", n);
  const Top1Screen s =
      screen_top1(c, x, nx, d, ids, lo, n, cents, cnorm, k, ip, false, nullptr, nullptr, nullptr,
                  false);
  if (!s.g.screen) return;  // variant 0: no screen, nothing to measure
  out->variant = s.bound == BOUND_F16_TAGGED ? EMH_SCREEN_BIG_F16
                 : s.g.big ? (s.g.tpp == 1 ? EMH_SCREEN_BIG_TAGGED : EMH_SCREEN_BIG_SORTED)
                           : (c->screen == SCREEN_F32 ? EMH_SCREEN_SMALL_F32 : EMH_SCREEN_SMALL_BF16);
  out->parts = s.g.parts;
  out->tiles_per_part = s.g.tpp;
  launch_margin(c, x, nx, d, ids, lo, n, cents, cnorm, ip, s.cand, s.g.parts, s.L, s.xnorm,
                s.bound, out, s.ncand, s.mean);
}

void launch_topk(emh_ctx* c, const float* q, size_t m, const float* data, size_t n, size_t d,
                 size_t kk, bool exclude_self, uint32_t* ids, float* sims, emh_screen_report* rep) {
  if (m == 0) return;
  if (kk > (size_t)KMAX && !rep) {  // beyond the screen's lists: the exact top-k
    launch_topk_long(c, q, m, data, n, d, kk, exclude_self, ids, sims);
    return;
  }
  EMH_ENSURE(kk >= 1 && kk <= (size_t)KMAX, "topk: kk = %zu must be in 1..16", kk);
  EMH_ENSURE(d <= 16384, "topk: d = %zu above the supported 16384", d);
  EMH_ENSURE(m < (1u << 31) && n < (1u << 31), "topk: shape too large");
  if (n > 0 && screen5_knn_fits(c, m, n, d)) {
    // The one-pass large-tile screen, then the same check.
    Cand* cand = nullptr;
    float* xnorm = nullptr;
    const float* mean = nullptr;
    int L = 0;
    const int parts = screen5_knn(c, q, m, data, n, d, kk, exclude_self, &cand, &L, &xnorm, &mean);
    if (rep) {
      *rep = emh_screen_report{};
      rep->variant = EMH_SCREEN_BIG_KNN;
      rep->parts = parts;
      rep->tiles_per_part = 0;
      launch_margin(c, q, m, d, nullptr, 0, m, data, nullptr, true, cand, parts, L, xnorm,
                    BOUND_LINES, rep, nullptr, mean);
      return;
    }
    uint32_t* fb = (uint32_t*)c->fblist.get(m * 4);
    launch_verifyk(c, q, m, data, n, d, kk, cand, parts, L, xnorm, ids, sims, fb, BOUND_LINES);
    launch_exactk(c, q, m, data, n, d, kk, exclude_self, fb, ids, sims);
    return;
  }
  const int TR = 64;
  const int row_tiles = (int)((m + TR - 1) / TR);
  const int ntiles = (int)((n + TC - 1) / TC);
  int parts = choose_parts(row_tiles, std::max(ntiles, 1), c->cus);
  const int tpp = (std::max(ntiles, 1) + parts - 1) / parts;
  parts = (std::max(ntiles, 1) + tpp - 1) / tpp;
  Cand* cand = (Cand*)c->cand.get((size_t)parts * m * LK * sizeof(Cand));
  uint32_t* fb = (uint32_t*)c->fblist.get(m * 4);
  float* xnorm = (float*)c->xnorm.get(m * 4);
  launch_fill_u32(c, c->small, 3, 0);
  if (n > 0) {
    ProfScope prof(c, EMH_PROF_SCREEN, 2.0 * (double)m * (double)n * (double)d,
                   prof_take(c, EMH_PROF_SCREEN));
    const unsigned blocks = (unsigned)(row_tiles * parts);
    launch_screen_kn(c, ScreenArgs{blocks, q, m, d, nullptr, 0, m, data, nullptr, n, tpp, parts,
                                   ntiles, cand, xnorm},
                     exclude_self);
  } else {
    parts = 1;
    launch_fill_u32(c, (uint32_t*)cand, m * LK * 2, NONE);  // empty lists
    launch_fill_u32(c, (uint32_t*)xnorm, m, 0);
  }
  if (rep) {  // the diagnostic: measure the lists, change nothing
    *rep = emh_screen_report{};
    if (n == 0) return;
    rep->variant = c->screen == SCREEN_F32 ? EMH_SCREEN_SMALL_F32 : EMH_SCREEN_SMALL_BF16;
    rep->parts = parts;
    rep->tiles_per_part = tpp;
    launch_margin(c, q, m, d, nullptr, 0, m, data, nullptr, true, cand, parts, LK, xnorm,
                  c->screen != SCREEN_F32 ? BOUND_BF16 : BOUND_F32, rep);
    return;
  }
  launch_verifyk(c, q, m, data, n, d, kk, cand, parts, LK, xnorm, ids, sims, fb,
                 c->screen == SCREEN_F32 ? BOUND_F32 : BOUND_BF16);
  launch_exactk(c, q, m, data, n, d, kk, exclude_self, fb, ids, sims);
}

}  // namespace emh
