// Grouped MFMA GEMM: precision dispatch and host-side tile planning (the kernels are in
// gemm_kernels.hpp, instantiated by gemm_fp64.hip, gemm_fp32.hip, gemm_c64.hip, gemm_fp32x3.hip
// and gemm_mix.hip).
#define CXA_GEMM_TU main
#include "gemm_kernels.hpp"

namespace cxa {

int launch_grouped_gemm(const GemmLaunch &g, hipStream_t s) {
  if (g.outs && g.dot_part)
    return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: no dot epilogue on mix launches");
  if (g.outs) return launch_mix(g, s);
  switch (g.prec) {
    case CXA_PREC_FP64: return launch_gemm_fp64(g, s);
    case CXA_PREC_FP32: return launch_gemm_fp32(g, s);
    case CXA_PREC_FP32X3: return launch_gemm_fp32x3(g, s);
    default: break;
  }
  return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: unsupported precision %d", g.prec);
}

int default_kind(int M, int N) {
  if (M <= 16 && N <= 16) return TK_1x1;
  if (M <= 16) return TK_1x2;
  if (N <= 16) return TK_2x1;
  return TK_2x2;
}

namespace {

int64_t tiles_of(const GBlk &b, int t) {
  return (int64_t)((b.M + t - 1) / t) * ((b.N + t - 1) / t);
}

// The choice, from counts of tiles and the mean K in chunks of 16.  A 16 x 16 tile is the finest
// split of the output, and a wave works through its K one MFMA after another, so few tiles leave SIMDs
// idle: up to kFew of them (two, complex four, times the CUs; single products half) the four waves
// of a workgroup share a tile's K, which then also hides their load latency.  Beyond, tiles of one
// wave: the default ones from kManyDirect of them (three per CU), else 16 x 16.  With more than
// kShortChunks of K (lists of complex128 blocks kShortC128) the LDS tiles, which read every operand
// element once per 32 or 64 rows instead of once per 16 or 32, unless they cover more than 1.15
// times the area of the default tiles.  64 x 64 tiles (a quarter of the chunk loads and barriers
// per flop) from kMany64 of them, real types only: a complex one's registers leave one or two
// waves per SIMD.
// Measured, us:
//   split 16x16 / LDS 32x32: real products of n = 128 3.9 / 5.2, 256 4.9 / 7.3, 512 (1024 tiles)
//   21.2 / 11.5; complex128 n = 256 6.4 / 13.9, 384 x 960 x 192 (288 tiles) 27 / 43, 512 30 / 26;
//   default / 16x16: FP32 20000 x 33 x 20 (625 of them) 5.0 / 4.8, 600 x 600, K = 100 7.0 / 5.7,
//   1000 x 1000 (1024) 7.3 / 9.5, 200 blocks of 60 x 60 (800), K = 50 5.7 / 7.4;
//   direct / LDS (64x64 of real types): 3000 x 3000, K = 33 FP32 19.0 / 30.7, complex64 41.7 / 67.6;
//   K = 100 FP32 31 / 41, FP64 47.7 / 45.1, complex128 137 / 147; 1600 x 1600 complex128, K = 200
//   87 / 77, 1000 x 1000 (1024 LDS tiles) 37 / 43 in a list and 44 / 36 by itself; 60 blocks of
//   160 x 160, K = 400 complex128 107 / 86; covering twice the area: 100000 x 10 x 100 FP64 19.6 /
//   30.7, 10 x 400 x 20000 FP64 13 / 31; 200 blocks of 300 x 8, K = 100 complex64 15.6 / 24.5.
constexpr int64_t kFewReal = 512, kFewCplx = 1024, kMany64 = 192, kManyDirect = 768;
constexpr int64_t kShortChunks = 7, kShortC128 = 13, kRoundLow = 768, kRoundHigh = 1400;

// Blocks counted in tiles and in their work, the chunks of K times the area that the tiles cover.
struct Cover {
  int64_t n16 = 0, n32 = 0, n64 = 0, def = 0;     // tiles: by size, and of the default kinds
  int64_t work = 0;                               // chunks of K over all 16 x 16 tiles
  int64_t area32 = 0, area64 = 0, area_def = 0;   // times the area covered, in 16 x 16
  bool lds = true, wide = false;  // LDS tiles can, direct tiles need 64-bit offsets
  void add(const GBlk &b, const GSeg *segs) {
    if (b.M <= 0 || b.N <= 0) return;
    const int kind = default_kind(b.M, b.N);
    const int64_t t16 = tiles_of(b, 16), t32 = tiles_of(b, 32), t64 = tiles_of(b, 64);
    const int64_t td = (int64_t)((b.M + tile_rows(kind) - 1) / tile_rows(kind)) *
                       ((b.N + tile_cols(kind) - 1) / tile_cols(kind));
    if (b.wide & kWideStrides) wide = true;
    int64_t chunks = 0;
    for (int s = 0; s < b.nseg; ++s) {
      chunks += (segs[s].K + 15) / 16;
      lds = lds && lds_ok(b, segs[s]);
    }
    n16 += t16;
    n32 += t32;
    n64 += t64;
    def += td;
    work += t16 * chunks;
    area32 += 4 * t32 * chunks;
    area64 += 16 * t64 * chunks;
    area_def += tile_rows(kind) * tile_cols(kind) / 256 * td * chunks;
  }
  // lean tiles (TC_LEAN): of complex128 always
  bool lean(int prec, bool cplx) const {
    return !wide && ((cplx && prec == CXA_PREC_FP64) || work <= kShortChunks * n16);
  }
  // direct tiles rather than LDS ones (c128: a list of complex128 blocks)
  bool stay_direct(bool c128) const { return work <= (c128 ? kShortC128 : kShortChunks) * n16; }
  // direct tiles: the default ones where they are many, 16 x 16 otherwise
  int direct(int kind) const { return def >= kManyDirect ? kind : (int)TK_1x1; }
  // beyond the few tiles and the short K: LDS tiles unless they cover much more than direct ones or
  // (c128) are about the four that a CU holds at a time, in a single round
  int large(int kind, bool cplx, bool c128) const {
    if (!lds) return kind;
    const bool l64 = !cplx && n64 >= kMany64;
    const bool round = c128 && n32 >= kRoundLow && n32 < kRoundHigh;
    if (!round && 20 * (l64 ? area64 : area32) <= 23 * area_def) return l64 ? TK_L64 : TK_L32;
    return direct(kind);
  }
};

// Few tiles (under two per SIMD of a 256-CU device), each with a long K (in chunks of 16).
constexpr int64_t kSplitTiles = 2048, kSplitChunks = 8;

}  // namespace

bool lean_tiles(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs, int prec,
                bool cplx) {
  Cover c;
  for (const GBlk &b : blks) c.add(b, segs.data() + b.seg0);
  return c.lean(prec, cplx);
}

Tiling default_tiling(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs, int prec,
                      bool cplx, bool in_order) {
  Cover c;
  bool narrow = !cplx;
  for (const GBlk &b : blks) {
    c.add(b, segs.data() + b.seg0);
    if (b.M > 0 && b.N > kRowsN) narrow = false;
  }
  if (narrow && prec == CXA_PREC_FP32) return {-1, 0};
  if (c.work <= 2 * c.n16) return {narrow ? -1 : c.direct(-1), 0};
  if (c.n16 <= (cplx ? kFewCplx : kFewReal)) return {TK_1x1, in_order ? 0 : 4};
  if (narrow) return {-1, 0};
  const bool c128 = cplx && prec == CXA_PREC_FP64;
  return {c.stay_direct(c128) ? c.direct(-1) : c.large(-1, cplx, c128), 0};
}

Tiling plan_tiling(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs, int prec,
                   bool cplx, bool in_order) {
  const Tiling t = default_tiling(blks, segs, prec, cplx, in_order);
  const bool four_sums = t.split > 0 || (prec == CXA_PREC_FP32 && t.kind == TK_L64);
  if (cplx || t.kind < 0 || four_sums) return t;
  Cover c;
  for (const GBlk &b : blks) c.add(b, segs.data() + b.seg0);
  // (the default tiles' share of the work: their chunks of K, not those of 16 x 16 tiles)
  int64_t work = 0;
  for (const GBlk &b : blks) {
    Cover one;
    one.add(b, segs.data() + b.seg0);
    if (one.n16) work += one.def * (one.work / one.n16);
  }
  return c.def < kSplitTiles && work >= kSplitChunks * c.def ? Tiling{-1, 0} : t;
}

// One block of one segment (a dense product): the same rule with the whole K in one segment.
Tiling single_tiling(const GBlk &b, const GSeg &s, int prec, bool cplx) {
  Cover c;
  c.add(b, &s);
  const int kind = default_kind(b.M, b.N);
  if (c.n16 <= (cplx ? kFewCplx : kFewReal) / 2 && s.K > 32) return {TK_1x1, 4};
  return {c.stay_direct(false) ? c.direct(kind) : c.large(kind, cplx, false), 0,
          c.lean(prec, cplx)};
}

void seal_block(GBlk &b, const GSeg *segs) {
  // the elements of a tile's chunk: up to 64 rows and 16 k, of up to 16 bytes
  const int64_t lim = int64_t(1) << 31;
  int64_t chunks = 0;
  b.wide = kContigA | kContigB;
  for (int i = b.seg0; i < b.seg0 + b.nseg; ++i) {
    const GSeg &s = segs[i];
    chunks += (s.K + 15) / 16;
    if (16 * (64 * s.sam + 16 * s.sak) >= lim || 16 * (64 * s.sbn + 16 * s.sbk) >= lim)
      b.wide |= kWideStrides;
    if (s.sak != 1) b.wide &= ~kContigA;
    if (s.sbk != 1) b.wide &= ~kContigB;
  }
  b.chunks = (int32_t)std::min<int64_t>(chunks, INT32_MAX);
}

int make_tiles(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs,
               std::vector<GTile> &tiles, int *per_xcd, int kind_override, bool allow_rows) {
  struct Item {
    GTile t;
    int64_t cost;
  };
  // the row class is taken when every block is narrow (all of a launch's tiles share a class)
  bool all_narrow = allow_rows;
  for (const GBlk &b : blks)
    if (b.M > 0 && b.N > kRowsN) all_narrow = false;
  int cls = TC_MIXED;
  if (is_lds(kind_override)) cls = TC_LDS;
  else if (kind_override == TK_4x2 && allow_rows) cls = TC_BIG;  // allow_rows: real dtypes only
  else if (kind_override == TK_ROWS ? all_narrow : (kind_override < 0 && all_narrow))
    cls = TC_ROWS;
  // blocks in operand order: first segment's A offset, then its B offset (the scratch
  // vectors keep their capacity between calls: plans of tens of thousands of tiles are made
  // per DMRG bond, and fresh pages cost more than the planning itself)
  thread_local std::vector<int> order;
  order.clear();
  for (size_t bi = 0; bi < blks.size(); ++bi)
    if (blks[bi].M > 0 && blks[bi].N > 0) order.push_back((int)bi);
  auto key = [&](int bi) {
    const GBlk &b = blks[bi];
    return b.nseg > 0 ? std::make_pair(segs[b.seg0].a_off, segs[b.seg0].b_off)
                      : std::make_pair(INT64_MAX, INT64_MAX);
  };
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return key(x) < key(y); });
  thread_local std::vector<Item> items;
  items.clear();
  auto k_of = [&](const GBlk &b) {
    int64_t ksum = 0;
    for (int s = 0; s < b.nseg; ++s) ksum += segs[b.seg0 + s].K;
    return ksum;
  };
  // rows of short K (the MPO steps, K of a few): a wave's four loads and stores take less than
  // reading its tile, block and segment records, so it takes four times the rows
  auto short_rows = [&](const GBlk &b) {
    return b.N <= kShortRowsN && b.M > tile_rows(TK_ROWS) && k_of(b) <= kShortRowsK;
  };
  int64_t rows = 0;
  if (cls == TC_ROWS)
    for (int bi : order)
      if (short_rows(blks[bi])) rows += blks[bi].M;
  for (int bi : order) {
    const GBlk &b = blks[bi];
    int kind;
    if (cls == TC_ROWS)
      kind = TK_ROWS;
    else if (cls == TC_BIG)
      kind = TK_4x2;
    else if (cls == TC_LDS || (kind_override >= 0 && kind_override <= TK_1x2))
      kind = kind_override;
    else
      kind = default_kind(b.M, b.N);
    const int64_t ksum = k_of(b);
    int tr = tile_rows(kind), tc = kind == TK_ROWS ? b.N : tile_cols(kind);
    if (kind == TK_ROWS && rows >= kShortRowsMin && short_rows(b)) tr *= kShortRows;
    for (int m0 = 0; m0 < b.M; m0 += tr)
      for (int n0 = 0; n0 < b.N; n0 += tc)
        items.push_back({GTile{(int32_t)bi, m0, kind == TK_ROWS ? tr : n0, kind},
                         (ksum + 16) * tr * tc});
  }
  // kXcds contiguous ranges of equal tile count (at these sizes a tile's time is mostly its
  // fixed chain of dependent loads, so equal counts balance better than equal flops, and the
  // ranges need no padding beyond the last few tiles)
  // Within a range the tiles go in decreasing cost, ties in list order.  A block's tiles share
  // one cost and sit together, so the range is sorted as runs of equal cost (one per block
  // piece): the same order as sorting the tiles, for hundreds of runs instead of thousands of
  // tiles.
  const size_t per = (items.size() + kXcds - 1) / kXcds;
  const size_t P = per ? (per + kWaves - 1) / kWaves * kWaves : 0;
  tiles.assign(kXcds * P, GTile{-1, 0, 0, 0});
  struct Run {
    size_t at, len;
    int64_t cost;
  };
  thread_local std::vector<Run> runs;
  for (int x = 0; x < kXcds; ++x) {
    const size_t lo = std::min(items.size(), x * per), hi = std::min(items.size(), lo + per);
    runs.clear();
    for (size_t i = lo; i < hi; ++i) {
      if (!runs.empty() && runs.back().cost == items[i].cost) ++runs.back().len;
      else runs.push_back({i, 1, items[i].cost});
    }
    std::stable_sort(runs.begin(), runs.end(),
                     [](const Run &a, const Run &b) { return a.cost > b.cost; });
    size_t o = x * P;
    for (const Run &r : runs)
      for (size_t i = 0; i < r.len; ++i) tiles[o++] = items[r.at + i].t;
  }
  *per_xcd = (int)P;
  return cls;
}

bool has_rows4(const std::vector<GTile> &tiles) {
  for (const GTile &t : tiles)
    if (t.blk >= 0 && t.kind == TK_ROWS && t.n0 > tile_rows(TK_ROWS)) return true;
  return false;
}

bool prefer_splitk(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs,
                   const std::vector<GTile> &tiles, int tile_class) {
  if (tiles.empty() || tile_class == TC_BIG || tile_class == TC_LDS) return false;
  // a tile's work is its block's: summed once per block, then once per tile
  thread_local std::vector<int64_t> bwork;
  bwork.assign(blks.size(), -1);
  int64_t work = 0, n = 0;
  for (const GTile &t : tiles) {
    if (t.blk < 0) continue;
    int64_t &w = bwork[t.blk];
    if (w < 0) {
      const GBlk &b = blks[t.blk];
      w = 0;
      for (int s = 0; s < b.nseg; ++s)
        w += tile_class == TC_ROWS ? segs[b.seg0 + s].K : (segs[b.seg0 + s].K + 15) / 16;
    }
    ++n;
    work += w;
  }
  if (n == 0) return false;
  const double avg = (double)work / (double)n;
  return n < kSplitTiles && avg >= (tile_class == TC_ROWS ? 64.0 : (double)kSplitChunks);
}

}  // namespace cxa
