// Grouped MFMA GEMM: precision dispatch and host-side tile planning (the kernels are in
// gemm_kernels.hpp, instantiated by gemm_fp64.hip, gemm_fp32.hip, gemm_fp32x3.hip and
// gemm_mix.hip).
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

// The choice from the number of 16 x 16 tiles, their mean K in 16-deep chunks and the number of
// 64 x 64 tiles.  A 16 x 16 tile is the finest split of the output, and a wave works through its
// K one MFMA after another, so few tiles leave SIMDs idle: up to kFew of them (two, complex four,
// times the CUs) the four waves of a workgroup share a tile's K, which then also hides their load
// latency.  Above that the LDS tiles read every operand element once per 32 or 64 rows instead
// of once per 16, in contiguous runs.  Measured (us, split 16 x 16 / 32 x 32 LDS):
//   real, product of n = 128: 3.9 / 5.2, 256: 4.9 / 7.3, 512 (1024 tiles): 21.2 / 11.5;
//   complex128, n = 256: 6.4 / 13.9, 384 x 960 x 192 (288 tiles): 27 / 43, 512: 30 / 26;
//   block contractions of a chi = 512 complex128 MPS (about 830 tiles): 12-20 / 31 (the direct
//   32 x 32 tiles 100); two-site .R launch in FP64, chi = 512: 4.8 / 5.8, 2048: 43 / 35.
// 64 x 64 tiles (a quarter of the chunk loads and barriers per flop) pay once they give most CUs
// a tile: n = 700 (121 tiles) 36 us against 23 in FP64, 900 (225 tiles) 44 against 46, 1600 165
// against 177.  They are real-only: a complex 64 x 64 tile's registers leave one or two waves
// per SIMD (n = 1600, complex128: 578 us against 525).
constexpr int64_t kFewReal = 512, kFewCplx = 1024, kMany64 = 192;

// Few tiles (under two per SIMD of a 256-CU device), each with a long K (in chunks of 16).
constexpr int64_t kSplitTiles = 2048, kSplitChunks = 8;

// Whether the default tiles of these (real) blocks have their K split over four waves.
bool splits_by_default(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs) {
  int64_t n = 0, work = 0;
  for (const GBlk &b : blks) {
    if (b.M <= 0 || b.N <= 0) continue;
    const int kind = default_kind(b.M, b.N);
    const int64_t t = (int64_t)((b.M + tile_rows(kind) - 1) / tile_rows(kind)) *
                      ((b.N + tile_cols(kind) - 1) / tile_cols(kind));
    n += t;
    for (int s = b.seg0; s < b.seg0 + b.nseg; ++s) work += t * ((segs[s].K + 15) / 16);
  }
  return n < kSplitTiles && work >= kSplitChunks * n;
}

}  // namespace

Tiling default_tiling(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs, int prec,
                      bool cplx, bool in_order) {
  int64_t n16 = 0, n64 = 0, work = 0, pad64 = 0, pad32 = 0;
  bool narrow = !cplx, lds = true;
  for (const GBlk &b : blks) {
    if (b.M <= 0 || b.N <= 0) continue;
    const int64_t t = tiles_of(b, 16);
    n16 += t;
    n64 += tiles_of(b, 64);
    if (b.N > kRowsN) narrow = false;
    for (int s = b.seg0; s < b.seg0 + b.nseg; ++s) {
      const int64_t chunks = (segs[s].K + 15) / 16;
      work += t * chunks;
      pad64 += 16 * tiles_of(b, 64) * chunks;
      pad32 += 4 * tiles_of(b, 32) * chunks;
      lds = lds && lds_ok(b, segs[s]);
    }
  }
  // K of up to two chunks: an output-bound launch (the MPO steps).  Narrow real blocks stream
  // their rows (their default), others take one wave per tile: the smallest tiles while they
  // are few (4.2 us against 4.5 for 128 blocks of 128 x 10, K = 10)
  if (narrow && prec == CXA_PREC_FP32) return {-1, 0};
  if (work <= 2 * n16) return {narrow || n16 > 4 * kFewReal ? -1 : (int)TK_1x1, 0};
  if (n16 <= (cplx ? kFewCplx : kFewReal)) return {TK_1x1, in_order ? 0 : 4};
  if (!lds || narrow) return {-1, 0};
  if (cplx || n64 < kMany64) return {TK_L32, 0};
  // Ragged blocks: 64x64 tiles that cover much more than 32x32 ones lose it again.  Real blocks
  // of 160 x 160, K = 400, 120 of them (1.44 times the area): direct 32x32 tiles 59 us in FP64 and
  // 34 in FP32, 64x64 79 and 54; of 300 x 300 (the same area), 60 of them: 111 and 60 against 90
  // and 61.
  return {20 * pad64 > 23 * pad32 ? TK_2x2 : TK_L64, 0};
}

Tiling plan_tiling(const std::vector<GBlk> &blks, const std::vector<GSeg> &segs, int prec,
                   bool cplx, bool in_order) {
  const Tiling t = default_tiling(blks, segs, prec, cplx, in_order);
  const bool four_sums = t.split > 0 || (prec == CXA_PREC_FP32 && is_lds(t.kind));
  if (!cplx && t.kind >= 0 && !four_sums && splits_by_default(blks, segs)) return {-1, 0};
  return t;
}

// One block of one segment (a dense product): the same rule with the whole K in one segment.  A
// tall K = 10 product of 36864 x 10 takes 4.5 us in direct tiles and 7.9 in LDS tiles.
Tiling single_tiling(const GBlk &b, const GSeg &s, bool cplx) {
  const int64_t n16 = tiles_of(b, 16);
  if (n16 <= (cplx ? kFewCplx : kFewReal) / 2) return {TK_1x1, s.K > 32 ? 4 : 0};
  if (s.K <= 32 || !lds_ok(b, s)) return {default_kind(b.M, b.N), 0};
  return {!cplx && tiles_of(b, 64) >= kMany64 ? TK_L64 : TK_L32, 0};
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
    int64_t ksum = 0;
    for (int s = 0; s < b.nseg; ++s) ksum += segs[b.seg0 + s].K;
    int tr = tile_rows(kind), tc = kind == TK_ROWS ? b.N : tile_cols(kind);
    // rows of short K (the MPO steps, K of a few): a wave's four loads and stores take less than
    // reading its tile, block and segment records, so it takes four times the rows
    if (kind == TK_ROWS && ksum <= kShortRowsK && b.N <= kShortRowsN && b.M > tr)
      tr *= kShortRows;
    for (int m0 = 0; m0 < b.M; m0 += tr)
      for (int n0 = 0; n0 < b.N; n0 += tc)
        items.push_back({GTile{(int32_t)bi, m0, kind == TK_ROWS ? tr : n0, kind}, (ksum + 16) * tr * tc});
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
