#pragma once

// Grouped GEMM tiles staged through LDS (included by gemm_kernels.hpp's translation units).
//
// A workgroup of four waves owns a BM x BN tile and walks the K dimension of its block's segments
// in chunks of BK.  Each chunk's A rows and B columns are read from global memory once per
// workgroup (one element, or one k-quad of a packed operand, per lane and load), rounded to the
// arithmetic's type and put into LDS k-contiguous, and every wave reads its fragments from there
// as 16-byte vectors: lane (r, g) = (lane % 16, lane / 16) takes the four consecutive k from 4 g of
// row (column) r of every 16, so MFMA j sums k = 4 g + j over the four lane groups, as the direct
// tiles do (the two give the same bits where a direct tile is not split, real FP32 aside).  A row's
// LDS stride is its bytes plus 16, an odd multiple of 16 bytes modulo the 256 bytes of one pass over
// the banks: the 16 rows of a lane group fall on different banks.
//
// Lanes walk whichever index of an operand has the smaller stride (decided per segment), so that
// row-major and column-major operands are both read in contiguous runs; the direct tiles of
// gemm_kernels.hpp fix the lane layout to the fragment's, where each load of a row-major operand
// touches 64 different cache sectors and the address path bounds the launch.
//
// Pipeline: two LDS buffers and one set of staging registers.  While the MFMAs of chunk c run,
// the loads of chunk c + 1 are in flight; the staging registers are written to the other buffer
// after them, and the one barrier per chunk waits for LDS only, not for global loads.
// (Included after the definitions it uses: GBlk / GSeg accessors, load_or_zero, store_c, mma.)

// The element type in LDS of an operand with elements T in an arithmetic of op_t.
template <typename T, typename op_t>
struct LdsElem {
  using g = T;     // as loaded
  using s = op_t;  // as staged
  static __device__ __forceinline__ s conv(g v, op_t) { return (s)v; }
};
template <>
struct LdsElem<cd, double> {
  using g = d2v;
  using s = d2v;
  static __device__ __forceinline__ s conv(g v, double sign) { return s{v.x, sign * v.y}; }
};
template <>
struct LdsElem<cf, float> {
  using g = f2v;
  using s = f2v;
  static __device__ __forceinline__ s conv(g v, float sign) { return s{v.x, sign * v.y}; }
};

// Tile geometry of an LDS kind: 64 x 64 (a wave computes 32 x 32) with 128-byte LDS rows, and
// 32 x 32 (a wave 16 x 16) with 256-byte rows, whose chunks are twice as deep because a chunk
// then carries as many MFMAs per barrier and wave as it can hold in the same staging registers.
template <int KIND, typename ES>
struct LdsGeo {
  static constexpr int BM = KIND == TK_L64 ? 64 : 32, BN = BM;
  static constexpr int BK = (KIND == TK_L64 ? 128 : 256) / (int)sizeof(ES);
  static constexpr int LD = BK + 16 / (int)sizeof(ES);
  static constexpr int NT = 64 * kWaves;
  static constexpr int MI = BM / 32, NI = BN / 32;  // 16 x 16 tiles of a wave (2 x 2 waves)
  static constexpr int KPL = BK / 4;                // k per lane and chunk
  // sets of staging registers: two chunks in flight where one workgroup may have a CU for itself
  static constexpr int D = KIND == TK_L64 ? 1 : 2;
  static constexpr size_t bytes = 2 * (size_t)(BM + BN) * LD * sizeof(ES);
};

// One operand of a tile: this thread's part of the chunk being loaded.  Rows are A's m or B's n.
template <typename T, typename op_t, int BR, int BK, int LD, int NT, bool QUAD>
struct LdsSide {
  using E = LdsElem<T, op_t>;
  using G = typename E::g;
  using ES = typename E::s;
  typedef typename std::conditional<QUAD, T, op_t>::type qe;
  typedef qe q4 __attribute__((ext_vector_type(4)));
  using V = typename std::conditional<QUAD, q4, G>::type;
  static constexpr int N = QUAD ? (BR * BK / 4) / NT : (BR * BK) / NT;
  static_assert(N >= 1 && NT % BR == 0 && NT % BK == 0, "staging layout");
  uint64_t base;    // address of (row 0, k 0) of the next chunk (uniform)
  int64_t adv;      // bytes from chunk to chunk (uniform)
  uint32_t off[N];  // this thread's elements from base; kNoLoad: not read
  int put_at[N];    // where they go in an LDS buffer
  int row0, dr;     // row of its first element within the tile, and the step of the others
  int k0, dk;       // the same for k within the chunk

  // Which elements of every chunk of the tile this thread loads: k runs over the lanes, or the
  // rows do.
  __device__ __forceinline__ void lay(bool along_k, int tid) {
    if (QUAD) along_k = false;
    k0 = along_k ? tid % BK : tid / BR * (QUAD ? 4 : 1);
    row0 = along_k ? tid / BK : tid % BR;
    dr = along_k ? NT / BK : 0;
    dk = along_k ? 0 : NT / BR * (QUAD ? 4 : 1);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      put_at[i] = (row0 + i * dr) * LD + (k0 + i * dk);
      __asm__("" : "+v"(put_at[i]));  // kept, not computed again for every chunk
    }
  }
  // first: the address of (row 0, k 0) of the tile's rows in the segment; sr, sk: the segment's
  // element strides (QUAD: element (row, k) at (k >> 2) * sk + row * 4 + (k & 3)); rows: rows of
  // the tile inside the block; kleft: the segment's K
  __device__ __forceinline__ void enter(uint64_t first, int64_t sr, int64_t sk, int rows,
                                        int kleft) {
    base = first;
    adv = (int64_t)(QUAD ? BK / 4 : BK) * sk * (int64_t)sizeof(G);
    const uint32_t s_r = QUAD ? 4 : (uint32_t)sr, s_k = (uint32_t)sk;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t row = row0 + i * dr, k = k0 + i * dk;
      off[i] = (int)row < rows ? (row * s_r + (QUAD ? k >> 2 : k) * s_k) * (uint32_t)sizeof(G)
                               : kNoLoad;
    }
    if (kleft < BK) last(kleft);
  }
  // the next chunk has only kleft < BK values of k (none after the last segment)
  __device__ __forceinline__ void last(int kleft) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (k0 + i * dk >= kleft) off[i] = kNoLoad;
  }
  __device__ __forceinline__ void load(V (&v)[N]) {
    const __amdgpu_buffer_rsrc_t r = buffer_at(base);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = buffer_get<V>(r, off[i], 0);
    base += adv;
  }
  __device__ __forceinline__ void store(const V (&v)[N], ES *lds, op_t sign) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      ES *d = lds + put_at[i];
      if constexpr (QUAD) {
        struct alignas(16) Four {
          ES e[4];
        };
        *(Four *)__builtin_assume_aligned(d, 16) =
            Four{{E::conv(v[i].x, sign), E::conv(v[i].y, sign), E::conv(v[i].z, sign),
                  E::conv(v[i].w, sign)}};
      } else {
        *d = E::conv(v[i], sign);
      }
    }
  }
};

// Workgroup barrier that orders LDS accesses only: loads from global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One tile.  conj: bit 0 conjugates A, bit 1 conjugates B (complex types).  dslot: the
// dot-product epilogue's slot of this tile (real types; see GemmLaunch::dot_part) or null.
template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int KIND, int PK,
          typename SEGS>
__device__ __forceinline__ void wg_tile_lds(char *smem, const char *__restrict__ Abase,
                                            const char *__restrict__ Bbase,
                                            char *__restrict__ Cbase, const GBlk &blk, SEGS segs,
                                            int m0, int n0, int conj, const double *dotx,
                                            double *dslot, int64_t nslots) {
  constexpr bool F64 = PREC == CXA_PREC_FP64;
  using op_t = typename std::conditional<F64, double, float>::type;
  using acc_t = typename std::conditional<F64, f64x4, f32x4>::type;
  using EA = LdsElem<TA, op_t>;
  using EB = LdsElem<TB, op_t>;
  using ES = typename EA::s;
  static_assert(std::is_same<ES, typename EB::s>::value, "one staged type");
  using Geo = LdsGeo<KIND, ES>;
  constexpr int BM = Geo::BM, BN = Geo::BN, BK = Geo::BK, LD = Geo::LD, NT = Geo::NT;
  constexpr int MI = Geo::MI, NI = Geo::NI, KPL = Geo::KPL, D = Geo::D;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ES *const sa = (ES *)smem, *const sb = sa + 2 * BM * LD;
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(BM, blk.M - m0), nt = min(BN, blk.N - n0);
  // this wave's part of the tile, and how much of it lies inside the block
  const int wm = (wave >> 1) * 16 * MI, wn = (wave & 1) * 16 * NI;
  const int mw = mt - wm, nw = nt - wn;
  using SideA = LdsSide<TA, op_t, BM, BK, LD, NT, (PK & kPackA) != 0>;
  using SideB = LdsSide<TB, op_t, BN, BK, LD, NT, (PK & kPackB) != 0>;
  SideA A;
  SideB B;
  const op_t sga = (conj & 1) ? op_t(-1) : op_t(1), sgb = (conj & 2) ? op_t(-1) : op_t(1);

  int s = 0, kleft = 0;  // the next chunk to load: its segment and the k left there
  bool first = true;
  auto enter = [&]() {  // the first segment from s on that has any k
    while (s < blk.nseg) {
      const GSeg sg = segs(blk.seg0 + s);
      if (sg.K > 0) {
        kleft = sg.K;
        if (first) {  // (the lane layout stays: off its best only where segments differ in order)
          A.lay(sg.sak <= sg.sam, tid);
          B.lay(sg.sbk <= sg.sbn, tid);
          first = false;
        }
        A.enter((uint64_t)(uintptr_t)at<const typename EA::g>(Abase, sg.a_off + m0 * sg.sam),
                sg.sam, sg.sak, mt, kleft);
        B.enter((uint64_t)(uintptr_t)at<const typename EB::g>(Bbase, sg.b_off + n0 * sg.sbn),
                sg.sbn, sg.sbk, nt, kleft);
        return;
      }
      ++s;
    }
    A.last(0);
    B.last(0);
  };
  struct Staged {
    typename SideA::V a[SideA::N];
    typename SideB::V b[SideB::N];
  };
  int ahead = 0;  // chunks loaded and not yet consumed
  auto load = [&](Staged &st) {  // the next chunk, or zeros after the last one
    A.load(st.a);
    B.load(st.b);
  };
  auto next = [&]() {  // after a load
    if (s < blk.nseg) {
      ++ahead;
      kleft -= BK;
      if (kleft <= 0) {
        ++s;
        enter();
      } else if (kleft < BK) {
        A.last(kleft);
        B.last(kleft);
      }
    }
  };
  auto put = [&](const Staged &st, int buf) {
    A.store(st.a, sa + buf * BM * LD, sga);
    B.store(st.b, sb + buf * BN * LD, sgb);
  };
  // Real FP32 sums K in four accumulators, 16-deep part p of the K of a segment in accumulator p % 4,
  // added up in FP64 at the end: the sums of the direct tiles' four-wave split, which these tiles
  // replace, bit for bit where a block has one segment.  (Parts dealt out by halves of a 64-deep
  // chunk leave the accumulators of 32 x 32 tiles up to 64 values of K apart: 1.35e-7 for 1.31e-7
  // off with 30 blocks of 100 x 100, K = 200.)
  constexpr int NACC = std::is_same<ES, float>::value ? 4 : 1;
  acc_t acc[NACC][MI][NI], aci[CPLX ? MI : 1][CPLX ? NI : 1];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
      for (int q = 0; q < NACC; ++q) acc[q][i][j] = acc_t{0, 0, 0, 0};
      if constexpr (CPLX) aci[i][j] = acc_t{0, 0, 0, 0};
    }
  // Fragments of half a chunk.  In every 16 values of k lane group g takes 4 g .. 4 g + 3, the
  // order in which the direct tiles sum K; half of a 16-deep chunk is two of the four.
  constexpr int KH = KPL / 2, KG = KH < 4 ? KH : 4, PARTS = KH / KG;
  constexpr int HALF = BK == 16 ? KG : BK / 2;
  static_assert(BK >= 16, "whole 16-deep parts");
  struct Frag {
    struct alignas(16) Vec {
      ES e[KG];
    };
    Vec a[MI][PARTS], b[NI][PARTS];
  };
  auto fetch = [&](Frag &f, int buf, int half) {
    const ES *pa = sa + buf * BM * LD + (wm + r) * LD + 4 * g + half * HALF;
    const ES *pb = sb + buf * BN * LD + (wn + r) * LD + 4 * g + half * HALF;
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
        f.a[i][q] = *(const typename Frag::Vec *)(pa + 16 * i * LD + 16 * q);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        f.b[j][q] = *(const typename Frag::Vec *)(pb + 16 * j * LD + 16 * q);
    }
  };
  auto multiply = [&](const Frag &f, int half) {  // (half of a pair of chunks: 0 .. 3)
#pragma unroll
    for (int k = 0; k < KH; ++k)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const ES &fa = f.a[i][k / KG].e[k % KG], &fb = f.b[j][k / KG].e[k % KG];
          if constexpr (CPLX) {
            const op_t ar = fa.x, ai = fa.y, br = fb.x, bi = fb.y;
            acc[0][i][j] = mma(ar, br, acc[0][i][j]);
            aci[i][j] = mma(ar, bi, aci[i][j]);
            acc[0][i][j] = mma(-ai, bi, acc[0][i][j]);
            aci[i][j] = mma(ai, br, aci[i][j]);
          } else {
            const int q = (PARTS * half + k / KG) % NACC;
            acc[q][i][j] = mma(fa, fb, acc[q][i][j]);
          }
        }
  };

  // The K loop.  Chunk c is consumed from LDS buffer c % 2 while chunks c + 1 .. c + D are loaded
  // or in flight.  Fragments are fetched half a chunk ahead of their MFMAs; the one barrier of a
  // chunk stands between its halves: by then every wave has fetched all of this chunk and put
  // its part of the next one, whose first half is then fetched under the second half's MFMAs.
  // The steady part has one exit per U chunks (the last of them may then be empty ones, which
  // are loaded but never consumed): with an exit after each, the accumulators would be copied,
  // after waiting for the MFMAs, on every chunk.  A wave whose part lies outside the block loads
  // and waits like the others but computes nothing.
  constexpr int U = D > 2 ? D : 2;
  constexpr int kMfmas = MI * NI * KH * (CPLX ? 4 : 1), kMem = SideA::N + SideB::N;
  constexpr int kPer = (kMem + kMfmas - 1) / kMfmas;
  Staged st[D];
  Frag f0, f1;
  const bool active = mw > 0 && nw > 0;
  enter();
  if (s < blk.nseg) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(st[d]);
      next();
    }
    put(st[0], 0);
    load(st[0]);
    next();
    lds_barrier();
    if (active) fetch(f0, 0, 0);
    while (s < blk.nseg) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (active) {
          fetch(f1, u & 1, 1);
          put(st[(u + 1) % D], (u + 1) & 1);
          load(st[(u + 1) % D]);
          multiply(f0, 2 * (u & 1));
          // the put's and the load's instructions between the MFMAs, which each keep the
          // matrix pipe busy for 32 or 64 cycles
#pragma unroll
          for (int q = 0; q < kMfmas; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // an MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);     // vector arithmetic
            __builtin_amdgcn_sched_group_barrier(0x200, kPer, 0);  // LDS writes
            __builtin_amdgcn_sched_group_barrier(0x020, kPer, 0);  // global loads
          }
          __builtin_amdgcn_sched_barrier(0);
        } else {
          put(st[(u + 1) % D], (u + 1) & 1);
          load(st[(u + 1) % D]);
        }
        lds_barrier();
        if (active) {
          fetch(f0, (u + 1) & 1, 0);
          __builtin_amdgcn_sched_barrier(0);
          multiply(f1, 2 * (u & 1) + 1);
        }
        next();
        --ahead;
      }
    }
#pragma unroll
    for (int u = 0; u <= D; ++u) {  // the last chunks, all loaded: at most D + 1
      if (ahead <= 0) break;
      const bool more = u < D && ahead > 1;
      if (active) fetch(f1, u & 1, 1);
      if (more) put(st[(u + 1) % D], (u + 1) & 1);
      if (active) multiply(f0, 2 * (u & 1));
      lds_barrier();
      if (active) {
        if (more) fetch(f0, (u + 1) & 1, 0);
        multiply(f1, 2 * (u & 1) + 1);
      }
      --ahead;
    }
  }

  double cx = 0.0, xx = 0.0;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * i + acc_row(F64, g, v), col = 16 * jj + r;
        if (row >= mw || col >= nw) continue;
        const int64_t e = (int64_t)(m0 + wm + row) * blk.ldc + (n0 + wn + col) * blk.csn;
        if constexpr (CPLX) {
          store_cplx<op_t>(at<typename EA::g>(Cbase, blk.c_off) + e, (double)acc[0][i][jj][v],
                           (double)aci[i][jj][v], blk);
        } else {
          double val = (double)acc[0][i][jj][v];
#pragma unroll
          for (int q = 1; q < NACC; ++q) val += (double)acc[q][i][jj][v];
          store_c(at<TC>(Cbase, blk.c_off) + e, val, blk);
          if (dslot) {
            const double xe = dotx[blk.c_off + e];
            cx += val * xe;
            xx += xe * xe;
          }
        }
      }
  if constexpr (!CPLX) {
    if (dslot) {  // wave partials, summed in wave order
      cx = wave_sum(cx);
      xx = wave_sum(xx);
      double *red = (double *)smem;
      __syncthreads();  // the buffers are free
      if (lane == 0) {
        red[wave] = cx;
        red[kWaves + wave] = xx;
      }
      __syncthreads();
      if (tid == 0) {
        double a = red[0], b = red[kWaves];
#pragma unroll
        for (int q = 1; q < kWaves; ++q) {
          a += red[q];
          b += red[kWaves + q];
        }
        dslot[0] = a;
        dslot[nslots] = b;
      }
    }
  }
}

template <int PREC, typename TA, bool CPLX>
using lds_elem_t = typename LdsElem<TA, typename std::conditional<PREC == CXA_PREC_FP64, double,
                                                                   float>::type>::s;

// grouped launch: one workgroup per tile of the list
template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int KIND, int PK>
__global__ __launch_bounds__(64 * kWaves, 2) void k_grouped_lds(
    const GTile *__restrict__ tiles, int per_xcd, const GBlk *__restrict__ blks,
    const GSeg *__restrict__ segs, const char *A, const char *B, char *C, int conj,
    const double *dotx, double *dotp) {
  __shared__ alignas(16) char smem[LdsGeo<KIND, lds_elem_t<PREC, TA, CPLX>>::bytes];
  const int x = blockIdx.x % kXcds;
  const GTile *range = tiles + (int64_t)x * per_xcd;
  const int stride = gridDim.x / kXcds;
  for (int t = blockIdx.x / kXcds; t < per_xcd; t += stride) {
    const GTile tl = range[t];
    double *dslot = dotp ? dotp + (int64_t)x * per_xcd + t : nullptr;
    if (tl.blk < 0) {  // padding (uniform over the workgroup)
      if (dslot && threadIdx.x == 0) dslot[0] = dslot[(int64_t)kXcds * per_xcd] = 0.0;
      continue;
    }
    const GBlk blk = blks[tl.blk];
    wg_tile_lds<PREC, TA, TB, TC, CPLX, KIND, PK>(smem, A, B, C, blk, SegArray{segs}, tl.m0,
                                                      tl.n0, conj, dotx, dslot,
                                                      (int64_t)kXcds * per_xcd);
    __syncthreads();  // the next tile reuses the buffers
  }
}

// Single block with one segment, tiles from the workgroup index.  Workgroup w runs on XCD
// w % kXcds: each XCD takes a contiguous range of an order that walks bands of eight tile rows
// column by column, so that the tiles in flight on an XCD share their A rows and B columns in
// its L2.
template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int KIND>
__global__ __launch_bounds__(64 * kWaves, 2) void k_single_lds(GBlk blk, GSeg seg, int tiles_m,
                                                            int tiles_n, int ntiles,
                                                            const char *A, const char *B,
                                                            char *C, int conj) {
  using Geo = LdsGeo<KIND, lds_elem_t<PREC, TA, CPLX>>;
  __shared__ alignas(16) char smem[Geo::bytes];
  const int per = (ntiles + kXcds - 1) / kXcds;
  const int t = (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
  if ((int)(blockIdx.x / kXcds) >= per || t >= ntiles) return;  // uniform over the workgroup
  const int band = t / (8 * tiles_n), in = t - band * 8 * tiles_n;
  const int rows = min(8, tiles_m - 8 * band);
  const int tn = in / rows, tm = 8 * band + (in - tn * rows);
  wg_tile_lds<PREC, TA, TB, TC, CPLX, KIND, 0>(smem, A, B, C, blk, SegOne{seg}, tm * Geo::BM,
                                                   tn * Geo::BN, conj, nullptr, nullptr, 0);
}
