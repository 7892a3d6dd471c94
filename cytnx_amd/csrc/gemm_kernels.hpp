#pragma once

// Grouped, persistent MFMA GEMM for gfx950.
//
// One launch runs a list of tiles drawn from any number of independent output blocks.  Three
// execution shapes share the task format:
//
//  * MFMA wave tiles: one wave owns a 16*MI x 16*NI tile and walks the K dimension of every
//    segment of its block in chunks of 16 with MFMA 16x16x4 instructions.  Fragments are loaded
//    straight from global memory (the operands are L2/MALL-resident at these sizes) with the k
//    index assigned so that each lane reads 4 consecutive k values: MFMA number j of a chunk
//    takes k = k0 + 4*(lane/16) + j for both A (row lane%16) and B (column lane%16).  The MFMA
//    sums over its 4 k slots, so any assignment identical for A and B is exact; this one makes
//    row-major A loads 32-byte contiguous per lane and B loads 128-byte contiguous per 16 lanes.
//  * Workgroup split-K: the four waves of a workgroup take the same MFMA tile and interleave its
//    K chunks; the partial accumulators meet in LDS and are summed in fixed wave order, so the
//    result is deterministic.  Used when a launch has few tiles with long K.
//  * Row streaming: for blocks with N <= 8 (the MPO steps, K and N of a few MPO states) each
//    lane owns one output row and accumulates in FP64 registers; loads of A are coalesced across
//    lanes, B is a broadcast, C rows are contiguous.
//
// Precision modes: FP64 (v_mfma_f64_16x16x4_f64), FP32 (v_mfma_f32_16x16x4_f32, operands
// rounded to FP32), FP32X3 (FP64 operands split x = hi + lo in FP32; hi*hi + hi*lo + lo*hi on
// FP32 MFMA, the two cross terms in their own accumulator, combined in FP64 at the end).
//
// This header holds the kernel templates; the translation units gemm_fp64.hip, gemm_fp32.hip,
// gemm_fp32_a64.hip, gemm_fp32x3.hip and gemm_mix.hip each instantiate one precision family
// (so they compile in parallel), and gemm.hip holds the dispatch and the host-side tile
// planning.  Define
// CXA_GEMM_TU (a distinct token per translation unit) before including it: each unit carries
// its own zero cell.
#include <algorithm>
#include <type_traits>

#include "cxa_common.hpp"
#include "gemm.hpp"

#ifndef CXA_GEMM_TU
#error "define CXA_GEMM_TU before including gemm_kernels.hpp"
#endif
#define CXA_GEMM_CAT2(a, b) a##b
#define CXA_GEMM_CAT(a, b) CXA_GEMM_CAT2(a, b)
#define CXA_GEMM_ZERO_CELL CXA_GEMM_CAT(gemm_zero_cell_, CXA_GEMM_TU)

namespace cxa {


// Thirty-two zero bytes in device memory (zero-initialised, never written).  An operand element
// outside its block is read from here (the address is selected, not the value), so fragment
// loads need no branch and no wait at the load site; the MFMA that consumes them sees exact
// zeros.  External linkage keeps the compiler from folding these loads to constants, which
// would turn the selects back into branches around the loads.
__device__ __align__(32) double CXA_GEMM_ZERO_CELL[4];

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct alignas(16) cd {
  double re, im;
};
struct alignas(8) cf {
  float re, im;
};

constexpr int kWaves = 4;

// Operand layouts of a launch (template bit set PK): B, A k4-packed (GemmLaunch::b_k4 / a_k4),
// mix outputs written k4-packed (GemmLaunch::c_k4).
constexpr int kPackB = 1, kPackA = 2, kPackC = 4;

__device__ __forceinline__ f64x4 mma64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f64x4 mma(double a, double b, f64x4 c) { return mma64(a, b, c); }
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return mma32(a, b, c); }

// Accumulator row held in register v by lane group g = lane/16 (column = lane%16), measured on
// gfx950: v_mfma_f64_16x16x4_f64 interleaves rows (g + 4v), v_mfma_f32_16x16x4_f32 blocks
// them (4g + v).
__device__ __forceinline__ int acc_row(bool f64, int g, int v) {
  return f64 ? g + 4 * v : 4 * g + v;
}

// Wait for every outstanding vector-memory load (s_waitcnt vmcnt(0); expcnt and lgkmcnt left
// at their maxima).  Issued where a load pipeline ends, when every load it issued has already
// been consumed, so it costs nothing at run time; it tells the compiler's wait analysis that no
// fragment load is still in flight, which it cannot prove by itself across the ring's
// conditional prefetches, and which it would otherwise answer with waits on the next tile's
// first loads.
__device__ __forceinline__ void drain_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Operand and result pointers live in the global address space: loads through them are
// global_load (counted by vmcnt alone), where generic pointers would give flat loads that also
// hold lgkmcnt, so every wait for a scalar descriptor load would drain the operand pipeline.
template <typename T>
using gptr = __attribute__((address_space(1))) T *;

// base + element offset computed on integers: a batched call passes absolute addresses (in
// elements) as offsets from a null base, which pointer arithmetic may not express.  Offsets in
// elements let one task list serve FP64 and FP32 copies of the same block layout.
template <typename T, typename B>
__device__ __forceinline__ gptr<T> at(B *base, int64_t elem_off) {
  return (gptr<T>)(reinterpret_cast<uintptr_t>(base) +
                   (uintptr_t)elem_off * (uintptr_t)sizeof(T));
}

template <typename T>
__device__ __forceinline__ gptr<const T> zero_cell() {
  static_assert(sizeof(T) <= sizeof(CXA_GEMM_ZERO_CELL), "zero cell too small");
  return (gptr<const T>)(&CXA_GEMM_ZERO_CELL[0]);
}

// *p when `valid`, else 0, as one unconditional load.  The selected address passes through an
// empty asm operand so that the compiler cannot split the load into "valid ? *p : 0" (a branch
// around the load, which costs the load pipeline its in-order wait counts).
template <typename T>
__device__ __forceinline__ T load_or_zero(gptr<const T> p, bool valid) {
  uint64_t a = reinterpret_cast<uint64_t>(valid ? p : zero_cell<T>());
  __asm__("" : "+v"(a));
  return *reinterpret_cast<gptr<const T>>(a);
}

// Loads through a buffer descriptor: 32-bit offsets per lane from a scalar base plus a scalar
// offset, so a chunk's addresses cost no vector arithmetic, and an offset of kNoLoad reads as
// zero without a memory access (elements outside the block or past the segment's K).  The
// elements of a tile's chunk lie within 2^31 bytes of the base (checked on the host: seal_block,
// lds_ok), and so do the scalar offsets, so no sum wraps.
constexpr uint32_t kNoLoad = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_at(uint64_t base) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)kNoLoad, 0x00027000);
}

template <typename V>
__device__ __forceinline__ V buffer_get(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  typedef int i2 __attribute__((ext_vector_type(2)));
  typedef int i4 __attribute__((ext_vector_type(4)));
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
  } else if constexpr (sizeof(V) == 8) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
  } else if constexpr (sizeof(V) == 16) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
  } else {
    static_assert(sizeof(V) == 32, "load width");
    struct Two {
      i4 a, b;
    };
    return __builtin_bit_cast(
        V, Two{__builtin_bit_cast(i4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0)),
               __builtin_bit_cast(
                   i4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff + 16, 0))});
  }
}

struct SegArray {
  const GSeg *p;
  __device__ __forceinline__ GSeg operator()(int i) const { return p[i]; }
};
struct SegOne {
  GSeg s;
  __device__ __forceinline__ GSeg operator()(int) const { return s; }
};

// ---------------------------------------------------------------------------------------
// real MFMA tiles
// ---------------------------------------------------------------------------------------
template <int PREC, int MI, int NI>
struct RealAcc {
  static constexpr bool F64 = (PREC == CXA_PREC_FP64);
  using acc_t = typename std::conditional<F64, f64x4, f32x4>::type;
  // Chunks in flight per wave: enough loads outstanding to cover an L2/MALL round trip with a
  // tile's whole K range at the usual block sizes (K <= 64 is one round trip), within a register
  // budget that keeps several waves per SIMD.
  static constexpr int depth =
      (MI * NI >= 8 || (PREC != CXA_PREC_FP32 && MI * NI >= 4)) ? 2 : F64 && MI * NI == 2 ? 3 : 4;
  acc_t hi[MI][NI];
  acc_t lo[MI][NI];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        hi[i][j] = acc_t{0, 0, 0, 0};
        lo[i][j] = acc_t{0, 0, 0, 0};
      }
  }
  __device__ __forceinline__ double get(int i, int j, int v) const {
    double x = (double)hi[i][j][v];
    if constexpr (PREC == CXA_PREC_FP32X3) x += (double)lo[i][j][v];
    return x;
  }
};

// Operand fragments of one 16-deep K chunk (per lane: 4 k values per 16-row / 16-column
// group), held as loaded (operand dtype).  Rounding to FP32 and the FP32X3 hi/lo split happen
// when the chunk is consumed, so the loads of the chunks in flight are not waited for early.
template <typename TA, typename TB, int MI, int NI>
struct Frag {
  TA a[MI][4];
  TB b[NI][4];
};

// `live` is false once the cursor has passed the end of its K range: every element then reads
// the zero cell (the pipelines load only chunks inside the range, so this is a guard).  With
// kPackA / kPackB in PK the A / B operand is k4-packed (element (m, k) at (k >> 2) * sak +
// m * 4 + (k & 3), element (k, n) at (k >> 2) * sbk + n * 4 + (k & 3) from the segment's
// origin, whole quads): the 4 k of a lane's row or column are one vector load.
template <typename TA, typename TB, int MI, int NI, int PK = 0>
__device__ __forceinline__ void load_frag(Frag<TA, TB, MI, NI> &f, gptr<const TA> Ap,
                                          gptr<const TB> Bp, const GSeg &sg, int k0, int mt,
                                          int nt, int r, int g, bool live) {
  if constexpr ((PK & kPackA) != 0) {
    typedef TA ta4 __attribute__((ext_vector_type(4)));
    const bool quad = live && k0 + 4 * g < sg.K;
    const int64_t qoff = (int64_t)((k0 >> 2) + g) * sg.sak;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = 16 * i + r;
      const ta4 v = load_or_zero<ta4>((gptr<const ta4>)(Ap + (qoff + (int64_t)row * 4)),
                                      quad && row < mt);
      f.a[i][0] = v.x;
      f.a[i][1] = v.y;
      f.a[i][2] = v.z;
      f.a[i][3] = v.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = 16 * i + r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + 4 * g + j;
        f.a[i][j] = load_or_zero<TA>(Ap + ((int64_t)row * sg.sam + (int64_t)k * sg.sak),
                                     live && row < mt && k < sg.K);
      }
    }
  }
  if constexpr ((PK & kPackB) != 0) {
    typedef TB tb4 __attribute__((ext_vector_type(4)));
    const bool quad = live && k0 + 4 * g < sg.K;  // quads past K are not stored
    const int64_t qoff = (int64_t)((k0 >> 2) + g) * sg.sbk;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int col = 16 * i + r;
      const tb4 v = load_or_zero<tb4>((gptr<const tb4>)(Bp + (qoff + (int64_t)col * 4)),
                                      quad && col < nt);
      f.b[i][0] = v.x;
      f.b[i][1] = v.y;
      f.b[i][2] = v.z;
      f.b[i][3] = v.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int col = 16 * i + r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + 4 * g + j;
        f.b[i][j] = load_or_zero<TB>(Bp + ((int64_t)k * sg.sbk + (int64_t)col * sg.sbn),
                                     live && col < nt && k < sg.K);
      }
    }
  }
}

template <int PREC, typename TA, typename TB, int MI, int NI>
__device__ __forceinline__ void mma_frag(RealAcc<PREC, MI, NI> &acc,
                                         const Frag<TA, TB, MI, NI> &f) {
  constexpr bool X3 = (PREC == CXA_PREC_FP32X3);
  using op_t = typename std::conditional<PREC == CXA_PREC_FP64, double, float>::type;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    op_t a[MI], b[NI];
    float alo[MI], blo[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      a[i] = (op_t)f.a[i][j];
      if constexpr (X3) alo[i] = (float)((double)f.a[i][j] - (double)a[i]);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      b[i] = (op_t)f.b[i][j];
      if constexpr (X3) blo[i] = (float)((double)f.b[i][j] - (double)b[i]);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int jj = 0; jj < NI; ++jj) {
        if constexpr (PREC == CXA_PREC_FP64) {
          acc.hi[i][jj] = mma64(a[i], b[jj], acc.hi[i][jj]);
        } else {
          acc.hi[i][jj] = mma32(a[i], b[jj], acc.hi[i][jj]);
          if constexpr (X3) {
            acc.lo[i][jj] = mma32(a[i], blo[jj], acc.lo[i][jj]);
            acc.lo[i][jj] = mma32(alo[i], b[jj], acc.lo[i][jj]);
          }
        }
      }
  }
}

// Complex tiles (C128 on FP64 MFMA, C64 on FP32 MFMA): four real products per step.  sa, sb: -1
// conjugates A, B as they are consumed (the adjoint contractions).
template <typename op_t, int MI, int NI>
struct CplxAcc {
  static constexpr bool F64 = std::is_same<op_t, double>::value;
  using acc_t = typename std::conditional<F64, f64x4, f32x4>::type;
  static constexpr int depth = MI * NI == 1 ? (F64 ? 3 : 4) : (MI * NI == 2 || !F64 ? 2 : 1);
  acc_t re[MI][NI], im[MI][NI];
  op_t sa, sb;
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) re[i][j] = im[i][j] = acc_t{0, 0, 0, 0};
  }
};

template <typename op_t, typename T, int MI, int NI>
__device__ __forceinline__ void mma_frag(CplxAcc<op_t, MI, NI> &acc, const Frag<T, T, MI, NI> &f) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const op_t ar = f.a[i][k].x, ai = acc.sa * f.a[i][k].y;
        const op_t br = f.b[j][k].x, bi = acc.sb * f.b[j][k].y;
        acc.re[i][j] = mma(ar, br, acc.re[i][j]);
        acc.im[i][j] = mma(ar, bi, acc.im[i][j]);
        acc.re[i][j] = mma(-ai, bi, acc.re[i][j]);
        acc.im[i][j] = mma(ai, br, acc.im[i][j]);
      }
}

// Walks the 16-deep K chunks c of a block's concatenated segments with c % nslices == slice,
// in order; all fields are wave-uniform.
template <typename TA, typename TB, typename SEGS>
struct ChunkCursor {
  SEGS segs;
  int seg0, nseg, nslices, m0, n0;
  int s, k0;  // current segment and chunk start within it
  GSeg sg;
  gptr<const TA> Ap;
  gptr<const TB> Bp;
  __device__ __forceinline__ void enter(const char *Abase, const char *Bbase) {
    sg = segs(seg0 + s);
    Ap = at<const TA>(Abase, sg.a_off) + (int64_t)m0 * sg.sam;
    Bp = at<const TB>(Bbase, sg.b_off) + (int64_t)n0 * sg.sbn;
  }
  __device__ __forceinline__ bool live() const { return s < nseg; }
  template <int MI, int NI, int PK>
  __device__ __forceinline__ void load(Frag<TA, TB, MI, NI> &f, int mt, int nt, int r,
                                       int g) const {
    load_frag<TA, TB, MI, NI, PK>(f, Ap, Bp, sg, k0, mt, nt, r, g, live());
  }
  // skip `nchunk` chunks forward (crossing segment ends); past the last segment the cursor
  // stays exhausted (live() false)
  __device__ __forceinline__ void skip(int nchunk, const char *Abase, const char *Bbase) {
    k0 += 16 * nchunk;
    bool moved = false;
    while (s < nseg) {
      const int span = 16 * ((sg.K + 15) >> 4);
      if (k0 < span) break;
      k0 -= span;
      ++s;
      if (s < nseg) {
        sg = segs(seg0 + s);
        moved = true;
      }
    }
    if (moved && s < nseg) enter(Abase, Bbase);
  }
};

// One operand's part of a wave's chunks: NR groups of 16 rows (A's m or B's n), one row per lane
// and group, 4 consecutive k.
// WIDE: k is the contiguous index, and a lane's 4 k come in one or two 16-byte loads (which need
// no more than 4-byte alignment) where 4 loads would each touch the cache lines of all 16 rows.
// The last, partial chunk of a segment goes by elements: what lies past K may be anything.
template <typename T, int NR, bool QUAD, bool WIDE>
struct ChunkSide {
  using qe = typename std::conditional<QUAD || WIDE, T, float>::type;  // (real operands)
  typedef qe t4 __attribute__((ext_vector_type(4)));
  uint64_t base;     // address of (row 0, k 0) of the next chunk (uniform)
  int64_t adv;       // bytes from chunk to chunk (uniform)
  uint32_t sk;       // bytes from k to k + 1 (uniform; QUAD: not used)
  uint32_t off[NR];  // this lane's first element of each group; kNoLoad: outside the block
  // first: the address of (row 0, k 0); sr, st: the segment's strides along the rows and k (QUAD:
  // from quad to quad); step: chunks from one of the wave's chunks to its next
  __device__ __forceinline__ void enter(uint64_t first, int64_t sr, int64_t st, int rows,
                                        int step, int r, int g) {
    base = first;
    adv = (int64_t)(QUAD ? 4 : 16) * step * st * (int64_t)sizeof(T);
    sk = (uint32_t)st * (uint32_t)sizeof(T);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const uint32_t row = 16 * i + r;
      const uint32_t e = row * (QUAD ? 4u : (uint32_t)sr) +
                         (uint32_t)(QUAD ? g : 4 * g) * (uint32_t)st;
      off[i] = (int)row < rows ? e * (uint32_t)sizeof(T) : kNoLoad;
    }
  }
  // kleft: k left in the segment (QUAD: whole quads, zero past K)
  __device__ __forceinline__ void load(T (&v)[NR][4], int kleft, int g) const {
    const __amdgpu_buffer_rsrc_t rs = buffer_at(base);
    if constexpr (QUAD) {
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const t4 x = buffer_get<t4>(rs, 4 * g < kleft ? off[i] : kNoLoad, 0);
        v[i][0] = x.x;
        v[i][1] = x.y;
        v[i][2] = x.z;
        v[i][3] = x.w;
      }
    } else {
      if constexpr (WIDE) {
        if (kleft >= 16) {  // (uniform)
#pragma unroll
          for (int i = 0; i < NR; ++i) {
            const t4 x = buffer_get<t4>(rs, off[i], 0);
            v[i][0] = x.x;
            v[i][1] = x.y;
            v[i][2] = x.z;
            v[i][3] = x.w;
          }
          return;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < NR; ++i)
          v[i][j] = buffer_get<T>(rs, 4 * g + j < kleft ? off[i] : kNoLoad, j * sk);
    }
  }
};

// The chunks of a wave in order, like ChunkCursor, for tiles whose addresses fit 32-bit offsets.
// Past the last chunk every load reads zeros.  ONE: the block has a single segment.
// W: sides read with wide loads (bit 0 A, bit 1 B).
template <typename TA, typename TB, int MI, int NI, int PK, bool ONE, int W, typename SEGS>
struct ChunkStream {
  SEGS segs;
  int seg0, nseg, step, m0, n0, mt, nt, r, g;
  int s, k0, K;  // current segment, chunk start within it, and its extent
  GSeg nx;       // the next segment, read while this one's chunks run
  ChunkSide<TA, MI, (PK & kPackA) != 0, (W & 1) != 0> a;
  ChunkSide<TB, NI, (PK & kPackB) != 0, (W & 2) != 0> b;
  // to the chunk `first` chunks from the start (nseg > 0)
  __device__ __forceinline__ void start(int first, const char *Abase, const char *Bbase) {
    s = 0;
    k0 = 16 * first;
    nx = segs(seg0);
    enter(Abase, Bbase);
  }
  // into segment s, whose descriptor is nx, k0 from its start, stepping over whole segments
  __device__ __forceinline__ void enter(const char *Abase, const char *Bbase) {
    GSeg sg = nx;
    if constexpr (!ONE) {
      while (true) {
        nx = segs(seg0 + min(s + 1, nseg - 1));
        const int span = 16 * ((sg.K + 15) >> 4);
        if (k0 < span) break;
        k0 -= span;
        if (++s >= nseg) {
          K = k0 = 0;
          return;
        }
        sg = nx;
      }
    }
    K = sg.K;
    a.enter((uint64_t)(uintptr_t)(at<const TA>(Abase, sg.a_off) + (int64_t)m0 * stride_a(sg)),
            sg.sam, sg.sak, mt, step, r, g);
    b.enter((uint64_t)(uintptr_t)(at<const TB>(Bbase, sg.b_off) + (int64_t)n0 * stride_b(sg)),
            sg.sbn, sg.sbk, nt, step, r, g);
    a.base += (int64_t)((PK & kPackA) ? k0 >> 2 : k0) * sg.sak * (int64_t)sizeof(TA);
    b.base += (int64_t)((PK & kPackB) ? k0 >> 2 : k0) * sg.sbk * (int64_t)sizeof(TB);
  }
  static __device__ __forceinline__ int64_t stride_a(const GSeg &sg) {
    return (PK & kPackA) ? 4 : sg.sam;
  }
  static __device__ __forceinline__ int64_t stride_b(const GSeg &sg) {
    return (PK & kPackB) ? 4 : sg.sbn;
  }
  __device__ __forceinline__ void load(Frag<TA, TB, MI, NI> &f) const {
    a.load(f.a, K - k0, g);
    b.load(f.b, K - k0, g);
  }
  __device__ __forceinline__ void next(const char *Abase, const char *Bbase) {
    k0 += 16 * step;
    a.base += a.adv;
    b.base += b.adv;
    if constexpr (!ONE) {
      if (k0 >= K) {
        k0 -= 16 * ((K + 15) >> 4);
        if (++s < nseg)
          enter(Abase, Bbase);
        else
          s = nseg, K = k0 = 0;
      }
    }
  }
};

// Run `total` > 0 chunks through a ring of D fragment sets, D of them in flight: load(d) fetches
// the next chunk into set d and next() goes on to the one after it, use(d) consumes set d.  No
// load of the ring is conditional: the compiler's wait for a set then leaves the D - 1 newer ones
// in flight, where a load under a condition would make it wait for all of them at every chunk.
// TAIL: ranges shorter than D and the last, partial round take only their own loads, in code of
// their own; without it (next() is long) ranges of one chunk do, and the loads past the last
// chunk, fewer than D chunks, read zeros without a memory access.
template <int D, bool TAIL, typename LOAD, typename NEXT, typename USE>
__device__ __forceinline__ void run_chunks(int total, LOAD load, NEXT next, USE use) {
  constexpr int SHORT = TAIL ? D - 1 : 1;
  if (total <= SHORT) {
#pragma unroll
    for (int d = 0; d < SHORT; ++d)
      if (d < total) {
        load(d);
        if (d + 1 < SHORT) next();
      }
#pragma unroll
    for (int d = 0; d < SHORT; ++d)
      if (d < total) use(d);
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(d);
      next();
    }
    for (; total > (TAIL ? 2 * D - 1 : D); total -= D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        use(d);
        load(d);
        next();
      }
    }
    if constexpr (TAIL) {  // D .. 2 D - 1 chunks left, D of them loaded
#pragma unroll
      for (int d = 0; d < D; ++d) {
        use(d);
        if (d < total - D) {
          load(d);
          next();
        }
      }
      total -= D;
    }
#pragma unroll
    for (int d = 0; d < (TAIL ? D - 1 : D); ++d)
      if (d < total) use(d);
  }
  drain_loads();
}

// Accumulate the chunks c with c % nslices == slice of the block's concatenated K range.
// A ring of ACC::depth fragment sets keeps that many chunks' loads in flight across the
// whole range (segment boundaries included): the MFMAs of chunk c issue while chunks
// c+1 .. c+depth-1 are still arriving, and chunk c+depth is loaded into the set just consumed.
// LEAN: see TC_LEAN; no split of K (nslices 1) and no kWideStrides.
template <typename TA, typename TB, int MI, int NI, int PK, bool LEAN = false, typename ACC,
          typename SEGS>
__device__ __forceinline__ void mfma_accumulate(ACC &acc,
                                                const char *__restrict__ Abase,
                                                const char *__restrict__ Bbase, const GBlk &blk,
                                                SEGS segs, int m0, int n0, int lane, int slice,
                                                int nslices) {
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16 * MI, blk.M - m0);
  const int nt = min(16 * NI, blk.N - n0);
  const int total = (blk.chunks - slice + nslices - 1) / nslices;
  if (total <= 0) return;
  if (!LEAN && (blk.wide & kWideStrides)) {
    ChunkCursor<TA, TB, SEGS> cur{segs, blk.seg0, blk.nseg, nslices, m0, n0, 0, 0};
    cur.enter(Abase, Bbase);
    cur.skip(slice, Abase, Bbase);  // also steps over empty leading segments
    for (int c = 0; c < total; ++c) {
      Frag<TA, TB, MI, NI> f;
      cur.template load<MI, NI, PK>(f, mt, nt, r, g);
      cur.skip(nslices, Abase, Bbase);
      mma_frag(acc, f);
    }
    drain_loads();
    return;
  }
  auto run = [&](auto w) {
    if constexpr (LEAN) {
      const int nseg = std::is_same<SEGS, SegOne>::value ? 1 : blk.nseg;  // (total > 0)
      for (int s = 0; s < nseg; ++s) {
        const GSeg sg = segs(blk.seg0 + s);
        ChunkSide<TA, MI, false, (decltype(w)::value & 1) != 0> a;
        ChunkSide<TB, NI, false, (decltype(w)::value & 2) != 0> b;
        a.enter((uint64_t)(uintptr_t)(at<const TA>(Abase, sg.a_off) + (int64_t)m0 * sg.sam), sg.sam,
                sg.sak, mt, 1, r, g);
        b.enter((uint64_t)(uintptr_t)(at<const TB>(Bbase, sg.b_off) + (int64_t)n0 * sg.sbn), sg.sbn,
                sg.sbk, nt, 1, r, g);
        for (int k0 = 0; k0 < sg.K; k0 += 16) {
          Frag<TA, TB, MI, NI> f;
          a.load(f.a, sg.K - k0, g);
          b.load(f.b, sg.K - k0, g);
          a.base += a.adv;
          b.base += b.adv;
          mma_frag(acc, f);
        }
      }
      drain_loads();
    } else {
      ChunkStream<TA, TB, MI, NI, PK, std::is_same<SEGS, SegOne>::value, decltype(w)::value, SEGS>
          st{segs, blk.seg0, blk.nseg, nslices, m0, n0, mt, nt, r, g};
      st.start(slice, Abase, Bbase);
      constexpr int D = ACC::depth;
      Frag<TA, TB, MI, NI> f[D];
      run_chunks<D, std::is_same<SEGS, SegOne>::value>(
          total, [&](int d) { st.load(f[d]); }, [&]() { st.next(Abase, Bbase); },
          [&](int d) { mma_frag(acc, f[d]); });
    }
  };
  // The loads' widths are fixed per pipeline (a choice between them at every chunk would cost the
  // exact waits); unpacked real operands only, one side at a time.
  if constexpr (PK == 0 && std::is_arithmetic<TA>::value) {
    if (blk.wide & kContigA)
      run(std::integral_constant<int, 1>{});
    else if (blk.wide & kContigB)
      run(std::integral_constant<int, 2>{});
    else
      run(std::integral_constant<int, 0>{});
  } else {
    run(std::integral_constant<int, 0>{});
  }
}

template <typename TC>
__device__ __forceinline__ void store_c(gptr<TC> dst, double val, const GBlk &blk) {
  val *= blk.alpha;
  if (blk.beta != 0.0) val += blk.beta * (double)(*dst);
  *dst = (TC)val;
}

// The complex form: alpha and beta are complex (Gemm_Batch passes Scalars; contractions use
// alpha = 1, beta = 0).
template <typename op_t, typename C2>
__device__ __forceinline__ void store_cplx(C2 dst, double xr, double xi, const GBlk &blk) {
  double re = blk.alpha * xr - blk.alpha_im * xi, im = blk.alpha * xi + blk.alpha_im * xr;
  if (blk.beta != 0.0 || blk.beta_im != 0.0) {
    const auto o = *dst;
    re += blk.beta * (double)o.x - blk.beta_im * (double)o.y;
    im += blk.beta * (double)o.y + blk.beta_im * (double)o.x;
  }
  typedef op_t c2 __attribute__((ext_vector_type(2)));
  c2 w;
  w.x = (op_t)re;
  w.y = (op_t)im;
  *dst = w;
}

// Sum over the 64 lanes of a wave (butterfly; every lane gets the same value).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The dot-product epilogue of one tile: lane partials of C[e] * x[e] and of x[e]^2 summed over
// the wave into slot[0] and slot[nslots] (lane 0).  The C values come from the accumulators.
__device__ __forceinline__ void dot_epilogue(double cx, double xx, double *slot, int64_t nslots,
                                             int lane) {
  cx = wave_sum(cx);
  xx = wave_sum(xx);
  if (lane == 0) {
    slot[0] = cx;
    slot[nslots] = xx;
  }
}

template <int PREC, typename TA, typename TB, typename TC, int MI, int NI, int PK,
          bool LEAN = false, typename SEGS>
__device__ __forceinline__ void wave_tile_real(const char *__restrict__ Abase,
                                               const char *__restrict__ Bbase,
                                               char *__restrict__ Cbase, const GBlk &blk,
                                               SEGS segs, int m0, int n0, int lane,
                                               const double *__restrict__ dotx = nullptr,
                                               double *dslot = nullptr, int64_t nslots = 0) {
  RealAcc<PREC, MI, NI> acc;
  acc.zero();
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16 * MI, blk.M - m0), nt = min(16 * NI, blk.N - n0);
  // FP32 launches load the dot vector's values of this tile before the K loop, so that their
  // latency overlaps it instead of following it (FP64 launches load them after it: holding them
  // across the loop would cost FP64 tiles a wave per SIMD of occupancy)
  constexpr bool kPre = PREC == CXA_PREC_FP32;
  double xpre[MI][NI][4];
  if (kPre && dslot) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int jj = 0; jj < NI; ++jj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * i + acc_row(RealAcc<PREC, MI, NI>::F64, g, v);
          const int col = 16 * jj + r;
          // branch-free (the zero cell outside the tile), so that the K loop's wait counts
          // stay exact
          xpre[i][jj][v] = load_or_zero<double>(
              (gptr<const double>)(dotx + blk.c_off + (int64_t)(m0 + row) * blk.ldc + (n0 + col)),
              row < mt && col < nt);
        }
  }
  mfma_accumulate<TA, TB, MI, NI, PK, LEAN>(acc, Abase, Bbase, blk, segs, m0, n0, lane, 0, 1);
  gptr<TC> Cp = at<TC>(Cbase, blk.c_off);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * i + acc_row(RealAcc<PREC, MI, NI>::F64, g, v);
        const int col = 16 * jj + r;
        if (row < mt && col < nt)
          store_c(Cp + (int64_t)(m0 + row) * blk.ldc + (n0 + col) * blk.csn, acc.get(i, jj, v),
                  blk);
      }
  if (dslot) {  // uniform over the wave; only launches with an FP64 C and alpha 1, beta 0
    double cx = 0.0, xx = 0.0;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int jj = 0; jj < NI; ++jj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * i + acc_row(RealAcc<PREC, MI, NI>::F64, g, v);
          const int col = 16 * jj + r;
          if (row < mt && col < nt) {
            const double xe =
                kPre ? xpre[i][jj][v]
                     : dotx[blk.c_off + (int64_t)(m0 + row) * blk.ldc + (n0 + col)];
            cx += acc.get(i, jj, v) * xe;
            xx += xe * xe;
          }
        }
    dot_epilogue(cx, xx, dslot, nslots, lane);
  }
}

// Split-K tile: every wave of the workgroup (WAVES of them) calls this for the same tile; wave
// w takes the K chunks c with c % WAVES == w, and the partial tiles are summed in wave order.
template <int PREC, typename TA, typename TB, typename TC, int MI, int NI, int WAVES, int PK,
          typename SEGS, typename RED>
__device__ __forceinline__ void wg_tile_real(const char *__restrict__ Abase,
                                             const char *__restrict__ Bbase,
                                             char *__restrict__ Cbase, const GBlk &blk,
                                             SEGS segs, int m0, int n0, int lane, int wave,
                                             RED red,
                                             const double *__restrict__ dotx = nullptr,
                                             double *dslot = nullptr, int64_t nslots = 0) {
  RealAcc<PREC, MI, NI> acc;
  acc.zero();
  // The waves share the epilogue: wave w sums, stores and (with a dot vector) multiplies the
  // tile values idx = w, w + WAVES, ... of every lane; the dot-vector entries of those values
  // are loaded before the K loop, so that their latency overlaps it instead of following it.
  constexpr int E = MI * NI * 4;
  constexpr int PER = (E + WAVES - 1) / WAVES;
  constexpr bool F64L = RealAcc<PREC, MI, NI>::F64;
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16 * MI, blk.M - m0), nt = min(16 * NI, blk.N - n0);
  auto where = [&](int idx, int *row, int *col) {  // position of value idx of this lane
    const int ij = idx >> 2;
    *row = 16 * (ij / NI) + acc_row(F64L, g, idx & 3);
    *col = 16 * (ij % NI) + r;
  };
  double xpre[PER];
#pragma unroll
  for (int t = 0; t < PER; ++t) xpre[t] = 0.0;
  if (dslot) {
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      const int idx = wave + t * WAVES;
      int row, col;
      where(idx, &row, &col);
      const bool in = idx < E && row < mt && col < nt;
      if constexpr (PREC == CXA_PREC_FP32) {
        // branch-free (the zero cell outside the tile), so that the K loop's wait counts stay
        // exact (measured: FP32 launch 8.8 -> 8.2 us; the same form made the FP64 launch
        // 11 -> 14 us, which keeps the branch)
        xpre[t] = load_or_zero<double>(
            (gptr<const double>)(dotx + blk.c_off + (int64_t)(m0 + row) * blk.ldc + (n0 + col)),
            in);
      } else if (in) {
        xpre[t] = dotx[blk.c_off + (int64_t)(m0 + row) * blk.ldc + (n0 + col)];
      }
    }
  }
  mfma_accumulate<TA, TB, MI, NI, PK>(acc, Abase, Bbase, blk, segs, m0, n0, lane, wave,
                                        WAVES);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wave][(i * NI + jj) * 4 + v][lane] = acc.get(i, jj, v);
  __syncthreads();
  gptr<TC> Cp = at<TC>(Cbase, blk.c_off);
  double cx = 0.0, xx = 0.0;
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int idx = wave + t * WAVES;
    int row, col;
    where(idx, &row, &col);
    if (idx < E && row < mt && col < nt) {
      double s = red[0][idx][lane];
#pragma unroll
      for (int q = 1; q < WAVES; ++q) s += red[q][idx][lane];
      store_c(Cp + (int64_t)(m0 + row) * blk.ldc + (n0 + col) * blk.csn, s, blk);
      cx += s * xpre[t];
      xx += xpre[t] * xpre[t];
    }
  }
  if (dslot) {  // uniform over the workgroup: wave partials, then their sum in wave order
    __shared__ double dred[2][WAVES];
    cx = wave_sum(cx);
    xx = wave_sum(xx);
    if (lane == 0) {
      dred[0][wave] = cx;
      dred[1][wave] = xx;
    }
    __syncthreads();
    if (wave == 0 && lane == 0) {
      double a = dred[0][0], b = dred[1][0];
#pragma unroll
      for (int q = 1; q < WAVES; ++q) {
        a += dred[0][q];
        b += dred[1][q];
      }
      dslot[0] = a;
      dslot[nslots] = b;
    }
  }
  __syncthreads();
}

// Walks the k values kk of a block's concatenated segments with kk % nslices == slice, in
// order (wave-uniform).
template <typename SEGS>
struct RowCursor {
  SEGS segs;
  int seg0, nseg;
  int s, k;
  GSeg sg;
  __device__ __forceinline__ void skip(int n) {
    k += n;
    while (s < nseg && k >= sg.K) {
      k -= sg.K;
      ++s;
      if (s < nseg) sg = segs(seg0 + s);
    }
  }
};

// Row streaming for N <= kRowsN: lane = output row, FP64 accumulation.  The k values of all
// segments form one sequence; kRowsDepth loads of A run ahead of the FMAs that consume them
// (B rows are wave-uniform reads).
constexpr int kRowsDepth = 8;

// element offset of k along a row of A (k4-packed: quad stride sak, 4 consecutive k adjacent)
template <int PK>
__device__ __forceinline__ int64_t a_koff(int k, int64_t sak) {
  return (PK & kPackA) ? (int64_t)(k >> 2) * sak + (k & 3) : (int64_t)k * sak;
}

template <typename TA, typename TB, int PK, typename SEGS>
__device__ __forceinline__ void rows_accumulate(double (&acc)[kRowsN], const char *Abase,
                                                const char *Bbase, const GBlk &blk, SEGS segs,
                                                int row, bool valid, int slice, int nslices) {
  const int N = blk.N;
#pragma unroll
  for (int n = 0; n < kRowsN; ++n) acc[n] = 0.0;
  int total = 0, kb = 0;
  for (int s = 0; s < blk.nseg; ++s) {
    const int K = segs(blk.seg0 + s).K;
    const int first = ((slice - kb) % nslices + nslices) % nslices;
    if (first < K) total += (K - first + nslices - 1) / nslices;
    kb += K;
  }
  if (total == 0) return;
  RowCursor<SEGS> lc{segs, blk.seg0, blk.nseg, 0, 0};
  lc.sg = segs(blk.seg0);
  lc.skip(slice);  // also steps over empty leading segments
  RowCursor<SEGS> cc = lc;
  TA a[kRowsDepth];  // as loaded; widened to FP64 where consumed
#pragma unroll
  for (int d = 0; d < kRowsDepth; ++d) {
    if (d < total) {
      a[d] = load_or_zero<TA>(at<const TA>(Abase, lc.sg.a_off) + ((int64_t)row * lc.sg.sam +
                                                                  a_koff<PK>(lc.k, lc.sg.sak)),
                              valid);
      lc.skip(nslices);
    }
  }
  for (int base = 0; base < total; base += kRowsDepth) {
#pragma unroll
    for (int d = 0; d < kRowsDepth; ++d) {
      const int c = base + d;
      if (c < total) {
        gptr<const TB> bk = at<const TB>(Bbase, cc.sg.b_off) +
                            ((PK & kPackB) ? (int64_t)(cc.k >> 2) * cc.sg.sbk + (cc.k & 3)
                                 : (int64_t)cc.k * cc.sg.sbk);
#pragma unroll
        for (int n = 0; n < kRowsN; ++n)
          if (n < N) acc[n] += (double)a[d] * (double)bk[(int64_t)n * cc.sg.sbn];
        cc.skip(nslices);
        if (c + kRowsDepth < total) {
          a[d] = load_or_zero<TA>(
              at<const TA>(Abase, lc.sg.a_off) +
                  ((int64_t)row * lc.sg.sam + a_koff<PK>(lc.k, lc.sg.sak)),
              valid);
          lc.skip(nslices);
        }
      }
    }
  }
  drain_loads();
}

template <typename TA, typename TB, typename TC, int PK, typename SEGS>
__device__ __forceinline__ void wave_rows(const char *__restrict__ Abase,
                                          const char *__restrict__ Bbase,
                                          char *__restrict__ Cbase, const GBlk &blk, SEGS segs,
                                          int m0, int lane) {
  const int row = m0 + lane;
  const bool valid = row < blk.M;
  double acc[kRowsN];
  rows_accumulate<TA, TB, PK>(acc, Abase, Bbase, blk, segs, row, valid, 0, 1);
  if (!valid) return;
  gptr<TC> Cp = at<TC>(Cbase, blk.c_off) + (int64_t)row * blk.ldc;
#pragma unroll
  for (int n = 0; n < kRowsN; ++n)
    if (n < blk.N) store_c(Cp + n * blk.csn, acc[n], blk);
}

// Row tile of short K: kShortRows rows per lane (64 apart), N <= kShortRowsN.  Bound by the chain
// of dependent loads (records, then B, then A) and by its stores: the A values of four k run
// ahead for all rows, B comes through scalar loads, and where the block is contiguous in C its
// rows are put together in LDS, so that the stores are.  `out`: kShortRows * 64 * kShortRowsN
// values of this wave.  The MPO step of an environment update at bond dimension 2048 (19 MB
// written, K of 1 to 4, N of 1 or 3): 21.4 us with one row per lane, 12.6 us so.
template <typename TA, typename TB, typename TC, int PK, typename SEGS>
__device__ __forceinline__ void wave_rows_short(const char *__restrict__ Abase,
                                                const char *__restrict__ Bbase,
                                                char *__restrict__ Cbase, const GBlk &blk,
                                                SEGS segs, int m0, int lane, double *out) {
  constexpr int R = kShortRows, NB = kShortRowsN, D = 4;
  const int N = blk.N;
  int total = 0;
  for (int s = 0; s < blk.nseg; ++s) total += segs(blk.seg0 + s).K;
  double acc[R][NB];
#pragma unroll
  for (int q = 0; q < R; ++q)
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[q][n] = 0.0;
  if (total > 0) {
    RowCursor<SEGS> lc{segs, blk.seg0, blk.nseg, 0, 0};
    lc.sg = segs(blk.seg0);
    lc.skip(0);
    TA a[D][R];
    TB b[D][NB];
    auto load = [&](int d) {
      gptr<const TA> ak = at<const TA>(Abase, lc.sg.a_off) + a_koff<PK>(lc.k, lc.sg.sak);
      typedef const TB __attribute__((address_space(4))) *sptr;  // uniform: scalar loads
      const sptr bk = (sptr)(at<const TB>(Bbase, lc.sg.b_off) +
                             ((PK & kPackB) ? (int64_t)(lc.k >> 2) * lc.sg.sbk + (lc.k & 3)
                                            : (int64_t)lc.k * lc.sg.sbk));
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int row = m0 + 64 * q + lane;
        a[d][q] = load_or_zero<TA>(ak + (int64_t)row * lc.sg.sam, row < blk.M);
      }
#pragma unroll
      for (int n = 0; n < NB; ++n) b[d][n] = bk[n < N ? (int64_t)n * lc.sg.sbn : 0];
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < total) {
        load(d);
        lc.skip(1);
      }
    for (int base = 0; base < total; base += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (base + d >= total) break;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int q = 0; q < R; ++q) acc[q][n] += (double)a[d][q] * (double)b[d][n];
        if (base + d + D < total) {
          load(d);
          lc.skip(1);
        }
      }
    }
    drain_loads();
  }
  gptr<TC> Cp = at<TC>(Cbase, blk.c_off) + (int64_t)m0 * blk.ldc;
  const int rows = min(64 * R, blk.M - m0);
  if (blk.csn == 1 && blk.ldc == N) {
    __builtin_amdgcn_wave_barrier();  // the last tile's reads
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int n = 0; n < NB; ++n)
        if (n < N) out[(64 * q + lane) * N + n] = acc[q][n];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int e = lane; e < rows * N; e += 64) store_c(Cp + e, out[e], blk);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  } else {
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int n = 0; n < NB; ++n)
        if (64 * q + lane < rows && n < N)
          store_c(Cp + ((int64_t)(64 * q + lane) * blk.ldc + n * blk.csn), acc[q][n], blk);
  }
}

// Split-K row tile: the four waves take interleaved k values of the same 64 rows.
template <typename TA, typename TB, typename TC, int PK, typename SEGS>
__device__ __forceinline__ void wg_rows(const char *__restrict__ Abase,
                                        const char *__restrict__ Bbase, char *__restrict__ Cbase,
                                        const GBlk &blk, SEGS segs, int m0, int lane, int wave,
                                        double (*red)[16][64]) {
  const int row = m0 + lane;
  const bool valid = row < blk.M;
  double acc[kRowsN];
  rows_accumulate<TA, TB, PK>(acc, Abase, Bbase, blk, segs, row, valid, wave, kWaves);
#pragma unroll
  for (int n = 0; n < kRowsN; ++n) red[wave][n][lane] = acc[n];
  __syncthreads();
  if (wave == 0 && valid) {
    gptr<TC> Cp = at<TC>(Cbase, blk.c_off) + (int64_t)row * blk.ldc;
#pragma unroll
    for (int n = 0; n < kRowsN; ++n)
      if (n < blk.N)
        store_c(Cp + n * blk.csn,
                ((red[0][n][lane] + red[1][n][lane]) + red[2][n][lane]) + red[3][n][lane], blk);
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------------------
// complex MFMA tiles: elements move as two-wide vectors (x = real, y = imaginary; same size and
// alignment as the structs), which load and store through global-address-space pointers.
// conj: bit 0 conjugates A, bit 1 conjugates B.
// ---------------------------------------------------------------------------------------
typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
template <typename CT>
struct CplxOf;
template <>
struct CplxOf<cd> {
  using op = double;
  using vec = d2v;
};
template <>
struct CplxOf<cf> {
  using op = float;
  using vec = f2v;
};

template <typename CT, int MI, int NI, bool LEAN = false, typename SEGS>
__device__ __forceinline__ void wave_tile_cplx(const char *__restrict__ Abase,
                                               const char *__restrict__ Bbase,
                                               char *__restrict__ Cbase, const GBlk &blk,
                                               SEGS segs, int m0, int n0, int lane, int conj) {
  using op_t = typename CplxOf<CT>::op;
  using c2 = typename CplxOf<CT>::vec;
  static_assert(sizeof(c2) == sizeof(CT), "complex element layout");
  CplxAcc<op_t, MI, NI> acc;
  acc.zero();
  acc.sa = (conj & 1) ? op_t(-1) : op_t(1);
  acc.sb = (conj & 2) ? op_t(-1) : op_t(1);
  mfma_accumulate<c2, c2, MI, NI, 0, LEAN>(acc, Abase, Bbase, blk, segs, m0, n0, lane, 0, 1);
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16 * MI, blk.M - m0), nt = min(16 * NI, blk.N - n0);
  gptr<c2> Cp = at<c2>(Cbase, blk.c_off);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int jj = 0; jj < NI; ++jj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * i + acc_row(CplxAcc<op_t, MI, NI>::F64, g, v);
        const int col = 16 * jj + r;
        if (row < mt && col < nt)
          store_cplx<op_t>(Cp + ((int64_t)(m0 + row) * blk.ldc + (n0 + col) * blk.csn),
                           (double)acc.re[i][jj][v], (double)acc.im[i][jj][v], blk);
      }
}

// Split-K 16 x 16 tile: wave w of the workgroup takes the K chunks c with c % WAVES == w; the
// partial tiles meet in LDS and value idx of every lane is summed in wave order and stored by
// wave idx % WAVES.  A lone wave runs its K range's MFMAs one after another on one SIMD: where a
// launch has fewer tiles than SIMDs, the split spreads a tile over the CU's four.
template <typename CT, int WAVES, typename SEGS>
__device__ __forceinline__ void wg_tile_cplx(const char *__restrict__ Abase,
                                             const char *__restrict__ Bbase,
                                             char *__restrict__ Cbase, const GBlk &blk, SEGS segs,
                                             int m0, int n0, int lane, int wave, int conj,
                                             typename CplxOf<CT>::op (*red)[8][64]) {
  using op_t = typename CplxOf<CT>::op;
  using c2 = typename CplxOf<CT>::vec;
  CplxAcc<op_t, 1, 1> acc;
  acc.zero();
  acc.sa = (conj & 1) ? op_t(-1) : op_t(1);
  acc.sb = (conj & 2) ? op_t(-1) : op_t(1);
  mfma_accumulate<c2, c2, 1, 1, 0>(acc, Abase, Bbase, blk, segs, m0, n0, lane, wave, WAVES);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    red[wave][v][lane] = acc.re[0][0][v];
    red[wave][4 + v][lane] = acc.im[0][0][v];
  }
  __syncthreads();
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16, blk.M - m0), nt = min(16, blk.N - n0);
  if (wave < 4) {
    const int row = acc_row(CplxAcc<op_t, 1, 1>::F64, g, wave);
    if (row < mt && r < nt) {
      double re = (double)red[0][wave][lane], im = (double)red[0][4 + wave][lane];
#pragma unroll
      for (int q = 1; q < WAVES; ++q) {
        re += (double)red[q][wave][lane];
        im += (double)red[q][4 + wave][lane];
      }
      store_cplx<op_t>(
          at<c2>(Cbase, blk.c_off) + ((int64_t)(m0 + row) * blk.ldc + (n0 + r) * blk.csn), re, im,
          blk);
    }
  }
  __syncthreads();
}

// Tile classes: each class is its own kernel instantiation so that it carries only its own
// register budget (occupancy matters most for the memory-bound row tiles).  TC_LEAN is TC_MIXED for
// launches of short K.
// TC_ROWS4 is TC_ROWS for launches that hold tiles of kShortRows rows per lane (GemmLaunch::rows4):
// their registers (83 to 99 for 40 to 55) and LDS would hold the others to five workgroups a CU
// (10^6 rows of N = 6, K = 10: FP32 46 us for 39; 300000 of N = 8, K = 20: 44 for 34).
enum TileClass { TC_MIXED = 0, TC_ROWS = 1, TC_BIG = 2, TC_LDS = 3, TC_LEAN = 4, TC_ROWS4 = 5 };
// A lean tile walks the segments and their chunks one at a time, with one set of fragments and
// 32-bit offsets only, so that four waves (complex128: three) fit a SIMD where the ring's registers
// leave two: with few chunks of K there is little to pipeline, and other waves hide the latency of
// a tile's first loads and its stores.  Products of 3000 x 3000, us, ring / lean: FP32 K = 17
// 17.6 / 15.9, 100 32.1 / 31.2; FP64 K = 5 22.9 / 17.5, 17 26.6 / 22.5; complex64 K = 17 37.5 /
// 32.1, 50 58.1 / 51.4.  Complex128 tiles hold so many values that the ring had no depth for them:
// they are always lean (200 blocks of 300 x 8, K = 200: 42 / 40; 100000 x 10, K = 200: 96 / 85).
template <typename T>
constexpr int kLeanWaves = std::is_same<T, cd>::value ? 3 : std::is_same<T, cf>::value ? 5 : 4;

template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int CLS, int PK,
          typename SEGS>
__device__ __forceinline__ void run_tile(int kind, const char *A, const char *B, char *C,
                                         const GBlk &blk, SEGS segs, int m0, int n0, int lane,
                                         int conj, const double *dotx = nullptr,
                                         double *dslot = nullptr, int64_t nslots = 0) {
  constexpr bool L = CLS == TC_LEAN;
  if constexpr (CPLX) {
    switch (kind) {
      case TK_1x1: wave_tile_cplx<TA, 1, 1, L>(A, B, C, blk, segs, m0, n0, lane, conj); break;
      case TK_2x1: wave_tile_cplx<TA, 2, 1, L>(A, B, C, blk, segs, m0, n0, lane, conj); break;
      case TK_1x2: wave_tile_cplx<TA, 1, 2, L>(A, B, C, blk, segs, m0, n0, lane, conj); break;
      default: wave_tile_cplx<TA, 2, 2, L>(A, B, C, blk, segs, m0, n0, lane, conj); break;
    }
  } else if constexpr (CLS == TC_ROWS || CLS == TC_ROWS4) {
    wave_rows<TA, TB, TC, PK>(A, B, C, blk, segs, m0, lane);
  } else if constexpr (CLS == TC_BIG) {
    wave_tile_real<PREC, TA, TB, TC, 4, 2, PK>(A, B, C, blk, segs, m0, n0, lane, dotx, dslot,
                                               nslots);
  } else {
    switch (kind) {
      case TK_1x1:
        wave_tile_real<PREC, TA, TB, TC, 1, 1, PK, L>(A, B, C, blk, segs, m0, n0, lane, dotx, dslot,
                                                      nslots);
        break;
      case TK_2x1:
        wave_tile_real<PREC, TA, TB, TC, 2, 1, PK, L>(A, B, C, blk, segs, m0, n0, lane, dotx, dslot,
                                                      nslots);
        break;
      case TK_1x2:
        wave_tile_real<PREC, TA, TB, TC, 1, 2, PK, L>(A, B, C, blk, segs, m0, n0, lane, dotx, dslot,
                                                      nslots);
        break;
      default:
        wave_tile_real<PREC, TA, TB, TC, 2, 2, PK, L>(A, B, C, blk, segs, m0, n0, lane, dotx, dslot,
                                                      nslots);
        break;
    }
  }
}

// grouped launch: tiles, blocks and segments come from device arrays; one wave per tile.
// Workgroup w runs on XCD w % kXcds and takes tiles from that XCD's range of the list.
template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int CLS, int PK>
__global__ __launch_bounds__(64 * kWaves, CLS == TC_LEAN ? kLeanWaves<TA> : 2) void k_grouped(
    const GTile *__restrict__ tiles, int per_xcd, const GBlk *__restrict__ blks,
    const GSeg *__restrict__ segs, const char *A, const char *B, char *C, int conj,
    const double *dotx, double *dotp) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x % kXcds;
  const GTile *range = tiles + (int64_t)x * per_xcd;
  const int stride = (gridDim.x / kXcds) * kWaves;
  for (int t = (blockIdx.x / kXcds) * kWaves + wave; t < per_xcd; t += stride) {
    const GTile tl = range[t];
    double *dslot = dotp ? dotp + (int64_t)x * per_xcd + t : nullptr;
    if (tl.blk < 0) {  // padding
      if (dslot && lane == 0) dslot[0] = dslot[(int64_t)kXcds * per_xcd] = 0.0;
      continue;
    }
    const GBlk blk = blks[tl.blk];
    if constexpr (CLS == TC_ROWS4) {
      __shared__ double out[kWaves][kShortRows * 64 * kShortRowsN];
      if (tl.n0 > 64) {  // (uniform over the wave)
        wave_rows_short<TA, TB, TC, PK>(A, B, C, blk, SegArray{segs}, tl.m0, lane, out[wave]);
        continue;
      }
    }
    run_tile<PREC, TA, TB, TC, CPLX, CLS, PK>(tl.kind, A, B, C, blk, SegArray{segs}, tl.m0,
                                               tl.n0, lane, conj, dotx, dslot,
                                               (int64_t)kXcds * per_xcd);
  }
}

// grouped launch with workgroup split-K: one workgroup per tile (real dtypes; the mixed MFMA
// class or the row class)
template <int PREC, typename TA, typename TB, typename TC, int CLS, int WAVES, int PK>
__global__ __launch_bounds__(64 * WAVES, 2) void k_grouped_split(
    const GTile *__restrict__ tiles, int per_xcd, const GBlk *__restrict__ blks,
    const GSeg *__restrict__ segs, const char *A, const char *B, char *C,
    const double *dotx, double *dotp) {
  static_assert(CLS != TC_ROWS || WAVES == kWaves, "row tiles split over four waves");
  __shared__ double red[WAVES][16][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
    const SegArray sa{segs};
    if constexpr (CLS == TC_ROWS) {
      for (int m = tl.m0; m < min(blk.M, tl.m0 + tl.n0); m += 64)
        wg_rows<TA, TB, TC, PK>(A, B, C, blk, sa, m, lane, wave, red);
    } else {
      switch (tl.kind) {
        case TK_1x1:
          wg_tile_real<PREC, TA, TB, TC, 1, 1, WAVES, PK>(A, B, C, blk, sa, tl.m0, tl.n0, lane,
                                                          wave,
                                                     red, dotx, dslot,
                                                     (int64_t)kXcds * per_xcd);
          break;
        case TK_2x1:
          wg_tile_real<PREC, TA, TB, TC, 2, 1, WAVES, PK>(A, B, C, blk, sa, tl.m0, tl.n0, lane,
                                                          wave,
                                                     red, dotx, dslot,
                                                     (int64_t)kXcds * per_xcd);
          break;
        case TK_1x2:
          wg_tile_real<PREC, TA, TB, TC, 1, 2, WAVES, PK>(A, B, C, blk, sa, tl.m0, tl.n0, lane,
                                                          wave,
                                                     red, dotx, dslot,
                                                     (int64_t)kXcds * per_xcd);
          break;
        default:
          wg_tile_real<PREC, TA, TB, TC, 2, 2, WAVES, PK>(A, B, C, blk, sa, tl.m0, tl.n0, lane,
                                                          wave,
                                                     red, dotx, dslot,
                                                     (int64_t)kXcds * per_xcd);
          break;
      }
    }
  }
}

// the complex form: 16 x 16 tiles
template <typename CT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void k_grouped_split_cplx(
    const GTile *__restrict__ tiles, int per_xcd, const GBlk *__restrict__ blks,
    const GSeg *__restrict__ segs, const char *A, const char *B, char *C, int conj) {
  __shared__ typename CplxOf<CT>::op red[WAVES][8][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const GTile *range = tiles + (int64_t)(blockIdx.x % kXcds) * per_xcd;
  for (int t = blockIdx.x / kXcds; t < per_xcd; t += gridDim.x / kXcds) {
    const GTile tl = range[t];
    if (tl.blk < 0) continue;  // padding (uniform over the workgroup)
    const GBlk blk = blks[tl.blk];
    wg_tile_cplx<CT, WAVES>(A, B, C, blk, SegArray{segs}, tl.m0, tl.n0, lane, wave, conj, red);
  }
}

// single block, 16 x 16 tiles split over the waves of a workgroup
template <int PREC, typename TA, typename TB, typename TC, bool CPLX>
__global__ __launch_bounds__(64 * kWaves, 2) void k_single_split(GBlk blk, GSeg seg, int tiles_n,
                                                               const char *A, const char *B,
                                                               char *C, int conj) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = (int)(blockIdx.x / tiles_n) * 16, n0 = (int)(blockIdx.x % tiles_n) * 16;
  if constexpr (CPLX) {
    __shared__ typename CplxOf<TA>::op red[kWaves][8][64];
    wg_tile_cplx<TA, kWaves>(A, B, C, blk, SegOne{seg}, m0, n0, lane, wave, conj, red);
  } else {
    __shared__ double red[kWaves][4][64];
    wg_tile_real<PREC, TA, TB, TC, 1, 1, kWaves, 0>(A, B, C, blk, SegOne{seg}, m0, n0, lane, wave,
                                                   red);
  }
}

#include "gemm_lds.hpp"

// ---------------------------------------------------------------------------------------
// mix launches: one workgroup per tile of an item, of kMixSlices waves (wave s computes slice s:
// the longest dependent load chain of a tile is one slice's K range) or of 4 waves (wave w
// computes slices w and w + 4: no idle waves on items with up to 4 slices); the slice tiles meet
// in LDS, and the waves then write the item's outputs, each a fixed-order weighted sum of the
// slice tiles.
// ---------------------------------------------------------------------------------------
struct SegStride {
  const GSeg *p;
  int base, stride;
  __device__ __forceinline__ GSeg operator()(int i) const { return p[base + i * stride]; }
};

// Segment i of `segs` (nseg <= NACC) accumulates into acc[i]; one load pipeline runs across
// all of them (as in mfma_accumulate).
template <int PREC, typename TA, typename TB, int MI, int NI, int NACC, int PK, typename SEGS>
__device__ __forceinline__ void mfma_accumulate_multi(RealAcc<PREC, MI, NI> (&acc)[NACC],
                                                      const char *__restrict__ Abase,
                                                      const char *__restrict__ Bbase, SEGS segs,
                                                      int nseg, int M, int N, int m0, int n0,
                                                      int lane, bool wide) {
  constexpr int D = RealAcc<PREC, MI, NI>::depth;
  const int r = lane & 15, g = lane >> 4;
  const int mt = min(16 * MI, M - m0);
  const int nt = min(16 * NI, N - n0);
  int nc[NACC];
  int total = 0;
#pragma unroll
  for (int q = 0; q < NACC; ++q) {
    nc[q] = q < nseg ? (segs(q).K + 15) >> 4 : 0;
    total += nc[q];
  }
  if (total == 0) return;
  int cs = 0, left = nc[0];
#pragma unroll
  for (int q = 1; q < NACC; ++q)
    if (left == 0 && cs == q - 1) {
      cs = q;
      left = nc[q];
    }
  // chunk -> accumulator bookkeeping
  auto consume = [&](const Frag<TA, TB, MI, NI> &fr) {
#pragma unroll
    for (int q = 0; q < NACC; ++q)
      if (q == cs) mma_frag(acc[q], fr);
    if (--left == 0) {
#pragma unroll
      for (int q = 1; q < NACC; ++q)
        if (left == 0 && cs == q - 1) {
          cs = q;
          left = nc[q];
        }
    }
  };
  if (wide) {
    ChunkCursor<TA, TB, SEGS> cur{segs, 0, nseg, 1, m0, n0, 0, 0};
    cur.enter(Abase, Bbase);
    cur.skip(0, Abase, Bbase);
    for (int c = 0; c < total; ++c) {
      Frag<TA, TB, MI, NI> f;
      cur.template load<MI, NI, PK>(f, mt, nt, r, g);
      cur.skip(1, Abase, Bbase);
      consume(f);
    }
    drain_loads();
    return;
  }
  ChunkStream<TA, TB, MI, NI, PK, NACC == 1, 0, SEGS> st{segs, 0, nseg, 1, m0, n0, mt, nt, r, g};
  st.start(0, Abase, Bbase);
  Frag<TA, TB, MI, NI> f[D];
  run_chunks<D, NACC == 1>(
      total, [&](int d) { st.load(f[d]); }, [&]() { st.next(Abase, Bbase); },
      [&](int d) { consume(f[d]); });
}

template <int PREC, typename TA, typename TB, typename TC, int MI, int NI, int WAVES, int PK>
__global__ __launch_bounds__(64 * WAVES, MI *NI == 4 && WAVES == 4 ? 2 : 4) void k_mix(
    const GTile *__restrict__ tiles, int per_xcd, const GBlk *__restrict__ items,
    const GSeg *__restrict__ slices, const MixOut *__restrict__ outs, const char *A, const char *B,
    char *C) {
  using acc_t = typename std::conditional<PREC == CXA_PREC_FP32, float, double>::type;
  constexpr int E = MI * NI * 4;              // accumulator values per lane and slice
  constexpr int NACC = kMixSlices / WAVES;    // slices per wave
  constexpr bool F64 = RealAcc<PREC, MI, NI>::F64;
  __shared__ acc_t xs[kMixSlices][E][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const GTile *range = tiles + (int64_t)(blockIdx.x % kXcds) * per_xcd;
  const int stride = gridDim.x / kXcds;
  for (int t = blockIdx.x / kXcds; t < per_xcd; t += stride) {
    const GTile tl = range[t];
    if (tl.blk < 0) continue;  // padding (uniform over the workgroup)
    const GBlk it = items[tl.blk];
    const int mine = it.nseg > wave ? (it.nseg - wave + WAVES - 1) / WAVES : 0;
    // this wave's first output record, loaded before the K loop so that its latency overlaps
    // the loop instead of following it
    MixOut o_first{};
    if (wave < it.nout) o_first = outs[it.out0 + wave];
    if (mine > 0) {
      RealAcc<PREC, MI, NI> acc[NACC];
#pragma unroll
      for (int q = 0; q < NACC; ++q) acc[q].zero();
      mfma_accumulate_multi<PREC, TA, TB, MI, NI, NACC, PK>(
          acc, A, B, SegStride{slices, it.seg0 + wave, WAVES}, mine, it.M, it.N, tl.m0, tl.n0,
          lane, (it.wide & kWideStrides) != 0);
#pragma unroll
      for (int q = 0; q < NACC; ++q) {
        const int sl = wave + q * WAVES;
        if (sl < it.nseg) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int jj = 0; jj < NI; ++jj)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                xs[sl][(i * NI + jj) * 4 + v][lane] = (acc_t)acc[q].get(i, jj, v);
        }
      }
    }
    __syncthreads();
    // Each lane writes rows 16i + 4g .. 16i + 4g + 3 of its column: the slice tiles are in LDS,
    // so the values come from whichever lane and register held those rows (the FP64 MFMA
    // layout spreads four consecutive rows over the four lane groups), and a packed output
    // gets them as one k-quad store where the quad is aligned and whole.
    const int mt = min(16 * MI, it.M - tl.m0), nt = min(16 * NI, it.N - tl.n0);
    for (int j = wave; j < it.nout; j += WAVES) {
      const MixOut o = j == wave ? o_first : outs[it.out0 + j];
      gptr<TC> Cp = at<TC>(C, o.c_off);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int jj = 0; jj < NI; ++jj) {
          const int col = 16 * jj + r;
          const int row0 = 16 * i + 4 * g;
          TC vals[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            // row row0 + v sits in lane group gs, register slot vs (acc_row(F64, gs, vs))
            const int gs = F64 ? v : g, vs = F64 ? g : v;
            const int e = (i * NI + jj) * 4 + vs;
            const int src = r + 16 * gs;
            double val = 0.0;
#pragma unroll
            for (int q = 0; q < kMixSlices; ++q)
              if (q < it.nseg) val += o.coef[q] * (double)xs[q][e][src];
            vals[v] = (TC)val;
          }
          if (col < nt) {
            if constexpr ((PK & kPackC) != 0) {  // c_off: region base, ldc: first k
              const int64_t kk = o.ldc + tl.m0 + row0;
              const int64_t cpos = (int64_t)(tl.n0 + col) * 4;
              const int64_t qs = 4 * (int64_t)it.N;
              if ((kk & 3) == 0 && row0 + 3 < mt) {
                typedef TC tc4 __attribute__((ext_vector_type(4)));
                tc4 w;
                w.x = vals[0];
                w.y = vals[1];
                w.z = vals[2];
                w.w = vals[3];
                *(gptr<tc4>)(Cp + ((kk >> 2) * qs + cpos)) = w;
              } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  if (row0 + v < mt)
                    Cp[((kk + v) >> 2) * qs + cpos + ((kk + v) & 3)] = vals[v];
              }
            } else {
#pragma unroll
              for (int v = 0; v < 4; ++v)
                if (row0 + v < mt)
                  Cp[(int64_t)(tl.m0 + row0 + v) * o.ldc + (tl.n0 + col)] = vals[v];
            }
          }
        }
    }
    __syncthreads();  // the next tile reuses xs
  }
}

// Packed (k4) B operands are built for the fixed operands of a chain: FP32 copies in FP32 mode,
// the FP64 tensors otherwise; only those kernel variants exist.
template <int PREC, typename TB>
constexpr bool k4_ok() {
  return PREC == CXA_PREC_FP32 ? std::is_same<TB, float>::value
                               : std::is_same<TB, double>::value;
}

template <int PREC, typename TA, typename TB, typename TC, int MI, int NI, int PK>
void launch_mix_kind_t(const GemmLaunch &g, int grid, hipStream_t s) {
  const char *A = (const char *)g.A, *B = (const char *)g.B;
  char *C = (char *)g.C;
  if (g.splitk)  // four waves, two slices each
    hipLaunchKernelGGL((k_mix<PREC, TA, TB, TC, MI, NI, 4, PK>), dim3(grid), dim3(64 * 4), 0,
                       s, g.tiles, g.per_xcd, g.blks, g.segs, g.outs, A, B, C);
  else  // one wave per slice
    hipLaunchKernelGGL((k_mix<PREC, TA, TB, TC, MI, NI, kMixSlices, PK>), dim3(grid),
                       dim3(64 * kMixSlices), 0, s, g.tiles, g.per_xcd, g.blks, g.segs, g.outs,
                       A, B, C);
}

// A packed (k4) A operand of a mix launch is the FP32 running vector of an FP32 chain, read
// with packed B and written to packed outputs; only that variant exists.
template <int PREC, typename TA, typename TB, typename TC>
constexpr bool mix_a4_ok() {
  return PREC == CXA_PREC_FP32 && std::is_same<TA, float>::value && k4_ok<PREC, TB>();
}

// mix layouts: plain, packed B, packed B with packed outputs, packed A and B with packed
// outputs (launch_mix_t checks the flags)
template <int PREC, typename TA, typename TB, typename TC, int MI, int NI>
void launch_mix_kind(const GemmLaunch &g, int grid, hipStream_t s) {
  if constexpr (mix_a4_ok<PREC, TA, TB, TC>()) {
    if (g.a_k4) {
      launch_mix_kind_t<PREC, TA, TB, TC, MI, NI, kPackA | kPackB | kPackC>(g, grid, s);
      return;
    }
  }
  if constexpr (k4_ok<PREC, TB>()) {
    if (g.b_k4 && g.c_k4) {
      launch_mix_kind_t<PREC, TA, TB, TC, MI, NI, kPackB | kPackC>(g, grid, s);
      return;
    }
    if (g.b_k4) {
      launch_mix_kind_t<PREC, TA, TB, TC, MI, NI, kPackB>(g, grid, s);
      return;
    }
  }
  launch_mix_kind_t<PREC, TA, TB, TC, MI, NI, 0>(g, grid, s);
}

template <int PREC, typename TA, typename TB, typename TC>
int launch_mix_t(const GemmLaunch &g, hipStream_t s) {
  if (g.per_xcd <= 0) return CXA_OK;
  if (g.ntiles != kXcds * g.per_xcd)
    return fail(CXA_ERR_INVALID, "mix GEMM: tile list of %d is not %d ranges of %d", g.ntiles,
                kXcds, g.per_xcd);
  if ((g.b_k4 && !k4_ok<PREC, TB>()) || (g.c_k4 && !g.b_k4) ||
      (g.a_k4 && !(mix_a4_ok<PREC, TA, TB, TC>() && g.b_k4 && g.c_k4)))
    return fail(CXA_ERR_UNSUPPORTED, "mix GEMM: no variant for these packed layouts / dtypes");
  const int grid = kXcds * std::min(g.per_xcd, 2048);
  switch (g.kind0) {
    case TK_1x1: launch_mix_kind<PREC, TA, TB, TC, 1, 1>(g, grid, s); break;
    case TK_2x1: launch_mix_kind<PREC, TA, TB, TC, 2, 1>(g, grid, s); break;
    case TK_1x2: launch_mix_kind<PREC, TA, TB, TC, 1, 2>(g, grid, s); break;
    case TK_2x2: launch_mix_kind<PREC, TA, TB, TC, 2, 2>(g, grid, s); break;
    default:
      return fail(CXA_ERR_INVALID, "mix GEMM: tile kind %d is not 16x16, 32x16, 16x32 or 32x32",
                  g.kind0);
  }
  CXA_HIP(hipGetLastError());
  return CXA_OK;
}

// single-block launch: one block with one segment, tiles derived from the launch index, so a
// plain GEMM needs no device-side task list (mixed MFMA class)
template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int CLS>
__global__ __launch_bounds__(64 * kWaves, CLS == TC_LEAN ? kLeanWaves<TA> : 2) void k_single(
    GBlk blk, GSeg seg, int kind, int tiles_n, int ntiles, const char *A, const char *B, char *C,
    int conj) {
  // (checked by launch_t: as constants they take no registers and no arithmetic per element)
  blk.csn = 1;
  blk.alpha = 1.0;
  blk.beta = blk.alpha_im = blk.beta_im = 0.0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tr = kind == TK_1x1 || kind == TK_1x2 ? 16 : 32;
  const int tc = kind == TK_1x1 || kind == TK_2x1 ? 16 : 32;
  for (int t = blockIdx.x * kWaves + wave; t < ntiles; t += gridDim.x * kWaves) {
    const int m0 = (t / tiles_n) * tr, n0 = (t % tiles_n) * tc;
    run_tile<PREC, TA, TB, TC, CPLX, CLS, 0>(kind, A, B, C, blk, SegOne{seg}, m0, n0, lane, conj);
  }
}

template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int PK, int KIND>
void launch_lds_kind(const GemmLaunch &g, int grid, hipStream_t s) {
  const char *A = (const char *)g.A, *B = (const char *)g.B;
  if constexpr (PK == 0) {
    if (g.single) {
      const int tm = (g.blk0.M + tile_rows(KIND) - 1) / tile_rows(KIND);
      const int tn = (g.blk0.N + tile_cols(KIND) - 1) / tile_cols(KIND);
      hipLaunchKernelGGL((k_single_lds<PREC, TA, TB, TC, CPLX, KIND>), dim3(grid),
                         dim3(64 * kWaves), 0, s, g.blk0, g.seg0, tm, tn, tm * tn, A, B,
                         (char *)g.C, g.conj);
      return;
    }
  }
  hipLaunchKernelGGL((k_grouped_lds<PREC, TA, TB, TC, CPLX, KIND, PK>), dim3(grid),
                     dim3(64 * kWaves), 0, s, g.tiles, g.per_xcd, g.blks, g.segs, A, B,
                     (char *)g.C, g.conj, g.dot_x, g.dot_part);
}

template <int PREC, typename TA, typename TB, typename TC, bool CPLX, int PK>
void launch_lds(const GemmLaunch &g, int kind, int grid, hipStream_t s) {
  if constexpr (!CPLX) {
    if (kind == TK_L64) {
      launch_lds_kind<PREC, TA, TB, TC, CPLX, PK, TK_L64>(g, grid, s);
      return;
    }
  }
  launch_lds_kind<PREC, TA, TB, TC, CPLX, PK, TK_L32>(g, grid, s);
}

// the real-dtype grouped launches of one class / split mode
template <int PREC, typename TA, typename TB, typename TC, int PK>
void launch_real(const GemmLaunch &g, int cls, int wg_grid, int wave_grid, hipStream_t s) {
  const int P = g.per_xcd;
  const char *A = (const char *)g.A, *B = (const char *)g.B;
  char *C = (char *)g.C;
  const double *dx = g.dot_x;
  double *dp = g.dot_part;
  if constexpr (PREC != CXA_PREC_FP32X3) {
    if (cls == TC_LDS) {
      launch_lds<PREC, TA, TB, TC, false, PK>(g, g.kind0, wg_grid, s);
      return;
    }
  }
  if (g.splitk && cls == TC_ROWS)
    hipLaunchKernelGGL((k_grouped_split<PREC, TA, TB, TC, TC_ROWS, kWaves, PK>), dim3(wg_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, nullptr,
                       nullptr);
  else if (g.splitk == 8 && cls == TC_MIXED)
    hipLaunchKernelGGL((k_grouped_split<PREC, TA, TB, TC, TC_MIXED, 8, PK>), dim3(wg_grid),
                       dim3(64 * 8), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, dx, dp);
  else if (g.splitk && cls == TC_MIXED)
    hipLaunchKernelGGL((k_grouped_split<PREC, TA, TB, TC, TC_MIXED, kWaves, PK>), dim3(wg_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, dx, dp);
  else if (cls == TC_ROWS && g.rows4)
    hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, false, TC_ROWS4, PK>), dim3(wave_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, g.conj,
                       nullptr, nullptr);
  else if (cls == TC_ROWS)
    hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, false, TC_ROWS, PK>), dim3(wave_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, g.conj,
                       nullptr, nullptr);
  else if (cls == TC_BIG)
    hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, false, TC_BIG, PK>), dim3(wave_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, g.conj, dx,
                       dp);
  else {
    if constexpr (PK == 0 && PREC != CXA_PREC_FP32X3) {
      if (g.lean && !dp) {
        hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, false, TC_LEAN, PK>), dim3(wave_grid),
                           dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, g.conj,
                           nullptr, nullptr);
        return;
      }
    }
    hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, false, TC_MIXED, PK>), dim3(wave_grid),
                       dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs, A, B, C, g.conj, dx,
                       dp);
  }
}

template <int PREC, typename TA, typename TB, typename TC, bool CPLX>
int launch_t(const GemmLaunch &g, hipStream_t s) {
  if (g.dot_part) {  // the dot epilogue: real MFMA tile classes with an FP64 C only
    bool ok = !CPLX && !g.single && g.tile_class != TC_ROWS && g.dot_x != nullptr;
    if constexpr (!std::is_same<TC, double>::value) ok = false;
    if (!ok)
      return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: no dot epilogue for this launch");
  }
  if (g.single) {
    if (g.a_k4 || g.b_k4 || g.c_k4)
      return fail(CXA_ERR_INVALID, "single-block GEMM: packed layouts are not supported");
    const GBlk &b = g.blk0;
    if (b.M <= 0 || b.N <= 0) return CXA_OK;
    if (b.csn != 1 || b.alpha != 1.0 || b.beta != 0.0 || b.alpha_im != 0.0 || b.beta_im != 0.0)
      return fail(CXA_ERR_INVALID, "single-block GEMM: plain products with unit stride along n only");
    const Tiling tl = single_tiling(b, g.seg0, PREC, CPLX);
    int kind = tl.kind;
    if constexpr (PREC != CXA_PREC_FP32X3) {
      if (is_lds(kind)) {
        const int64_t tm = (b.M + tile_rows(kind) - 1) / tile_rows(kind);
        const int64_t tn = (b.N + tile_cols(kind) - 1) / tile_cols(kind);
        if (tm * tn > INT32_MAX / 2)
          return fail(CXA_ERR_UNSUPPORTED, "GEMM too large: %lld tiles", (long long)(tm * tn));
        launch_lds<PREC, TA, TB, TC, CPLX, 0>(g, kind,
                                              kXcds * (int)((tm * tn + kXcds - 1) / kXcds), s);
        CXA_HIP(hipGetLastError());
        return CXA_OK;
      }
    }
    // single launches: mixed class (FP32X3 has no LDS tiles)
    if (kind == TK_ROWS || kind == TK_4x2 || is_lds(kind)) kind = TK_2x2;
    if constexpr (PREC != CXA_PREC_FP32X3) {
      if (tl.split > 0) {
        const int64_t tn = (b.N + 15) / 16, n = (int64_t)((b.M + 15) / 16) * tn;
        if (n > INT32_MAX)
          return fail(CXA_ERR_UNSUPPORTED, "GEMM too large: %lld tiles", (long long)n);
        hipLaunchKernelGGL((k_single_split<PREC, TA, TB, TC, CPLX>), dim3((unsigned)n),
                           dim3(64 * kWaves), 0, s, b, g.seg0, (int)tn, (const char *)g.A,
                           (const char *)g.B, (char *)g.C, g.conj);
        CXA_HIP(hipGetLastError());
        return CXA_OK;
      }
    }
    const int tiles_m = (b.M + tile_rows(kind) - 1) / tile_rows(kind);
    const int tiles_n = (b.N + tile_cols(kind) - 1) / tile_cols(kind);
    const int64_t nt64 = (int64_t)tiles_m * tiles_n;
    if (nt64 > INT32_MAX)
      return fail(CXA_ERR_UNSUPPORTED, "GEMM too large: %lld tiles", (long long)nt64);
    const int ntiles = (int)nt64;
    const int grid = std::min((ntiles + kWaves - 1) / kWaves, 8192);
    auto launch = [&](auto cls) {
      hipLaunchKernelGGL((k_single<PREC, TA, TB, TC, CPLX, decltype(cls)::value>), dim3(grid),
                         dim3(64 * kWaves), 0, s, b, g.seg0, kind, tiles_n, ntiles,
                         (const char *)g.A, (const char *)g.B, (char *)g.C, g.conj);
    };
    if constexpr (PREC != CXA_PREC_FP32X3) {
      if (tl.lean) {
        launch(std::integral_constant<int, TC_LEAN>{});
        CXA_HIP(hipGetLastError());
        return CXA_OK;
      }
    }
    launch(std::integral_constant<int, TC_MIXED>{});
    CXA_HIP(hipGetLastError());
    return CXA_OK;
  }
  if (g.per_xcd <= 0) return CXA_OK;
  if (g.ntiles != kXcds * g.per_xcd)
    return fail(CXA_ERR_INVALID, "grouped GEMM: tile list of %d is not %d ranges of %d",
                g.ntiles, kXcds, g.per_xcd);
  if (g.grid % kXcds)
    return fail(CXA_ERR_INVALID, "grouped GEMM: grid %d is not a multiple of %d", g.grid, kXcds);
  const int cls = g.tile_class;
  if (CPLX && cls != TC_MIXED && cls != TC_LDS)
    return fail(CXA_ERR_UNSUPPORTED, "complex GEMM tiles must be MFMA tiles of 32x32 or LDS tiles");
  if (cls == TC_LDS && g.kind0 != TK_L32 && (CPLX || g.kind0 != TK_L64))
    return fail(CXA_ERR_INVALID, "grouped GEMM: no LDS tile of kind %d for this dtype", g.kind0);
  const int P = g.per_xcd;
  const int wg_grid = g.grid > 0 ? g.grid : kXcds * std::min(P, 2048);
  const int wave_grid = g.grid > 0 ? g.grid : kXcds * std::min((P + kWaves - 1) / kWaves, 1024);
  if constexpr (!CPLX) {
    if (g.c_k4 || (g.a_k4 && !g.b_k4))
      return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: no variant for these packed layouts");
    if (g.a_k4) {
      if constexpr (k4_ok<PREC, TA>() && k4_ok<PREC, TB>())
        launch_real<PREC, TA, TB, TC, kPackA | kPackB>(g, cls, wg_grid, wave_grid, s);
      else
        return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: no packed-A variant for these dtypes");
    } else if (g.b_k4) {
      if constexpr (k4_ok<PREC, TB>())
        launch_real<PREC, TA, TB, TC, kPackB>(g, cls, wg_grid, wave_grid, s);
      else
        return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: no packed-B variant for these dtypes");
    } else {
      launch_real<PREC, TA, TB, TC, 0>(g, cls, wg_grid, wave_grid, s);
    }
  } else {
    if (g.a_k4 || g.b_k4 || g.c_k4)
      return fail(CXA_ERR_UNSUPPORTED, "grouped GEMM: packed layouts are real-only");
    if (cls == TC_LDS)
      launch_lds<PREC, TA, TB, TC, true, 0>(g, g.kind0, wg_grid, s);
    else if (g.splitk == 8)
      hipLaunchKernelGGL((k_grouped_split_cplx<TA, 8>), dim3(wg_grid), dim3(64 * 8), 0, s, g.tiles,
                         P, g.blks, g.segs, (const char *)g.A, (const char *)g.B, (char *)g.C,
                         g.conj);
    else if (g.splitk)
      hipLaunchKernelGGL((k_grouped_split_cplx<TA, 4>), dim3(wg_grid), dim3(64 * 4), 0, s, g.tiles,
                         P, g.blks, g.segs, (const char *)g.A, (const char *)g.B, (char *)g.C,
                         g.conj);
    else {
      auto launch = [&](auto c) {
        hipLaunchKernelGGL((k_grouped<PREC, TA, TB, TC, true, decltype(c)::value, 0>),
                           dim3(wave_grid), dim3(64 * kWaves), 0, s, g.tiles, P, g.blks, g.segs,
                           (const char *)g.A, (const char *)g.B, (char *)g.C, g.conj, nullptr,
                           nullptr);
      };
      if (g.lean)
        launch(std::integral_constant<int, TC_LEAN>{});
      else
        launch(std::integral_constant<int, TC_MIXED>{});
    }
  }
  CXA_HIP(hipGetLastError());
  return CXA_OK;
}

}  // namespace

// precision-family launchers (one translation unit each)
int launch_gemm_fp64(const GemmLaunch &g, hipStream_t s);
int launch_gemm_fp32(const GemmLaunch &g, hipStream_t s);
int launch_gemm_fp32_a64(const GemmLaunch &g, hipStream_t s);
int launch_gemm_c64(const GemmLaunch &g, hipStream_t s);
int launch_gemm_fp32x3(const GemmLaunch &g, hipStream_t s);
int launch_mix(const GemmLaunch &g, hipStream_t s);

}  // namespace cxa
