// FP64-MFMA kernels of the orthonormalization path (gfx950).
//
//   gemm_f64_kernel     row-major C = alpha*op(X)*op(Y) + beta*C + d*I, the
//                       back-multiply T*psi / Lambda*psi and the S->T GEMMs.
//   ovl_f64_kernel      split-K product over the plane-wave index, upper
//                       triangle tiles only for the symmetric overlap (and
//                       all tiles for the asymmetric Lambda product).
//   ovl_reduce_kernel   fixed-order sum of the split-K partials with the kx=0
//                       weight, mirror to the lower triangle, max|S - d I|.
//   ns_* kernels        guarded Newton-Schulz S->T iteration: one elementwise
//                       launch and one GEMM for the first iteration, two GEMM
//                       launches for every later one.
//
// What bounds the products: v_mfma_f64_16x16x4f64 (78.6 TFLOP/s nominal).  A
// register-only loop of independent MFMAs reaches 77 TF from two or four
// waves per SIMD but only 35-38 TF from one: a single wave issues at most
// every other MFMA slot, so with two waves per SIMD each must always have its
// next MFMA ready and no stall of one is made up by the other.  The tiles
// are therefore split so that four waves share a SIMD (at most 128 registers
// each), and the operands go from global memory to LDS by direct-to-LDS loads
// that need no registers.  T psi at n = 1024, npw = 262144: 17.1 ms (64 TF,
// MFMA busy 84 % at 2.29 GHz) with two waves of 64 x 64 per SIMD and register
// staging, 15.5 ms (71 TF, busy 91 % at 2.2 GHz) so; HBM fetch 17.3 -> 6.3 GB.
// What is left is mostly the clock, which falls as the matrix cores fill.
//
// Tiling: a BM x BN tile per workgroup of WR x WC waves; a wave owns WM x WN
// blocks of 16 x 16.  Operand lanes: lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; result register v of lane l holds D[l/16 + 4v][l%16]
// (measured on gfx950).  A stage is BK = 16 contraction indices.  MFMA
// (kk, e) of a stage contracts k = 8 kk + 2 g + e over the lane groups g =
// 0..3, the same for both operands and for every tile, so each output's sum
// runs in one order whatever the tile: all launch forms give the same bits.
//
// LDS panels (R rows of one operand, one stage):
//   KC  (k contiguous in memory): row-major rows of 128 bytes, the eight
//       16-byte k pairs of row r permuted by XOR with (r >> 1) & 7, so that
//       the 16-byte fragment reads of 16 consecutive rows cover all 64 banks.
//       A fragment read returns two consecutive k (both MFMAs e of a kk).
//   !KC (rows contiguous in memory): [k][row], as in memory.  A fragment read
//       returns two consecutive rows of one k, which feed two blocks: blocks
//       2b and 2b + 1 of a wave then hold the even and odd rows of a 32-row
//       span (a wave with one block reads 8 bytes per lane instead).
// MFMAs of blocks past an edge are not issued: row blocks (or spans) are dealt
// to the wave rows in turn, so a ragged last tile drops them from every wave
// alike; the overlap deals the blocks of a ragged or diagonal tile to its
// waves one by one.
#include <math.h>

#include <type_traits>

#include "oa_internal.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // 8-byte aligned pair

constexpr int NT = 256;  // threads of the elementwise kernels
constexpr int BK = 16;

__host__ __device__ __forceinline__ int cdiv(int a, int b) { return (a + b - 1) / b; }

// The dispatcher places workgroup b on XCD b % 8.  Give each XCD a contiguous
// range of logical ids so workgroups sharing operand panels share one L2.
__device__ __forceinline__ int xcd_logical(int b, int nb) {
  const int per = nb >> 3;
  return (b & 7) * per + (b >> 3);
}

// Tile configurations.  WPE waves per SIMD are allowed (512 / WPE registers a
// wave).  The LDS ring has NBUF slots of GRP stages each (NBUF - 1 slots in
// flight, one barrier per slot).
//   T128   the large products: 64 x 32 wave tiles, two workgroups per CU.  Two
//          stages suffice: one stage is 8192 MFMA cycles of a SIMD.  T psi at
//          n = 1024 / 512 / 301 (npw 262144 / 65536 / 20011): 15.5 / 1.05 /
//          0.175 ms; with 64 x 64 wave tiles 15.8 / 1.03 / 0.185; one
//          workgroup of 16 waves per CU and four stages 16.9 / 1.14 / 0.179.
//   T64    many small tiles: 32 x 32 wave tiles, four workgroups per CU.
//   T64W   few tiles (about one per CU): 16 x 32 wave tiles, so that a lone
//          workgroup still puts two waves on a SIMD.
//   T32    fewer still: a quarter of the tile, four times the workgroups.  Each
//          wave is one chain of MFMAs, of which a stage holds four: the LDS
//          latency and the barrier are paid once per GRP stages.
template <int BM_, int BN_, int WR_, int WC_, int WPE_, int NBUF_, int GRP_ = 1>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WR = WR_, WC = WC_, WPE = WPE_, NBUF = NBUF_;
  static constexpr int GRP = GRP_;
  static constexpr int NW = WR * WC, NTHR = 64 * NW;
  static constexpr int WM = BM / (16 * WR), WN = BN / (16 * WC);
  static constexpr int STAGE = (BM + BN) * BK;  // doubles of one stage, X panel then Y
  static constexpr int SMEM = NBUF * GRP * STAGE;
  static_assert(NBUF * GRP >= 2 && NBUF <= 4, "waits below");
};
typedef Tile<128, 128, 2, 4, 4, 2> T128;
typedef Tile<64, 64, 2, 2, 4, 2> T64;
typedef Tile<64, 64, 4, 2, 4, 2, 2> T64W;
typedef Tile<32, 32, 2, 2, 4, 2, 4> T32;

__device__ __forceinline__ bool aligned16(const void *p) {
  return ((uintptr_t)p & 15) == 0;
}

// c + (NEGB ? -1 : 1) a b.  The FP64 MFMAs take their operands' sign bits in the
// field that selects a lane group elsewhere (bit 1: B).
template <bool NEGB>
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, NEGB ? 2 : 0);
}

// Position of block i (16 rows) of a wave inside its panel, and the panel row
// of the block's operand lane idx.  PAIR: blocks 2b, 2b + 1 interleave the
// rows of one 32-row span.
template <int W, int NWAVE, bool KC>
struct RowMap {
  static constexpr bool PAIR = !KC && (W % 2) == 0;
  __device__ static __forceinline__ int first(int i, int wv) {
    return PAIR ? ((i / 2) * NWAVE + wv) * 32 + (i & 1) : (i * NWAVE + wv) * 16;
  }
  __device__ static __forceinline__ int row(int i, int wv, int idx) {
    return first(i, wv) + (PAIR ? 2 * idx : idx);
  }
};

// Fills one operand's R x BK panel of a stage.  The panel is R*8 chunks of 16
// bytes in LDS order; chunk pos = (w + NW*j)*64 + lane belongs to load j of
// wave w.  Three ways to fetch a stage:
//   dma     global_load_lds_dwordx4 straight into the panel: 16-byte aligned
//           operand, whole stage (rows past the edge read the last row, whose
//           products only reach outputs that are not stored)
//   pair    8-byte aligned pairs through registers (odd leading dimensions)
//   masked  element by element, zeros outside [rlim) x [klim): a stage cut by
//           the end of the contraction, or an edge tile that pair cannot read
template <int R, bool KC, int NW>
struct Panel {
  static constexpr int CH = R * BK / 2 / 64 / NW;
  static_assert(CH * NW * 64 * 2 == R * BK, "whole wave loads per stage");
  const double *p[CH];  // this lane's chunks of the next stage to fetch
  long step;            // elements from one stage to the next
  bool dmaok, pairok;

  __device__ __forceinline__ static int pos(int j, int w, int lane) {
    return (w + NW * j) * 64 + lane;
  }
  __device__ __forceinline__ static int kc_pair(int row, int slot) {
    return slot ^ ((row >> 1) & 7);
  }
  __device__ __forceinline__ void init(const double *b, long ld, int r0, int rlim, int k0, int w,
                                       int lane) {
    const bool inner = r0 + R <= rlim;
    const bool al = aligned16(b) && (ld % 2) == 0;
    dmaok = al && (KC ? (k0 % 2) == 0 : (inner || (rlim % 2) == 0));
    pairok = KC || inner;
    step = KC ? (long)BK : BK * ld;
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const int c = pos(j, w, lane);
      if (KC) {
        const int row = c >> 3;
        p[j] = b + (long)min(r0 + row, rlim - 1) * ld + k0 + 2 * kc_pair(row, c & 7);
      } else {
        const int kr = c / (R / 2), col = r0 + 2 * (c % (R / 2));
        p[j] = b + (long)(k0 + kr) * ld + (inner ? col : max(0, min(col, rlim - 2)));
      }
    }
  }
  // a whole stage straight into `buf`; the loads stay in flight
  __device__ __forceinline__ void dma(double *buf, int w) {
#pragma unroll
    for (int j = 0; j < CH; j++) {
      __builtin_amdgcn_global_load_lds(
          p[j], (__attribute__((address_space(3))) void *)(buf + (w + NW * j) * 128), 16, 0, 0);
      p[j] += step;
    }
  }
  // a whole stage into registers, and from them into `buf`
  __device__ __forceinline__ void pair(d2v (&v)[CH]) {
#pragma unroll
    for (int j = 0; j < CH; j++) {
      v[j] = *reinterpret_cast<const d2u *>(p[j]);
      p[j] += step;
    }
  }
  __device__ __forceinline__ static void put(const d2v (&v)[CH], double *buf, int w, int lane) {
#pragma unroll
    for (int j = 0; j < CH; j++)
      *reinterpret_cast<d2v *>(buf + 2 * pos(j, w, lane)) = v[j];
  }
  __device__ __forceinline__ static void masked(const double *b, long ld, int r0, int rlim,
                                                int k0, int klim, double *buf, int w, int lane) {
#pragma unroll 1
    for (int j = 0; j < 2 * CH; j++) {
      const int c = pos(j >> 1, w, lane), e = j & 1;
      const int row = KC ? r0 + (c >> 3) : r0 + 2 * (c % (R / 2)) + e;
      const int k = KC ? k0 + 2 * kc_pair(c >> 3, c & 7) + e : k0 + c / (R / 2);
      buf[2 * c + e] =
          (row < rlim && k < klim) ? b[KC ? (long)row * ld + k : (long)k * ld + row] : 0.0;
    }
  }
};

// The products a tile sums: op(X) op(Y) alone, with +-op(X1) op(Y1) before it
// (one part of a complex product), or with +-op(X1) (J Y1) before it (a real
// matrix times interleaved complex rows).
enum Seg { SEG_ONE = 0, SEG_TWO = 1, SEG_J = 2 };

__device__ __forceinline__ double flip_sign(double x, unsigned bit) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  return __builtin_bit_cast(double, u ^ ((unsigned long long)bit << 32));
}

// One operand's fragments of k step kk of a stage: get(e, i) is this lane's
// value of block i (of the first NI) for MFMA e.
// J (KC): the operand's k are interleaved (re, im) pairs and J y = i y = (-im,
// re) of it is multiplied: a fragment read holds a pair, so J is a swap of
// registers and the MFMA's negation of its B operand where neg(e).
template <int R, bool KC, int W, int NWAVE, int NI, bool J = false>
struct Frags {
  static constexpr bool PAIR = RowMap<W, NWAVE, KC>::PAIR;
  static constexpr int NF = PAIR ? (NI + 1) / 2 : NI;
  d2v f[KC ? NI : 2 * NF];
  __device__ __forceinline__ void load(const double *s, int wv, int kk, int lane) {
    const int r = lane & 15, g = lane >> 4;
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const int row = (i * NWAVE + wv) * 16 + r;
        f[i] = *reinterpret_cast<const d2v *>(s + row * BK +
                                              2 * ((4 * kk + g) ^ ((row >> 1) & 7)));
      }
    } else if constexpr (PAIR) {
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int b = 0; b < NF; b++)
          f[e * NF + b] = *reinterpret_cast<const d2v *>(s + (8 * kk + 2 * g + e) * R +
                                                         (b * NWAVE + wv) * 32 + 2 * r);
    } else {
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int i = 0; i < NI; i++)
          f[e * NF + i][0] = s[(8 * kk + 2 * g + e) * R + (i * NWAVE + wv) * 16 + r];
    }
  }
  __device__ __forceinline__ double get(int e, int i) const {
    if constexpr (KC) return f[i][J ? e ^ 1 : e];
    else if constexpr (PAIR) return f[e * NF + i / 2][i & 1];
    else return f[e * NF + i][0];
  }
  __device__ __forceinline__ static constexpr bool neg(int e) { return J && e == 0; }
  // Turns the fragments of Y1 (`first`) into those of +-Y1 or +-J Y1, J along the
  // rows: a few vector instructions beside MFMAs of 64 cycles.  (A loop of its
  // own per product made the compiler keep two sets of accumulators.)
  template <Seg SEG>
  __device__ __forceinline__ void sign(bool first, bool minus, int lane) {
    static_assert(!KC || SEG != SEG_J, "J along the rows");
    const unsigned m = first && minus ? 0x80000000u : 0u;
    const unsigned jm = m ^ (first ? 0x80000000u : 0u);
#pragma unroll
    for (int i = 0; i < (KC ? NI : 2 * NF); i++) {
      const d2v x = f[i];
      if constexpr (SEG == SEG_TWO || KC) {
        f[i] = d2v{flip_sign(x[0], m), flip_sign(x[1], m)};
      } else if constexpr (PAIR) {
        f[i] = d2v{flip_sign(first ? x[1] : x[0], jm), flip_sign(first ? x[0] : x[1], m)};
      } else {
        const double y = __shfl_xor(x[0], 1);  // the pair's other half
        f[i][0] = first ? flip_sign(y, lane & 1 ? m : jm) : x[0];
      }
    }
  }
  static_assert(KC || !J, "J along k only");
};

// The MFMAs of one stage over the first NI row blocks of the wave.  (A count
// tested per MFMA made the compiler copy the accumulators at every branch, so
// the count is a template argument and the choice lies outside the k loop.)
template <class C, bool XKC, bool YKC, int NI, bool YJ = false, Seg SEG = SEG_ONE>
__device__ __forceinline__ void mma_rows(const double *Xs, const double *Ys, int wr, int wc,
                                         int lane, d4 (&acc)[C::WM * C::WN], bool first = false,
                                         bool minus = false) {
  constexpr int WN = C::WN;
  if constexpr (NI > 0) {
#pragma unroll
    for (int kk = 0; kk < BK / 8; kk++) {
      Frags<C::BM, XKC, C::WM, C::WR, NI> a;
      Frags<C::BN, YKC, WN, C::WC, WN, YJ> b;
      a.load(Xs, wr, kk, lane);
      b.load(Ys, wc, kk, lane);
      if constexpr (SEG != SEG_ONE) b.template sign<SEG>(first, minus, lane);
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
          for (int j = 0; j < WN; j++)
            acc[i * WN + j] = b.neg(e) ? mfma<true>(a.get(e, i), b.get(e, j), acc[i * WN + j])
                                          : mfma<false>(a.get(e, i), b.get(e, j), acc[i * WN + j]);
    }
  }
}

// The MFMAs of one stage over NB single blocks (KC operands): block t has its
// operand rows at panel rows xr[t] and yr[t].
template <int NB, bool YJ>
__device__ __forceinline__ void mma_list(const double *Xs, const double *Ys,
                                         const int (&xr)[NB], const int (&yr)[NB], int lane,
                                         d4 (&acc)[NB]) {
  const int r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < BK / 8; kk++) {
    // rows start at multiples of 16, so the pair permutation depends on r only
    const int off = r * BK + 2 * ((4 * kk + g) ^ ((r >> 1) & 7));
#pragma unroll
    for (int t = 0; t < NB; t++) {
      const d2v a = *reinterpret_cast<const d2v *>(Xs + xr[t] * BK + off);
      const d2v b = *reinterpret_cast<const d2v *>(Ys + yr[t] * BK + off);
      acc[t] = mfma<YJ>(a[0], b[YJ ? 1 : 0], acc[t]);
      acc[t] = mfma<false>(a[1], b[YJ ? 0 : 1], acc[t]);
    }
  }
}

// Calls f(integral_constant<int, V>) with V = v clamped into [LO, HI].
template <int LO, int HI, class F>
__device__ __forceinline__ void count_switch(int v, F &&f) {
  if constexpr (LO < HI) {
    if (v <= LO) f(std::integral_constant<int, LO>{});
    else count_switch<LO + 1, HI>(v, f);
  } else {
    f(std::integral_constant<int, HI>{});
  }
}

// Runs mma(X panel, Y panel, first) over the stages of k in [ka, kb) of one
// tile; with SEG over those of (X1, Y1) first.  YSAME: the Y panel is the X
// panel (diagonal tile of a symmetric product), loaded once.  KZ: the first kz
// (even) columns are cleared in LDS, so that they add nothing, whatever they hold.
template <class C, bool XKC, bool YKC, bool YSAME, Seg SEG = SEG_ONE, bool KZ = false, class Mma>
__device__ __forceinline__ void kloop(const double *X, long ldx, int m0, int mlim,
                                      const double *Y, long ldy, int n0, int nlim, int ka,
                                      int kb, double *smem, Mma &&mma,
                                      const double *X1 = nullptr, const double *Y1 = nullptr,
                                      int kz = 0) {
  constexpr int NBUF = C::NBUF, G = C::GRP, YOFF = YSAME ? 0 : C::BM * BK;
  static_assert(!KZ || (XKC && YKC && G == 1 && SEG == SEG_ONE), "panels as cleared below");
  auto clear = [&](double *buf, int stage) {  // the two panels' rows lie one after another
    constexpr int R = C::BM + (YSAME ? 0 : C::BN);
    const int cols = min(BK, kz - stage * BK);
    if (!KZ || cols <= 0) return;
    for (int i = threadIdx.x; i < R * (cols / 2); i += C::NTHR) {
      const int row = i % R, pair = i / R;
      *reinterpret_cast<d2v *>(buf + row * BK + 2 * (pair ^ ((row >> 1) & 7))) = d2v{0.0, 0.0};
    }
    ring_barrier();
  };
  constexpr bool TWO = SEG != SEG_ONE;
  typedef Panel<C::BM, XKC, C::NW> PX;
  typedef Panel<C::BN, YKC, C::NW> PY;
  const int nfull = (kb - ka) / BK;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  PX lx;
  PY ly;
  auto start = [&](bool first, int k0) {
    lx.init(TWO && first ? X1 : X, ldx, m0, mlim, k0, w, lane);
    if (!YSAME) ly.init(TWO && first ? Y1 : Y, ldy, n0, nlim, k0, w, lane);
  };
  start(TWO, ka);
  const bool dx = lx.dmaok && !(TWO && !aligned16(X));
  const bool dy = YSAME || (ly.dmaok && !(TWO && !aligned16(Y)));
  auto dma = [&](double *buf) {
    lx.dma(buf, w);
    if (!YSAME) ly.dma(buf + YOFF, w);
  };
  if (dx && dy) {
    constexpr int PER = G * (PX::CH + (YSAME ? 0 : PY::CH));  // loads of a slot per wave
    // a product's whole slots, then rem stages: of a lone product after the loop,
    // of two as one more slot of each, so that the first ends before the second
    // begins in every tile
    const int ngrp = nfull / G, rem = nfull % G;
    const int per = TWO && rem > 0 ? ngrp + 1 : ngrp, total = TWO ? 2 * per : ngrp;
    auto stages = [&](int s) {
      return TWO && G > 1 && rem > 0 && (s == per - 1 || s == total - 1) ? rem : G;
    };
    auto issue = [&](int s, int m) {
      double *buf = smem + (s % NBUF) * (G * C::STAGE);
#pragma unroll
      for (int j = 0; j < G; j++)
        if (j < m) dma(buf + j * C::STAGE);
    };
    auto next = [&](int s) {
      if (s < total) {
        if (TWO && s == per) start(false, ka);
        issue(s, stages(s));
      } else if (!TWO && G > 1 && s == ngrp && rem > 0) {
        issue(s, rem);
      }
    };
#pragma unroll
    for (int s = 0; s < NBUF - 1; s++) next(s);
    for (int s = 0; s < total; s++) {
      // slots s + 1 .. min(total - 1, s + NBUF - 2) may stay in flight
      const int ahead = min(total - 1, s + NBUF - 2) - s;
      if (NBUF >= 4 && ahead >= 2) wait_vm<2 * PER>();
      else if (NBUF >= 3 && ahead >= 1) wait_vm<PER>();
      else wait_vm<0>();
      ring_barrier();
      next(s + NBUF - 1);
      if (KZ) clear(smem + (s % NBUF) * C::STAGE, s);
      const double *cur = smem + (s % NBUF) * (G * C::STAGE);
      const int m = stages(s);
      if (m == G) {
#pragma unroll
        for (int j = 0; j < G; j++)
          mma(cur + j * C::STAGE, cur + j * C::STAGE + YOFF, TWO && s < per);
      } else {
        for (int j = 0; j < m; j++)
          mma(cur + j * C::STAGE, cur + j * C::STAGE + YOFF, TWO && s < per);
      }
    }
    if (!TWO && G > 1 && rem > 0) {
      wait_vm<0>();
      ring_barrier();
      const double *cur = smem + (ngrp % NBUF) * (G * C::STAGE);
      for (int j = 0; j < rem; j++)
        mma(cur + j * C::STAGE, cur + j * C::STAGE + YOFF, false);
    }
  } else {
    // one operand at least goes through registers: loaded while the stage
    // before it is multiplied, stored after it
    const bool px = !dx && lx.pairok, py = !dy && ly.pairok;
    const int total = TWO ? 2 * nfull : nfull;
    d2v vx[PX::CH], vy[PY::CH];
    auto load = [&](int s) {
      double *buf = smem + (s & 1) * C::STAGE;
      if (TWO && s == nfull) start(false, ka);
      if (dx) lx.dma(buf, w);
      else if (px) lx.pair(vx);
      if (!YSAME) {
        if (dy) ly.dma(buf + YOFF, w);
        else if (py) ly.pair(vy);
      }
    };
    auto finish = [&](int s) {
      double *buf = smem + (s & 1) * C::STAGE;
      const bool first = TWO && s < nfull;
      const int k0 = ka + (TWO && !first ? s - nfull : s) * BK;
      if (!dx) {
        if (px) PX::put(vx, buf, w, lane);
        else PX::masked(first ? X1 : X, ldx, m0, mlim, k0, kb, buf, w, lane);
      }
      if (!YSAME && !dy) {
        if (py) PY::put(vy, buf + YOFF, w, lane);
        else PY::masked(first ? Y1 : Y, ldy, n0, nlim, k0, kb, buf + YOFF, w, lane);
      }
    };
    if (total > 0) {
      load(0);
      finish(0);
    }
    for (int s = 0; s < total; s++) {
      wait_vm<0>();
      ring_barrier();
      if (s + 1 < total) load(s + 1);
      if (KZ) clear(smem + (s & 1) * C::STAGE, s);
      const double *cur = smem + (s & 1) * C::STAGE;
      mma(cur, cur + YOFF, TWO && s < nfull);
      if (s + 1 < total) finish(s + 1);
    }
  }
  // the rest of a contraction that is no multiple of BK
  const int k0 = ka + nfull * BK;
  if (k0 < kb) {
#pragma nounroll
    for (int seg = TWO ? 0 : 1; seg < 2; seg++) {
      ring_barrier();
      PX::masked(TWO && !seg ? X1 : X, ldx, m0, mlim, k0, kb, smem, w, lane);
      if (!YSAME) PY::masked(TWO && !seg ? Y1 : Y, ldy, n0, nlim, k0, kb, smem + YOFF, w, lane);
      ring_barrier();
      if (KZ) clear(smem, nfull);
      mma(smem, smem + YOFF, TWO && !seg);
    }
  }
  ring_barrier();  // the ring may be refilled (a workgroup's next item)
}

// Field-by-field selection keeps the problem in scalar registers (indexing
// the kernel-argument array with blockIdx.y would copy it to scratch).
struct ProbRegs {
  int M, N, K;
  const double *X;
  long ldx;
  const double *Y;
  long ldy;
  double *C;
  long ldc;
  double alpha, beta, diag_add;
  int cw;
  double alpha_w;
  // second product of the same shape and layouts (SEG): (neg1 ? -1 : 1) X1 Y1
  const double *X1, *Y1;
  bool neg1;
};

__device__ __forceinline__ ProbRegs pick_problem(const oa_gemm_problem &p0,
                                                 const oa_gemm_problem &p1) {
  const bool y = blockIdx.y != 0;
  ProbRegs r;
  r.M = y ? p1.M : p0.M;
  r.N = y ? p1.N : p0.N;
  r.K = y ? p1.K : p0.K;
  r.X = y ? p1.X : p0.X;
  r.ldx = y ? p1.ldx : p0.ldx;
  r.Y = y ? p1.Y : p0.Y;
  r.ldy = y ? p1.ldy : p0.ldy;
  r.C = y ? p1.C : p0.C;
  r.ldc = y ? p1.ldc : p0.ldc;
  r.alpha = y ? p1.alpha : p0.alpha;
  r.beta = y ? p1.beta : p0.beta;
  r.diag_add = y ? p1.diag_add : p0.diag_add;
  r.cw = y ? p1.cw : p0.cw;
  r.alpha_w = y ? p1.alpha_w : p0.alpha_w;
  r.X1 = r.Y1 = nullptr;
  r.neg1 = false;
  return r;
}

struct NoEpi {
  __device__ __forceinline__ double operator()(int, int, int, double x) const { return x; }
};

// One BM x BN output tile `logical` of C = alpha*op(X)*op(Y) + beta*C + d*I (the
// product by SEG); epi(b, m, n, value) returns what is stored for
// each output, of the wave's block b = i * WN + j.
template <bool TX, bool TY, class C, Seg SEG, class Epi>
__device__ __forceinline__ void gemm_body(const ProbRegs &P, int logical, double *smem,
                                          Epi &&epi) {
  constexpr int WM = C::WM, WN = C::WN;
  typedef RowMap<WM, C::WR, !TX> RM;
  typedef RowMap<WN, C::WC, TY> CM;
  const int tmn = cdiv(P.M, C::BM), tnn = cdiv(P.N, C::BN);
  if (logical >= tmn * tnn) return;
  const int tm = logical % tmn, tn = logical / tmn;
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w / C::WC, wc = w % C::WC;
  int ni = 0;  // the wave's row blocks inside the matrix
#pragma unroll
  for (int i = 0; i < WM; i++)
    if (m0 + RM::first(i, wr) < P.M) ni = i + 1;
  d4 acc[WM * WN];
#pragma unroll
  for (int i = 0; i < WM * WN; i++) acc[i] = d4{0, 0, 0, 0};
  count_switch<0, WM>(ni, [&](auto c) {
    constexpr int NI = decltype(c)::value;
    kloop<C, !TX, TY, false, SEG>(P.X, P.ldx, m0, P.M, P.Y, P.ldy, n0, P.N, 0, P.K, smem,
                                  [&](const double *Xs, const double *Ys, bool first) {
                                    mma_rows<C, !TX, TY, NI, false, SEG>(
                                        Xs, Ys, wr, wc, lane, acc, first, P.neg1);
                                  },
                                  P.X1, P.Y1);
  });

  const int r = lane & 15, g = lane >> 4;
  const double alpha = P.alpha, beta = P.beta, dadd = P.diag_add;
  // explicit fma: single and grouped launches inline this body and must
  // round alike
#pragma unroll
  for (int i = 0; i < WM; i++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int m = m0 + RM::row(i, wr, g + 4 * v);
      if (m >= P.M) continue;
      double *crow = P.C + (long)m * P.ldc;
#pragma unroll
      for (int j = 0; j < WN; j++) {
        const int n = n0 + CM::row(j, wc, r);
        if (n >= P.N) continue;
        const double al = (n < P.cw) ? P.alpha_w : alpha, d = (m == n) ? dadd : 0.0;
        if constexpr (CM::PAIR) {
          // blocks j and j + 1 hold columns n and n + 1: one 16-byte access
          if (j & 1) continue;
          const int jo = j + 1 < WN ? j + 1 : j;  // j + 1, spelt so that it stays in range
          const double al1 = (n + 1 < P.cw) ? P.alpha_w : alpha;
          const double d1 = (m == n + 1) ? dadd : 0.0;
          if (n + 1 < P.N) {
            d2v o;
            if (beta == 0.0) {
              o[0] = fma(al, acc[i * WN + j][v], d);
              o[1] = fma(al1, acc[i * WN + jo][v], d1);
            } else {
              const d2v old = *reinterpret_cast<const d2u *>(crow + n);
              o[0] = fma(al, acc[i * WN + j][v], fma(beta, old[0], d));
              o[1] = fma(al1, acc[i * WN + jo][v], fma(beta, old[1], d1));
            }
            o[0] = epi(i * WN + j, m, n, o[0]);
            o[1] = epi(i * WN + jo, m, n + 1, o[1]);
            *reinterpret_cast<d2u *>(crow + n) = o;
            continue;
          }
        }
        const double o = (beta == 0.0) ? fma(al, acc[i * WN + j][v], d)
                                       : fma(al, acc[i * WN + j][v], fma(beta, crow[n], d));
        crow[n] = epi(i * WN + j, m, n, o);
      }
    }
}

template <bool TX, bool TY, class C>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void gemm_f64_kernel(oa_gemm_problem p0, oa_gemm_problem p1, int *mark) {
  if (mark && blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_store(mark, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const ProbRegs P = pick_problem(p0, p1);
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  gemm_body<TX, TY, C, SEG_ONE>(P, xcd_logical(blockIdx.x, gridDim.x), smem, NoEpi{});
}

// out = alpha (op(Mr) psi +- op(Mi) J psi) + beta out: the complex back-multiply
// in one pass over out, J psi never formed.
template <bool TX, class C>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void zback_f64_kernel(oa_gemm_problem p, const double *Mi, int neg) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  ProbRegs P = pick_problem(p, p);
  P.X1 = Mi;
  P.Y1 = p.Y;
  P.neg1 = neg != 0;
  gemm_body<TX, false, C, SEG_J>(P, xcd_logical(blockIdx.x, gridDim.x), smem, NoEpi{});
}

// ------------------------------------------------------------------ grouped
// Instance owning item t: the largest i with prefix[i] <= t.
__device__ __forceinline__ int group_find(const int *__restrict__ prefix, int count, int t) {
  int lo = 0, hi = count;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= t) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Workgroups of XCD x (= b % 8) walk the contiguous item range
// [x*per, (x+1)*per); the grid is a multiple of 8.
template <class F>
__device__ __forceinline__ void for_items(int total, F &&f) {
  const int per = cdiv(total, 8), slots = (int)gridDim.x >> 3, x = blockIdx.x & 7;
  for (int pos = blockIdx.x >> 3; pos < per; pos += slots) {
    const int item = x * per + pos;
    if (item < total) f(item);
  }
}

__device__ __forceinline__ void upper_tile(int tile, int T, int &bi, int &bj) {
  int b = 0, rem = tile;
  while (rem >= T - b) {
    rem -= T - b;
    b++;
  }
  bi = b;
  bj = b + rem;
}

// Tile (bi, bj), bi <= bj, of an upper triangle of T x T tiles: the tiles off
// the diagonal by rows, then the diagonal ones.  The tiles of one k chunk that
// start together then run in step and share their panels in L2 (a diagonal
// tile is done in 5/8 of the time; between the others it let them drift).
__device__ __forceinline__ void sym_tile(int tile, int T, int &bi, int &bj) {
  const int off = T * (T - 1) / 2;
  if (tile >= off) {
    bi = bj = tile - off;
  } else {
    upper_tile(tile, T - 1, bi, bj);
    bj++;
  }
}

// YJ: the product is X (J Y)^T.  With SYM that is the complex overlap's Im S =
// psi (J psi)^T on the upper tiles, whose strict upper triangle is all a
// Hermitian S needs.  Workgroup `block` of nblocks.
template <class C, bool SYM, bool YJ>
__device__ __forceinline__ void ovl_body(const oa_ovl_args &a, int block, int nblocks,
                                         double *smem) {
  constexpr int BM = C::BM, WM = C::WM, WN = C::WN;
  static_assert(C::BM == C::BN, "square tiles");
  typedef RowMap<WM, C::WR, true> RM;
  typedef RowMap<WN, C::WC, true> CM;
  const int Tm = cdiv(a.M, BM), Tn = cdiv(a.N, BM);
  const int ntiles = SYM ? Tm * (Tm + 1) / 2 : Tm * Tn;
  // The short kx = 0 slice (z = 0) takes the leading workgroups, which the
  // dispatcher spreads over all XCDs; the main chunks follow in XCD ranges.
  const int hx = a.kx0_end > 0 ? 1 : 0;
  const int nkx = hx ? cdiv(ntiles, 8) * 8 : 0;
  int tile, z;
  if (block < nkx) {
    if (block >= ntiles) return;
    tile = block;
    z = 0;
  } else {
    const int logical = xcd_logical(block - nkx, nblocks - nkx);
    if (logical >= ntiles * a.nz_main) return;
    tile = logical % ntiles;
    z = logical / ntiles + hx;
  }
  int bi, bj;
  if (SYM) sym_tile(tile, Tm, bi, bj);
  else { bi = tile % Tm; bj = tile / Tm; }
  int ka, kb;
  if (a.kx0_end > 0) {
    if (z == 0) { ka = 0; kb = a.kx0_end; }
    else { ka = a.kx0_end + (z - 1) * a.kchunk; kb = min(a.K, ka + a.kchunk); }
  } else {
    ka = z * a.kchunk;
    kb = min(a.K, ka + a.kchunk);
  }
  const int m0 = bi * BM, n0 = bj * BM;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w / C::WC, wc = w % C::WC;
  const int r = lane & 15, g = lane >> 4;
  double *pt = a.part + ((long)z * ntiles + tile) * (BM * BM);
  // blocks inside the matrix; a symmetric diagonal tile needs those on or
  // above its diagonal
  const bool diag = SYM && bi == bj;
  const int nbr = min(BM / 16, cdiv(a.M - m0, 16)), nbc = min(BM / 16, cdiv(a.N - n0, 16));
  const int nblk = diag ? nbr * (nbr + 1) / 2 : nbr * nbc;
  constexpr bool KZ = SYM && !YJ;
  const int kz = KZ && ka == 0 ? a.kx0_add : 0;
  if (nblk == (BM / 16) * (BM / 16)) {
    d4 acc[WM * WN];
#pragma unroll
    for (int i = 0; i < WM * WN; i++) acc[i] = d4{0, 0, 0, 0};
    kloop<C, true, true, false, SEG_ONE, KZ>(
        a.X, a.ldx, m0, a.M, a.Y, a.ldy, n0, a.N, ka, kb, smem,
        [&](const double *Xs, const double *Ys, bool) {
          mma_rows<C, true, true, WM, YJ>(Xs, Ys, wr, wc, lane, acc);
        },
        nullptr, nullptr, kz);
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
      for (int j = 0; j < WN; j++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          pt[RM::row(i, wr, g + 4 * v) * BM + CM::row(j, wc, r)] = acc[i * WN + j][v];
    return;
  }
  // the blocks of a partial tile, dealt to the waves in turn (a diagonal tile
  // of 128 has 36 of 64: 5 MFMA chains a wave instead of 8); a wave short of
  // one repeats the last, unstored
  count_switch<1, WM * WN>(cdiv(nblk, C::NW), [&](auto c) {
    constexpr int NB = decltype(c)::value;
    d4 acc[NB];
    int xr[NB], yr[NB];
#pragma unroll
    for (int t = 0; t < NB; t++) {
      acc[t] = d4{0, 0, 0, 0};
      const int idx = min(w + C::NW * t, nblk - 1);
      int rb, cb;
      if (diag) upper_tile(idx, nbr, rb, cb);
      else { rb = idx % nbr; cb = idx / nbr; }
      xr[t] = rb * 16;
      yr[t] = cb * 16;
    }
    auto mma = [&](const double *Xs, const double *Ys, bool) {
      mma_list<NB, YJ>(Xs, Ys, xr, yr, lane, acc);
    };
    if (diag)
      kloop<C, true, true, true, SEG_ONE, KZ>(a.X, a.ldx, m0, a.M, a.X, a.ldx, n0, a.N, ka, kb,
                                              smem, mma, nullptr, nullptr, kz);
    else
      kloop<C, true, true, false, SEG_ONE, KZ>(a.X, a.ldx, m0, a.M, a.Y, a.ldy, n0, a.N, ka, kb,
                                               smem, mma, nullptr, nullptr, kz);
#pragma unroll
    for (int t = 0; t < NB; t++)
      if (w + C::NW * t < nblk)
#pragma unroll
        for (int v = 0; v < 4; v++) pt[(xr[t] + g + 4 * v) * BM + yr[t] + r] = acc[t][v];
  });
}

template <class C, bool SYM, bool YJ>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void ovl_f64_kernel(oa_ovl_args a) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  ovl_body<C, SYM, YJ>(a, blockIdx.x, gridDim.x, smem);
}

// C = alpha * (sum over z of the partial tiles), in a fixed order: a workgroup
// owns 16 x 16 outputs, the four waves of z group q add z = q, q + 4, ... and
// the groups combine in order.  (One thread adding all z of an element, one
// load in flight at a time, took 32 us at n = 128 with 128 partials and 83 us
// over four uneven instances; this takes 6 and 20.)  The mirror tile is written
// from LDS, 128 bytes a row.
//   has_kx0: z = 0 holds the leading kx0 columns and counts half.
//   kx0_add: the partial tiles leave out the leading kx0_add columns of psi;
//            half their product is added here.  (Summed with the others and
//            half taken off again, a state that lives on these columns lost a
//            digit and an infinity in them became NaN.)
template <int BM, bool SYM>
__device__ __forceinline__ void ovl_reduce_body(const oa_ovl_args &a, int block,
                                                double (&sums)[4][256], double (&out)[16][17]) {
  constexpr int PB = BM / 16;  // patches per tile edge
  const int M = a.M, N = a.N, nz = a.nz;
  const bool has_kx0 = a.kx0_end > 0;
  const double *psi = a.X;
  const long ld = a.ldx, ldc = a.ldc;
  double *C = a.C;
  const int Tm = cdiv(M, BM), Tn = cdiv(N, BM);
  const int ntiles = SYM ? Tm * (Tm + 1) / 2 : Tm * Tn;
  const int tile = block / (PB * PB), patch = block % (PB * PB);
  int bi, bj;
  if (SYM) sym_tile(tile, Tm, bi, bj);
  else { bi = tile % Tm; bj = tile / Tm; }
  const int pi = (patch / PB) * 16, pj = (patch % PB) * 16;
  if (bi * BM + pi >= M || bj * BM + pj >= N || (SYM && bi == bj && pi > pj)) return;
  const int t = threadIdx.x & 255, q = threadIdx.x >> 8;
  const int lr = t >> 4, lc = t & 15;
  const double *p = a.part + (long)tile * (BM * BM) + (pi + lr) * BM + pj + lc;
  const long zs = (long)ntiles * (BM * BM);
  double s = 0.0;
#pragma unroll 8
  for (int z = q; z < nz; z += 4) {
    const double x = p[z * zs];
    s += (has_kx0 && z == 0) ? 0.5 * x : x;
  }
  sums[q][t] = s;
  __syncthreads();
  const bool dpatch = SYM && bi == bj && pi == pj;  // holds part of the diagonal
  if (q == 0) {
    const int i = bi * BM + pi + lr, j = bj * BM + pj + lc;
    const bool in = i < M && j < N && !(dpatch && lc < lr);
    s = ((sums[0][t] + sums[1][t]) + sums[2][t]) + sums[3][t];
    if (in) {
      double g = 0.0;
      for (int k = 0; k < a.kx0_add; k++) g = fma(psi[(long)i * ld + k], psi[(long)j * ld + k], g);
      s = a.alpha * fma(0.5, g, s);
      C[(long)i * ldc + j] = s;
    }
    out[lr][lc] = s;
    if (a.maxdev) {
      // on the bits of non-negative doubles; a NaN's compare above all others
      const double dv = fabs(s - (i == j ? a.diag : 0.0));
      unsigned long long u = in ? (unsigned long long)__double_as_longlong(dv) : 0ull;
      for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long w = __shfl_xor(u, o);
        u = w > u ? w : u;
      }
      if ((t & 63) == 0) atomicMax(a.maxdev, u);
    }
  }
  if (!SYM) return;
  __syncthreads();
  const int mi = bi * BM + pi + lc, mj = bj * BM + pj + lr;  // C[mj][mi] = out[lc][lr]
  if (q == 0 && mi < M && mj < N && !(dpatch && lr < lc)) C[(long)mj * ldc + mi] = out[lc][lr];
}

template <int BM, bool SYM>
__global__ __launch_bounds__(1024) void ovl_reduce_kernel(oa_ovl_args a) {
  __shared__ double sums[4][256];
  __shared__ double out[16][17];
  ovl_reduce_body<BM, SYM>(a, blockIdx.x, sums, out);
}

// The same over many instances: workgroups prefix[i] .. prefix[i + 1] - 1 are
// those of instance i's own launch, so the sums are the single launches' bit
// for bit.  Instances one after another leave the chip partly idle at both ends
// of every launch: twelve of n = 64 to 512 (npw 8192 to 65536) took 5.45 ms a
// step, together 4.91.
// The table is in order of falling work per workgroup, so the short ones fill
// the end.
template <class C>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void ovl_f64_grouped(const oa_ovl_args *__restrict__ t, const int *__restrict__ prefix,
                     int count) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  const int i = group_find(prefix, count, blockIdx.x);
  const oa_ovl_args a = t[i];
  ovl_body<C, true, false>(a, blockIdx.x - prefix[i], prefix[i + 1] - prefix[i], smem);
}

__global__ __launch_bounds__(1024) void ovl_reduce_grouped(const oa_ovl_args *__restrict__ t,
                                                           const int *__restrict__ prefix,
                                                           int count) {
  __shared__ double sums[4][256];
  __shared__ double out[16][17];
  const int i = group_find(prefix, count, blockIdx.x);
  const int block = blockIdx.x - prefix[i];
  if (t[i].bm == 128) ovl_reduce_body<128, true>(t[i], block, sums, out);
  else ovl_reduce_body<64, true>(t[i], block, sums, out);
}

template <class C>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void gemm_f64_grouped(const oa_gemm_problem *__restrict__ t, const int *__restrict__ prefix,
                      int count) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  const int i = group_find(prefix, count, blockIdx.x);
  const oa_gemm_problem &p = t[i];
  gemm_body<false, false, C, SEG_ONE>(
      pick_problem(p, p), xcd_logical(blockIdx.x - prefix[i], prefix[i + 1] - prefix[i]), smem,
      NoEpi{});
}

__global__ void fill_u64_kernel(unsigned long long *p, unsigned long long v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ------------------------------------------------------------------ S->T
// Ortho's iteration (ortho.C:848-971): C = 3I - A B, B' = B C / 2, A' = C A / 2
// until sqrt(sum (A - A')^2 / n^2) <= tol or maxit (collect_error, :109-146).
// The matrices live in buffers of np x np (n rounded up to 16, zero padding),
// so every product runs whole 16-byte-aligned stages whatever n.  Iteration i
// reads A[i%2], B[i%2] and writes the other pair.
//
// At n <= 1024 the iteration is bound by launches and their latency, not by
// its products (n = 128: 3 x 4 MFLOP), so its launches are few:
//   INIT  B = S/2 or S.  A = I makes the first iteration elementwise:
//         C = 3I - B, A' = C/2, with the residual of A' - I.
//   B1    B' = B C / 2; T = A' where INIT must not store it (`late`: T shares
//         memory with an S that other threads still read).
//   C     C = 3I - A B.
//   PAIR  B' and A' side by side; A' tiles also sum (A - A')^2 and store T.
// A residual left as partial sums by INIT or PAIR is added up by every
// workgroup of the next launch (B1 or C), each of which then knows by itself
// whether the loop has ended; the first one writes the report.  The sums run in
// one order whatever the tiles of either launch (PAIR leaves one per 32 x 32
// block, added up by 256 threads), so all launch forms end alike.  T holds the
// latest iterate throughout.  Before: four launches an iteration, of which a
// one-thread sum of 128 partials took 5 to 9 us, and a final copy to T.
enum NsMode { NS_B1 = 0, NS_C = 1, NS_PAIR = 2 };

// Sum of v over the workgroup in a fixed order; `red` holds one double per
// wave.  Every thread returns the sum.
__device__ __forceinline__ double block_sum(double v, double *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += red[w];
  __syncthreads();
  return s;
}

// Workgroup w of nwg of the first, elementwise iteration.  A non-finite S makes the
// residual NaN (the products of the identity with it would spread NaN), which
// ends the loop; see NS_B1.  Z: S and T hold complex pairs, the buffers a real
// and an imaginary plane (a.zs apart); the residual has two sums.
template <bool Z>
__device__ __forceinline__ void ns_init_body(const oa_ns_args &a, int w, int nwg, double *red) {
  const unsigned n = a.n, np = a.np, nn = np * np;
  const double half = (a.nspin == 1) ? 0.5 : 1.0, nan = __longlong_as_double(0x7ff8000000000000ll);
  double s = 0.0, si = 0.0;
  for (unsigned idx = w * NT + threadIdx.x; idx < nn; idx += nwg * NT) {
    const unsigned i = idx / np, j = idx - i * np;
    double b = 0.0, c = 0.0, x = 0.0, bi = 0.0, xi = 0.0;
    if (i < n && j < n) {
      const long k = (long)i * n + j;
      b = half * a.S[Z ? 2 * k : k];
      c = (i == j ? 3.0 : 0.0) - b;
      x = 0.5 * c;
      const double d = (i == j ? 1.0 : 0.0) - x;
      if (Z) {
        bi = half * a.S[2 * k + 1];
        xi = -0.5 * bi;
        if (!a.late) {
          a.T[2 * k] = x;
          a.T[2 * k + 1] = xi;
        }
        const bool ok = isfinite(d) && isfinite(xi);
        s = ok ? fma(d, d, s) : nan;
        si = ok ? fma(xi, xi, si) : nan;
      } else {
        if (!a.late) a.T[k] = x;
        s = (isfinite(d) || n == 1) ? fma(d, d, s) : nan;
      }
    }
    a.B[0][idx] = b;
    a.C[idx] = c;
    a.A[1][idx] = x;
    if (Z) {
      a.B[0][a.zs + idx] = bi;
      a.C[a.zs + idx] = -bi;
      a.A[1][a.zs + idx] = xi;
    }
  }
  s = block_sum(s, red);
  if (Z) si = block_sum(si, red);
  if (threadIdx.x == 0) {
    a.partial[w] = s;
    if (Z) a.partial[nwg + w] = si;
    if (w == 0) {
      a.rep->iterations = 0;
      a.rep->done = 0;
      a.rep->status = OA_SUCCESS;
      a.rep->pad = 0;
      a.rep->error = 0.0;
    }
  }
}

// Sum of npart partial sums by the first 256 threads.
__device__ __forceinline__ double partial_sum(const double *p, int npart, double *red) {
  double s = 0.0;
  if (threadIdx.x < NT)
#pragma unroll 4
    for (int i = threadIdx.x; i < npart; i += NT) s += p[i];
  return block_sum(s, red);
}

// Residual of the iteration `it` (1-based) from its npart partial sums (Z: of
// either part); returns whether the loop ends there.  `writer` stores the
// report.  The complex rule is the reference's Re sum (dA)^2, NaN where that is
// negative, or sum |dA|^2 (modulus).
template <bool Z>
__device__ __forceinline__ bool ns_update(const oa_ns_args &a, int it, int npart, bool writer,
                                          double *red, double &err) {
  double s = partial_sum(a.partial, npart, red);
  if (Z) {
    const double si = partial_sum(a.partial + npart, npart, red);
    s = a.modulus ? s + si : s - si;
  }
  err = sqrt(s / ((double)a.n * (double)a.n));
  const bool done = !(err > a.tol && it < a.maxit);
  if (writer && threadIdx.x == 0) {
    oa_ns_report r;
    r.iterations = it;
    r.done = done ? 1 : 0;
    r.status = (done && it >= a.maxit) ? OA_ERR_NOT_CONVERGED : OA_SUCCESS;
    r.pad = 0;
    r.error = err;
    *a.rep = r;
    if (a.mirror) {
      // host memory; `pad` is the word the host polls, stored when the rest
      // has arrived.  (A release at system scope would write back the whole L2;
      // these stores go through it, so waiting for them is enough, and the
      // clobber keeps the compiler from moving them.)
      __hip_atomic_store(&a.mirror->error, err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&a.mirror->status, r.status, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&a.mirror->done, r.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&a.mirror->iterations, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __hip_atomic_store(&a.mirror->pad, 2 * it + r.done, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  return done;
}

// Blocks of 32 rows of an S->T matrix of np rows: their squares share a partial
// sum of the residual.
__host__ __device__ __forceinline__ int ns_blocks(int np) { return cdiv(np, 32); }

// The partial sums of a tile's 32 x 32 blocks from the lanes' sums s[i * WN + j]
// over their four elements of block (i, j).  One tree for every tile: column
// pairs, eight columns each, the four row groups, the two halves of a 32 column
// span, the two 16 row blocks.  (PAIR lanes hold adjacent columns, other
// lanes one column of 16.)
template <class C>
__device__ __forceinline__ void ns_residual(const oa_ns_args &a, int part, int m0, int n0,
                                            const double (&s)[C::WM * C::WN], double *red) {
  constexpr bool PAIR = RowMap<C::WN, C::WC, false>::PAIR;
  static_assert(PAIR ? C::WN == 2 : C::WN == 1, "one column span per wave");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < C::WM; i++) {
    double x = PAIR ? s[i * C::WN] + s[i * C::WN + C::WN - 1] : s[i];
#pragma unroll
    for (int o = 1; o <= (PAIR ? 4 : 8); o <<= 1) x += __shfl_xor(x, o);
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    if (PAIR) x += __shfl_xor(x, 8);
    if (lane == 0) red[i * C::NW + w] = x;
  }
  __syncthreads();
  const int t = threadIdx.x, nb = ns_blocks(a.np);
  if (t < (C::BM / 32) * (C::BN / 32)) {
    const int rb = t / (C::BN / 32), cb = t % (C::BN / 32);
    // rows: block k = i * WR + wr of 16; columns: span wc, or the halves 2 cb, 2 cb + 1
    auto row = [&](int k) {
      const double *p = red + (k / C::WR) * C::NW + (k % C::WR) * C::WC;
      return PAIR ? p[cb] : p[2 * cb] + p[2 * cb + 1];
    };
    const double x = row(2 * rb) + row(2 * rb + 1);
    const int br = m0 / 32 + rb, bc = n0 / 32 + cb;
    if (br < nb && bc < nb) a.partial[(part * nb + br) * nb + bc] = x;
  }
  __syncthreads();  // red may be refilled
}

// Output tile `logical` of an NS_B1, NS_C or NS_PAIR launch after `it` iterations.
// `which` of the launch's products: 0 = B', 1 = A' of a pair; with Z the real
// and the imaginary part of each in turn (four real products in two sums).
template <class C, bool Z>
__device__ __forceinline__ void ns_gemm_body(const oa_ns_args &a, int mode, int it, int npart,
                                             int which, int logical, double *smem) {
  const int t = cdiv(a.np, C::BM);
  if (logical >= t * t) return;
  // one answer for the workgroup: during a C launch the first one stores the
  // report, and waves that saw it differently would go on to different items
  int ended = mode != NS_B1 && (a.rep->done || it > a.maxit);
  if (mode == NS_C) ended = __syncthreads_or(ended);
  if (ended) return;
  const int part = Z ? which & 1 : 0;
  const bool second = (Z ? which >> 1 : which) != 0;
  if (mode == NS_B1 || (mode == NS_C && it >= 2)) {
    double err;
    const bool done = ns_update<Z>(a, it, npart, logical == 0 && which == 0, smem, err);
    if (mode == NS_B1) {
      // S's identity product with a non-finite S is NaN everywhere (a complex
      // residual may also be NaN by its rule: then A' stands)
      bool bad = isnan(err);
      if (Z && bad) bad = isnan(partial_sum(a.partial, npart, smem));
      const double *x = a.A[1] + (part ? a.zs : 0);
      const bool put = bad || a.late;
      const int m0 = (logical % t) * C::BM, n0 = (logical / t) * C::BN;
      for (int e = threadIdx.x; put && e < C::BM * C::BN; e += C::NTHR) {
        const int m = m0 + e / C::BN, n = n0 + e % C::BN;
        if (m < a.n && n < a.n)
          a.T[Z ? 2 * ((long)m * a.n + n) + part : (long)m * a.n + n] =
              bad ? err : x[(long)m * a.np + n];
      }
    }
    if (done) return;
  }
  const int cur = it & 1, nxt = cur ^ 1;
  const double *X, *Y;
  double *O;
  ProbRegs P;
  P.alpha = 0.5;
  P.diag_add = 0.0;
  if (mode == NS_C) {
    X = a.A[cur]; Y = a.B[cur]; O = a.C;
    P.alpha = -1.0;
    P.diag_add = part ? 0.0 : 3.0;
  } else if (mode == NS_B1) {
    X = a.B[0]; Y = a.C; O = a.B[1];
  } else if (!second) {
    X = a.B[cur]; Y = a.C; O = a.B[nxt];
  } else {
    X = a.C; Y = a.A[cur]; O = a.A[nxt];
  }
  const long im = Z ? a.zs : 0;
  P.M = P.N = P.K = a.np;
  P.ldx = P.ldy = P.ldc = a.np;
  P.beta = 0.0;
  P.cw = 0;
  P.alpha_w = 0.0;
  P.X = X;
  P.Y = part ? Y + im : Y;
  P.C = part ? O + im : O;
  // re: Xr Yr - Xi Yi, im: Xr Yi + Xi Yr
  P.X1 = X + im;
  P.Y1 = part ? Y : Y + im;
  P.neg1 = part == 0;
  const bool res = mode == NS_PAIR && second;
  const double *old = part ? Y + im : Y;
  double s[C::WM * C::WN] = {};
  gemm_body<false, false, C, Z ? SEG_TWO : SEG_ONE>(P, logical, smem,
                                                    [&](int b, int m, int n, double x) {
    // the padding stays zero whatever the matrix holds: an infinity of a
    // diverging iterate times the zeros of the other operand's padding is NaN,
    // which the next product would carry into the matrix
    if (m >= a.n || n >= a.n) return 0.0;
    if (res) {
      const double d = old[(long)m * a.np + n] - x;
      s[b] = fma(d, d, s[b]);
      a.T[Z ? 2 * ((long)m * a.n + n) + part : (long)m * a.n + n] = x;
    }
    return x;
  });
  if (res)
    ns_residual<C>(a, part, (logical % t) * C::BM, (logical / t) * C::BN, s, smem);
}

template <bool Z>
__global__ __launch_bounds__(NT) void ns_init_kernel(oa_ns_args a) {
  __shared__ double red[NT / 64];
  ns_init_body<Z>(a, blockIdx.x, gridDim.x, red);
}

// A launch starts when the ones before it on the stream have ended.
__global__ void ns_mark_kernel(int *flag) {
  __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <class C, bool Z>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void ns_gemm_kernel(oa_ns_args a, int mode, int it, int npart) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  ns_gemm_body<C, Z>(a, mode, it, npart, blockIdx.y, xcd_logical(blockIdx.x, gridDim.x), smem);
}

// The same over many real instances (oa_ns_args tables): items are a.nwg INIT
// workgroups, or the output tiles of one problem (B1, C) or two (PAIR).
__global__ __launch_bounds__(NT) void ns_init_grouped(const oa_ns_args *__restrict__ t,
                                                      const int *__restrict__ prefix,
                                                      int count) {
  __shared__ double red[NT / 64];
  for_items(prefix[count], [&](int item) {
    const int i = group_find(prefix, count, item);
    ns_init_body<false>(t[i], item - prefix[i], t[i].nwg, red);
  });
}

template <class C>
__global__ __launch_bounds__(C::NTHR) __attribute__((amdgpu_waves_per_eu(C::WPE, C::WPE)))
void ns_gemm_grouped(const oa_ns_args *__restrict__ t, const int *__restrict__ prefix, int count,
                     int mode, int it) {
  __shared__ __attribute__((aligned(1024))) double smem[C::SMEM];
  for_items(prefix[count], [&](int item) {
    const int i = group_find(prefix, count, item);
    const oa_ns_args &a = t[i];
    const int tiles = cdiv(a.np, C::BM) * cdiv(a.np, C::BM), k = item - prefix[i];
    const int nb = ns_blocks(a.np);
    ns_gemm_body<C, false>(a, mode, it, mode == NS_B1 ? a.nwg : nb * nb, k / tiles, k % tiles,
                           smem);
  });
}

template <class K>
int grouped_grid(K kernel, int total, int threads = NT) {
  int per_cu = 1;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  static thread_local int cached_dev = -1, cached_cus = 256;
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev != cached_dev) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        cus > 0)
      cached_cus = cus;
    cached_dev = dev;
  }
  const int cap = cdiv(cached_cus * per_cu, 8) * 8;
  const int g = cdiv(max(total, 1), 8) * 8;
  return g < cap ? g : cap;
}

// The largest tile that still gives every CU its two workgroups (T128), then
// four (T64), then about one (T64W).  A ragged 128 tile costs almost a whole
// one (its shorter stages wait for their loads), a 64 tile's MFMAs 1.1 times
// as much: T psi at n = 301 (npw 20011) 161 us with T128, 142 with T64; n =
// 448 (40000) 555 / 523; n = 192 (30000) 106 / 79; but n = 384 (40000) 386 /
// 389; n = 777 (50021) 1946 / 2135; n = 96 (60000) 51 / 60.
enum TilePick { PICK_128, PICK_64, PICK_64W, PICK_32 };
// (t128, t64): tiles of the product; (all128, all64): those of the whole launch.
TilePick pick_tile(long t128, long t64, long all128, long all64) {
  const bool ragged = 40 * t128 > 11 * t64;  // 128^2 t128 > 1.1 * 64^2 t64
  if (all128 >= 512 && !ragged) return PICK_128;
  if (all64 >= 1024) return PICK_64;
  return all64 >= 192 ? PICK_64W : PICK_32;
}
long gemm_tiles(const oa_gemm_problem &p, int bm, int bn) {
  return (long)cdiv(p.M, bm) * cdiv(p.N, bn);
}

// Calls f(tile configuration).
template <class F>
void with_tile(TilePick t, F &&f) {
  switch (t) {
    case PICK_128: f(T128{}); break;
    case PICK_64: f(T64{}); break;
    case PICK_64W: f(T64W{}); break;
    case PICK_32: f(T32{}); break;
  }
}

template <bool TX, bool TY>
int launch_gemm(hipStream_t s, const oa_gemm_problem *p, int nprob, int *mark) {
  auto tiles = [&](int bm, int bn) {
    long t = 0;
    for (int i = 0; i < nprob; i++) t = max(t, gemm_tiles(p[i], bm, bn));
    return t;
  };
  const long t128 = tiles(128, 128), t64 = tiles(64, 64);
  with_tile(pick_tile(t128, t64, t128 * nprob, t64 * nprob), [&](auto c) {
    typedef decltype(c) C;
    hipLaunchKernelGGL((gemm_f64_kernel<TX, TY, C>),
                       dim3((unsigned)((tiles(C::BM, C::BN) + 7) / 8 * 8), nprob),
                       dim3(C::NTHR), 0, s, p[0], p[nprob > 1 ? 1 : 0], mark);
  });
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

template <bool TX>
int launch_zback(hipStream_t s, const oa_gemm_problem &p, const double *Mi, bool neg) {
  const long t128 = gemm_tiles(p, 128, 128), t64 = gemm_tiles(p, 64, 64);
  with_tile(pick_tile(t128, t64, t128, t64), [&](auto c) {
    typedef decltype(c) C;
    hipLaunchKernelGGL((zback_f64_kernel<TX, C>),
                       dim3((unsigned)((gemm_tiles(p, C::BM, C::BN) + 7) / 8 * 8)), dim3(C::NTHR), 0,
                       s, p, Mi, neg ? 1 : 0);
  });
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

// Split-K plan for the plane-wave products.
struct OvlPlan {
  int BM, ntiles, nz_main, kchunk, nz;
  int kx0_slice;  // columns of a kx = 0 slice (z = 0), 0 for none
};

// A kx = 0 plane of at most this many columns is cleared in the first chunk's
// panels and half its product added in the reduce; a wider one is a z slice of
// its own, weighted there.
constexpr int KX0_ADD_MAX = 32;

// Split depth nz for ntiles output tiles of BM over K columns, of which the
// blocks inside the matrix (and above the diagonal) are the fraction `fill`.
// The chunks go to the 8 XCDs in equal contiguous ranges of w workgroups; of a
// range, 32 CUs x wpc are resident at once (wpc = 2 for BM = 128, whose 64 KB
// LDS footprints share a CU's 160 KB; 4 for BM = 64).  The cost of a depth:
//   MFMA time of a CU, 2 flops per output and column at 0.3 TF (6.5 ps):
//   whole rounds cost the work they hold (partial tiles save a quarter, at
//   BM = 64 half, of what they leave out), the last one a full tile's path;
//   few workgroups on a CU reach only part of its rate.
//   2 to 3 us a workgroup (first loads, partial tile).
//   16 bytes per element of the nz*ntiles partial tiles, partly in L2.
// Measured depths, 128 tiles: n = 1024, npw = 262144: 14 (one round) 9.57 ms,
// 35 9.60, 56 8.92, 71 9.05, 113 8.87; n = 512, npw = 65536: 25 0.685, 38
// 0.853, 51 (one round) 0.659, 102 0.675, 256 0.696.  64 tiles: n = 777, npw =
// 50021: 11 1.247, 22 1.195, 45 1.131, 90 1.136; n = 301, npw = 20011: 34 93
// us, 51 92, 68 89, 136 95; n = 128, npw = 8192: 85 19.7, 128 22.9.
// Chunks keep at least 8 BK stages.  The choice depends on (M, N, K) only, so
// workspace sizing and launch agree for any kx = 0 split.
int ovl_depth(int ntiles, int K, int BM, double fill) {
  const int nzmax = max(1, min(512, cdiv(K, 8 * BK)));
  const bool big = BM == 128;
  const int wpc = big ? 2 : 4, slots = 32 * wpc;
  const double lone = big ? 1.15 : 2.6, el = (double)BM * BM, start = big ? 3e6 : 2e6;
  const double f = 1.0 - (big ? 0.25 : 0.5) * (1.0 - fill);
  int best = 1;
  double best_cost = 0.0;
  for (int nz = 1; nz <= nzmax; nz++) {
    const int w = cdiv(ntiles * nz, 8), full = w / slots, rest = w % slots;
    const double last = rest > 0 ? fmax((double)cdiv(rest, 32), lone) : wpc * (1.0 - f);
    const double cost = cdiv(K, nz) * (wpc * full * f + last) * 6.5 * el + cdiv(w, 32) * start +
                        (double)nz * ntiles * el * 2.5;
    if (nz == 1 || cost < best_cost) { best = nz; best_cost = cost; }
  }
  return best;
}

// max_part_bytes > 0 caps the depth so that the partial tiles (a kx = 0 slice
// included, whatever its width) fit that many bytes; nz_main = 0 reports that
// even one chunk does not fit.
OvlPlan plan_ovl(int M, int N, int K, int kx0_end, bool sym, size_t max_part_bytes = 0) {
  OvlPlan pl;
  auto tiles = [&](int bm) {
    const int a = cdiv(M, bm), b = cdiv(N, bm);
    return sym ? a * (a + 1) / 2 : a * b;
  };
  const int t128 = tiles(128), t64 = tiles(64);
  // A partial 128 tile costs almost a whole one, the MFMAs of 64 tiles 1.1 to
  // 1.2 times as much.  Overlap with 128 / 64 tiles: n = 301 (npw 20011) 124 /
  // 92 us, n = 384 (40000) 261 / 234, n = 448 (40000) 410 / 306, n = 512
  // (65536) 657 / 666, n = 777 (50021) 1363 / 1267, n = 1024 (262144) 9.0 / 12.9
  // ms.  Lambda: 301 198 / 145, 384 386 / 390, 448 634 / 539, 777 2212 / 2452.
  const bool small = M < 256 && t128 < 16;
  pl.BM = (small || t64 * (sym ? 1.12 : 1.2) < t128 * 4) ? 64 : 128;
  pl.ntiles = pl.BM == 128 ? t128 : t64;
  const long bm = cdiv(M, 16), bn = cdiv(N, 16), bt = pl.BM / 16;
  const double fill = (double)(sym ? bm * (bm + 1) / 2 : bm * bn) / (pl.ntiles * bt * bt);
  int nz = ovl_depth(pl.ntiles, max(K, 1), pl.BM, fill);
  if (max_part_bytes > 0) {
    // counted in 128 tiles from M = 256 on (64 tiles never need more)
    const size_t per = (size_t)(small ? t64 * 4096 : t128 * 16384) * sizeof(double);
    const long fit = (long)(max_part_bytes / per) - (kx0_end > 0 ? 1 : 0);
    if (fit < 1) {
      pl.nz_main = 0;
      pl.kchunk = 0;
      pl.nz = 0;
      return pl;
    }
    if (nz > fit) nz = (int)fit;
  }
  // the chunk length comes from K: a slice never adds more than one z
  pl.kchunk = cdiv(cdiv(max(K, 1), nz), BK) * BK;
  pl.kx0_slice = kx0_end > KX0_ADD_MAX ? kx0_end : 0;
  pl.nz_main = max(1, cdiv(max(K - pl.kx0_slice, 1), pl.kchunk));
  pl.nz = pl.nz_main + (pl.kx0_slice > 0 ? 1 : 0);
  return pl;
}

// X[r][c] *= s over the leading ncols columns of each row: one thread per
// element, rows strided over the grid.
__global__ void scale_cols_kernel(int rows, int ncols, double *X, long ld, double scale) {
  const long total = (long)rows * ncols;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long)gridDim.x * blockDim.x) {
    double *p = X + (i / ncols) * ld + (i % ncols);
    *p *= scale;
  }
}

}  // namespace

int oa_launch_scale_cols(hipStream_t s, int rows, int ncols, double *X, long ld, double scale) {
  const long total = (long)rows * ncols;
  if (total <= 0) return OA_SUCCESS;
  long blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(scale_cols_kernel, dim3((unsigned)blocks), dim3(256), 0, s, rows, ncols, X,
                     ld, scale);
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_launch_gemm_f64(hipStream_t s, bool tx, bool ty, const oa_gemm_problem *p, int nprob,
                       int *mark) {
  if (nprob < 1 || nprob > 2) return OA_ERR_UNSUPPORTED;
  if (!tx && !ty) return launch_gemm<false, false>(s, p, nprob, mark);
  if (!tx && ty) return launch_gemm<false, true>(s, p, nprob, mark);
  if (tx && !ty) return launch_gemm<true, false>(s, p, nprob, mark);
  return launch_gemm<true, true>(s, p, nprob, mark);
}

int oa_launch_zback_f64(hipStream_t s, bool tx, int n, int K, const double *Mr, const double *Mi,
                        long ldm, bool neg, const double *psi, long ld, double alpha, double beta,
                        double *out, long ldo) {
  const oa_gemm_problem p{n, K, n, Mr, ldm, psi, ld, out, ldo, alpha, beta, 0.0};
  return tx ? launch_zback<true>(s, p, Mi, neg) : launch_zback<false>(s, p, Mi, neg);
}

size_t oa_overlap_f64_ws_bytes(int n, int K) {
  const OvlPlan pl = plan_ovl(n, n, K, 0, true);
  // a kx0 slice adds one z
  return (size_t)(pl.nz + 1) * pl.ntiles * pl.BM * pl.BM * sizeof(double) + 256;
}

size_t oa_ntsplit_f64_ws_bytes(int M, int N, int K) {
  const OvlPlan pl = plan_ovl(M, N, K, 0, false);
  return (size_t)pl.nz * pl.ntiles * pl.BM * pl.BM * sizeof(double) + 256;
}

// Workgroups of a plan's launches.
static int ovl_blocks(const OvlPlan &pl) {
  return (pl.kx0_slice > 0 ? cdiv(pl.ntiles, 8) * 8 : 0) + cdiv(pl.ntiles * pl.nz_main, 8) * 8;
}
static int reduce_blocks(const OvlPlan &pl) {
  return pl.ntiles * (pl.BM / 16) * (pl.BM / 16);
}

// C = alpha X Y^T by the plan, the leading kx0_end columns at half weight.
static int fill_ovl(const OvlPlan &pl, int M, int N, int K, const double *X, long ldx,
                    const double *Y, long ldy, int kx0_end, double alpha, double *C, long ldc,
                    double diag, double *maxdev, void *ws, size_t ws_bytes, oa_ovl_args *a) {
  if (pl.nz_main < 1 ||
      (size_t)pl.nz * pl.ntiles * pl.BM * pl.BM * sizeof(double) > ws_bytes)
    return OA_ERR_CAPACITY;
  *a = oa_ovl_args{X, ldx, Y, ldy, M, N, K, pl.kx0_slice, pl.nz_main, pl.kchunk, (double *)ws,
                   pl.BM, pl.nz, pl.kx0_slice > 0 ? 0 : kx0_end, alpha, C, ldc, diag,
                   reinterpret_cast<unsigned long long *>(maxdev)};
  return OA_SUCCESS;
}

template <class T, bool SYM, bool YJ>
static void launch_ovl_tile(hipStream_t s, const OvlPlan &pl, const oa_ovl_args &a) {
  hipLaunchKernelGGL((ovl_f64_kernel<T, SYM, YJ>), dim3(ovl_blocks(pl)), dim3(T::NTHR), 0, s, a);
  if (a.maxdev) hipLaunchKernelGGL(fill_u64_kernel, dim3(1), dim3(64), 0, s, a.maxdev, 0ull, 1);
  hipLaunchKernelGGL((ovl_reduce_kernel<T::BM, SYM>), dim3(reduce_blocks(pl)), dim3(1024), 0, s,
                     a);
}

// YJ: X (J Y)^T.
template <bool SYM, bool YJ>
static int launch_ovl(hipStream_t s, const OvlPlan &pl, int M, int N, int K, const double *X,
                      long ldx, const double *Y, long ldy, int kx0_end, double alpha, double *C,
                      long ldc, double diag, double *maxdev, void *ws, size_t ws_bytes) {
  oa_ovl_args a;
  const int st = fill_ovl(pl, M, N, K, X, ldx, Y, ldy, kx0_end, alpha, C, ldc, diag, maxdev, ws,
                          ws_bytes, &a);
  if (st) return st;
  if (pl.BM == 128) launch_ovl_tile<T128, SYM, YJ>(s, pl, a);
  else launch_ovl_tile<T64, SYM, YJ>(s, pl, a);
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_ovl_fill(int n, int K, const double *psi, long ld, int kx0_end, double alpha, double *S,
                void *ws, size_t ws_bytes, oa_ovl_args *a, int *blocks, int *rblocks) {
  const OvlPlan pl = plan_ovl(n, n, K, kx0_end, true);
  *blocks = ovl_blocks(pl);
  *rblocks = reduce_blocks(pl);
  return fill_ovl(pl, n, n, K, psi, ld, psi, ld, kx0_end, alpha, S, n, 0.0, nullptr, ws, ws_bytes,
                  a);
}

int oa_ovl_grouped(hipStream_t s, int bm, const oa_group &g) {
  const oa_ovl_args *t = reinterpret_cast<const oa_ovl_args *>(g.args);
  if (bm == 128)
    hipLaunchKernelGGL(ovl_f64_grouped<T128>, dim3(g.total), dim3(T128::NTHR), 0, s, t, g.prefix,
                       g.count);
  else
    hipLaunchKernelGGL(ovl_f64_grouped<T64>, dim3(g.total), dim3(T64::NTHR), 0, s, t, g.prefix,
                       g.count);
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_ovl_reduce_grouped(hipStream_t s, const oa_group &g) {
  hipLaunchKernelGGL(ovl_reduce_grouped, dim3(g.total), dim3(1024), 0, s,
                     reinterpret_cast<const oa_ovl_args *>(g.args), g.prefix, g.count);
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

void oa_gemm_f64_group(const oa_gemm_problem *p, int count, int *tile, int *blocks) {
  long all128 = 0, all64 = 0;
  for (int i = 0; i < count; i++) {
    all128 += gemm_tiles(p[i], 128, 128);
    all64 += gemm_tiles(p[i], 64, 64);
  }
  for (int i = 0; i < count; i++) {
    tile[i] = pick_tile(gemm_tiles(p[i], 128, 128), gemm_tiles(p[i], 64, 64), all128, all64);
    with_tile((TilePick)tile[i], [&](auto c) {
      typedef decltype(c) C;
      blocks[i] = (int)((gemm_tiles(p[i], C::BM, C::BN) + 7) / 8 * 8);
    });
  }
}

int oa_gemm_f64_grouped(hipStream_t s, int tile, const oa_group &g) {
  with_tile((TilePick)tile, [&](auto c) {
    typedef decltype(c) C;
    hipLaunchKernelGGL(gemm_f64_grouped<C>, dim3(g.total), dim3(C::NTHR), 0, s,
                       reinterpret_cast<const oa_gemm_problem *>(g.args), g.prefix, g.count);
  });
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_launch_overlap_f64(hipStream_t s, int n, int K, const double *psi, long ld, int kx0_end,
                          double alpha, double *S, double diag, double *maxdev, void *ws,
                          size_t ws_bytes) {
  return launch_ovl<true, false>(s, plan_ovl(n, n, K, kx0_end, true), n, n, K, psi, ld, psi, ld,
                                 kx0_end, alpha, S, n, diag, maxdev, ws, ws_bytes);
}

int oa_launch_overlap_f64_fit(hipStream_t s, int n, int K, const double *psi, long ld,
                              int kx0_end, double alpha, double *S, double diag,
                              double *maxdev, void *ws, size_t ws_bytes) {
  return launch_ovl<true, false>(s, plan_ovl(n, n, K, kx0_end, true, ws_bytes), n, n, K, psi, ld,
                                 psi, ld, kx0_end, alpha, S, n, diag, maxdev, ws, ws_bytes);
}

int oa_launch_ntsplit_f64(hipStream_t s, int M, int N, int K, const double *X, long ldx,
                          const double *Y, long ldy, double alpha, double *C, long ldc, void *ws,
                          size_t ws_bytes, bool yj) {
  const OvlPlan pl = plan_ovl(M, N, K, 0, false);
  if (yj)
    return launch_ovl<false, true>(s, pl, M, N, K, X, ldx, Y, ldy, 0, alpha, C, ldc, 0.0, nullptr,
                                   ws, ws_bytes);
  return launch_ovl<false, false>(s, pl, M, N, K, X, ldx, Y, ldy, 0, alpha, C, ldc, 0.0, nullptr,
                                  ws, ws_bytes);
}

int oa_launch_overlap_j_f64(hipStream_t s, int n, int K, const double *psi, long ld, double alpha,
                            double *C, void *ws, size_t ws_bytes) {
  return launch_ovl<true, true>(s, plan_ovl(n, n, K, 0, true), n, n, K, psi, ld, psi, ld, 0, alpha,
                                C, n, 0.0, nullptr, ws, ws_bytes);
}

// Workspace of one S->T: A[2], B[2], C and the partial sums.
static long ns_np(int n) { return (long)cdiv(n, 16) * 16; }
static int ns_init_wg(int n) {
  const long b = (ns_np(n) * ns_np(n) + 4 * NT - 1) / (4 * NT);
  return (int)(b > 256 ? 256 : b);
}
static size_t ns_partials(int n) {
  const size_t t = (size_t)ns_blocks((int)ns_np(n));
  return t * t > 256 ? t * t : 256;
}

size_t oa_ns_ws_bytes(int n, bool z) {
  return (z ? 2 : 1) * ((size_t)(5 * ns_np(n) * ns_np(n)) + ns_partials(n)) * sizeof(double) + 256;
}

void oa_ns_fill(int n, const double *S, int nspin, double tol, int maxit, double *T,
                oa_ns_report *rep, oa_ns_report *mirror, void *ws, oa_ns_args *a, bool z,
                int modulus) {
  const long nn = (z ? 2 : 1) * ns_np(n) * ns_np(n);
  double *base = (double *)ws;
  a->S = S;
  a->n = n;
  a->np = (int)ns_np(n);
  a->nspin = nspin;
  a->A[0] = base;
  a->A[1] = base + nn;
  a->B[0] = base + 2 * nn;
  a->B[1] = base + 3 * nn;
  a->C = base + 4 * nn;
  a->partial = base + 5 * nn;
  a->nwg = ns_init_wg(n);
  a->maxit = maxit;
  a->tol = tol;
  a->T = T;
  a->rep = rep;
  a->mirror = mirror;
  const uintptr_t s0 = (uintptr_t)S, t0 = (uintptr_t)T,
                  len = (uintptr_t)(z ? 2 : 1) * n * n * sizeof(double);
  a->late = s0 != t0 && s0 < t0 + len && t0 < s0 + len;
  a->zs = z ? nn / 2 : 0;
  a->modulus = modulus;
}

// Edge of the tile of an S->T launch of nprob products.
static int ns_tile(int np, int nprob) {
  const long t128 = (long)cdiv(np, 128) * cdiv(np, 128) * nprob;
  const long t64 = (long)cdiv(np, 64) * cdiv(np, 64) * nprob;
  return t128 >= 512 ? 128 : (t64 >= 192 ? 64 : 32);
}

static int launch_ns(hipStream_t s, const oa_ns_args &a, int mode, int it) {
  const int z = a.zs ? 2 : 1, nprob = z * (mode == NS_PAIR ? 2 : 1);
  const int nb = ns_blocks(a.np), npart = mode == NS_B1 ? a.nwg : nb * nb;
  const int edge = ns_tile(a.np, nprob);
  with_tile(edge == 128 ? PICK_128 : (edge == 64 ? PICK_64W : PICK_32), [&](auto c) {
    typedef decltype(c) C;
    const int t = cdiv(a.np, C::BM);
    // a C launch after the last iteration only writes the report
    const bool last = mode == NS_C && it >= a.maxit;
    const dim3 g(last ? 1 : cdiv(t * t, 8) * 8, last ? 1 : nprob);
    if (a.zs)
      hipLaunchKernelGGL((ns_gemm_kernel<C, true>), g, dim3(C::NTHR), 0, s, a, mode, it, npart);
    else
      hipLaunchKernelGGL((ns_gemm_kernel<C, false>), g, dim3(C::NTHR), 0, s, a, mode, it, npart);
  });
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_ns_begin(hipStream_t s, const oa_ns_args &a) {
  if (a.zs) hipLaunchKernelGGL(ns_init_kernel<true>, dim3(a.nwg), dim3(NT), 0, s, a);
  else hipLaunchKernelGGL(ns_init_kernel<false>, dim3(a.nwg), dim3(NT), 0, s, a);
  return launch_ns(s, a, NS_B1, 1);
}

int oa_ns_check(hipStream_t s, const oa_ns_args &a, int it) { return launch_ns(s, a, NS_C, it); }

int oa_ns_iterate(hipStream_t s, const oa_ns_args &a, int it) {
  return launch_ns(s, a, NS_PAIR, it);
}

int oa_ns_mark(hipStream_t s, int *flag) {
  hipLaunchKernelGGL(ns_mark_kernel, dim3(1), dim3(1), 0, s, flag);
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}

int oa_launch_s_to_t(hipStream_t s, int n, const double *S, int nspin, double tol, int maxit,
                     double *T, oa_ns_report *rep, void *ws) {
  oa_ns_args a;
  oa_ns_fill(n, S, nspin, tol, maxit, T, rep, nullptr, ws, &a);
  int st = oa_ns_begin(s, a);
  for (int it = 1; it < maxit && st == OA_SUCCESS; it++) {
    st = oa_ns_check(s, a, it);
    if (st == OA_SUCCESS) st = oa_ns_iterate(s, a, it);
  }
  if (st == OA_SUCCESS && maxit > 1) st = oa_ns_check(s, a, maxit);
  return st;
}

int oa_ns_items(int phase, int n, int wm) {
  if (phase == OA_NS_INIT) return ns_init_wg(n);  // has no tile
  const int t = cdiv((int)ns_np(n), 32 * wm);
  switch (phase) {
    case OA_NS_B1:
    case OA_NS_C: return t * t;
    case OA_NS_PAIR: return 2 * t * t;
  }
  return 0;
}

template <class C>
static void launch_ns_grouped(hipStream_t s, const oa_group &g, int mode, int it) {
  hipLaunchKernelGGL(ns_gemm_grouped<C>, dim3(grouped_grid(ns_gemm_grouped<C>, g.total, C::NTHR)),
                     dim3(C::NTHR), 0, s, reinterpret_cast<const oa_ns_args *>(g.args), g.prefix,
                     g.count, mode, it);
}

int oa_ns_grouped(hipStream_t s, int phase, int wm, int it, const oa_group &g) {
  if (g.count <= 0 || g.total <= 0) return OA_SUCCESS;
  if (phase == OA_NS_INIT) {
    hipLaunchKernelGGL(ns_init_grouped, dim3(grouped_grid(ns_init_grouped, g.total)), dim3(NT), 0,
                       s, reinterpret_cast<const oa_ns_args *>(g.args), g.prefix, g.count);
  } else {
    const int mode = phase == OA_NS_B1 ? NS_B1 : (phase == OA_NS_C ? NS_C : NS_PAIR);
    if (wm == 4) launch_ns_grouped<T128>(s, g, mode, it);
    else if (wm == 2) launch_ns_grouped<T64W>(s, g, mode, it);
    else return OA_ERR_UNSUPPORTED;
  }
  return hipPeekAtLastError() == hipSuccess ? OA_SUCCESS : OA_ERR_HIP;
}
