// Split-BF16 GEMM ("bf16x3") for the O(n^6) products, and the kernels that
// produce its operands.
//
// Operands are stored in HBM already split: x = hi + lo with hi = bf16(x),
// lo = bf16(x - hi), with K contiguous (A as [M][ld], B transposed as
// [N][ld]), sixteen hi and their sixteen lo side by side; K is zero-padded to
// a multiple of 32 so the inner loop needs no bounds checks along K.
// C = alpha * A.B + beta * C is accumulated in FP32 by
// v_mfma_f32_32x32x16_bf16 from lo*hi + hi*lo + hi*hi (in that order for
// every accumulator) and written as FP64.
//
// Tiling: a 512-thread workgroup (8 wave64s, two per SIMD) owns a 256x256
// tile of C, each wave a 128x64 quadrant (4x2 MFMA 32x32 blocks, 128 FP32
// accumulators per lane).  K advances in steps of 16 through a ring of five
// LDS stages of 32 KB, all of a CU's 160 KB; an LDS row holds the 64 bytes
// of the row's step as four 16-byte chunks, chunk c at slot
// c ^ ((row >> 2) & 3).  Steps go from HBM straight into LDS
// (global_load_lds_dwordx4: each lane fetches the chunk that belongs at its
// slot), up to five ahead of their use: an L2 miss takes longer than the
// 1.5 steps that the earlier two stages of 32 K gave it.  One barrier per
// step.  The fragment reads of the next step and the loads are issued
// between the MFMAs of the current one (fragments double-buffered in
// registers): issued together after the barrier, all eight waves queue for
// the LDS and the address unit while the matrix cores idle, and left to the
// compiler the reads are sunk to their uses.  Rows past M (N) read the last
// row: their products land in accumulators that are never stored.  A last
// tile of at most 192 rows or columns runs fewer MFMAs and comes after the
// whole tiles in the launch, to fill its last round.
//
// Bound: the matrix cores, by counters at n = 114 60% (ladders) to 67% (rings)
// busy on a CU at work and 50 to 55% over a launch, whose CUs work 82 to 86%
// of the time; the rest is the start and the stores of a tile, which one
// workgroup per CU does not overlap, and the last round of tiles.
// The five products of a residual, ms: n = 114 17.65 -> 15.84 (1.21 PFLOP/s
// of bf16 MFMAs; a library bf16 product reaches 1.36 at its power limit),
// n = 66 2.32 -> 2.15, against two stages of 32 K.  Tried: the same with
// reads and loads in one burst after the barrier 18.6 at n = 114; one wave
// per SIMD with 128x128 wave tiles was slower.
#include "ftcc_internal.h"

#include <algorithm>

namespace ftcc {
namespace {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));

constexpr int BM = 256, BN = 256, BK = 16;
constexpr int GROUP_M = 8;
constexpr int ROWB = 4 * BK;           // bytes per LDS row: 16 hi, 16 lo
constexpr int OPB = BM * ROWB;         // one operand of one stage: 16 KB
constexpr int STAGEB = 2 * OPB;        // A then B
constexpr int NST = 5;                 // stages of the ring
constexpr int NL = 4;                  // loads of a wave per K step
constexpr size_t LDS_BYTES = NST * (size_t)STAGEB;
// operand of s_waitcnt: at most vm vector loads and lgkm LDS reads (15: any)
// in flight
constexpr int wait_for(int vm, int lgkm) {
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8);
}
typedef __attribute__((address_space(3))) void lds_void;

// One product of a grouped launch (the spin blocks of one O(n^6) product
// share C, alpha, beta and the batch; up to MAXP problems per launch).
constexpr int MAXP = 3;
struct SbProb {
  int M, N, Kp, tilesM, tilesN;
  int fullM, fullN;          // tiles before a short last row, column
  int full0, edge0;          // its first whole tile and edge tile
  const __bf16 *A;
  int64_t lda, sAb;
  const __bf16 *B;
  int64_t ldb, sBb;
  const int *rmap, *cmap;    // output scatter (nullptr: identity; -1 drops)
};
struct SbDev {
  int nprob, nb;
  int group_m;               // tile rows per band of the launch order
  int nfull;                 // whole tiles of the launch
  SbProb pr[MAXP];
  double *C;
  int64_t sCm, sCn, sCb;
  double alpha, beta;
};

// Workgroup -> (problem, batch, tile m, tile n).  Consecutive workgroup ids
// go to different XCDs, so each XCD first takes a contiguous run of the
// launch's whole tiles, in GROUP_M-row bands of a problem so that concurrent
// tiles share A/B panels, and then one of the edge tiles, which are shorter
// (see tile_product) and fill the last round of the CUs.
__device__ inline SbProb tile_of(const SbDev &p, int &bt, int &tm, int &tn) {
  const int nblk = gridDim.x, b = blockIdx.x, x = b % 8, j = b / 8;
  const int fq = p.nfull / 8, fr = p.nfull % 8;
  const int fn = fq + (x < fr ? 1 : 0), f0 = x * fq + min(x, fr);
  const int t0 = x * (nblk / 8) + min(x, nblk % 8);
  const bool whole = j < fn;
  const int lid = whole ? f0 + j : (t0 - f0) + (j - fn);
  SbProb pr = p.pr[0];
  for (int k = 1; k < MAXP; ++k)
    if (p.nprob > k && lid >= (whole ? p.pr[k].full0 : p.pr[k].edge0))
      pr = p.pr[k];
  const int local = lid - (whole ? pr.full0 : pr.edge0);
  const int fper = pr.fullM * pr.fullN;
  const int per = whole ? fper : pr.tilesM * pr.tilesN - fper;
  bt = local / per;
  const int t = local % per;
  if (whole) {
    const int span = p.group_m * pr.fullN;
    const int first_m = (t / span) * p.group_m;
    const int gsz = min(pr.fullM - first_m, p.group_m);
    tm = first_m + (t % span) % gsz;
    tn = (t % span) / gsz;
  } else {
    const int strip = (pr.tilesM - pr.fullM) * pr.tilesN;
    tm = t < strip ? pr.fullM : t - strip;
    tn = t < strip ? t : pr.fullN;
  }
  return pr;
}

// LDS slot of chunk c (0, 1: hi, 2, 3: lo, eight bf16 each) of row r: the
// sixteen lanes that read one chunk of sixteen rows hit distinct banks
__device__ inline int lds_slot(int row, int c) { return c ^ ((row >> 2) & 3); }

// One wave's share of a K step of one operand: rows [32w, 32w + 32) of the
// tile in two loads of sixteen rows x four chunks; the lane that lands at
// slot (lane & 3) of row r fetches the chunk stored there.  off: its byte
// offsets from the tile's first row, the same in every step (Off: 32 bits
// hold them for rows of less than 2^22 elements).
template <typename Off> struct Rows {
  const __bf16 *p;   // first row of the tile
  Off off[2];
};
template <typename Off>
__device__ inline Rows<Off> tile_rows(const __bf16 *p, int64_t ld, int row0,
                                      int rows, int wave, int lane) {
  Rows<Off> r;
  r.p = p + 2 * row0 * ld;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int rowl = wave * 32 + j * 16 + (lane >> 2);
    const int c = lds_slot(rowl, lane & 3);   // the map is an involution
    r.off[j] = (Off)min(rowl, rows - 1 - row0) * (Off)(4 * ld) + 16u * c;
  }
  return r;
}
// load q (0, 1: A, 2, 3: B) of K step t into a stage
template <typename Off>
__device__ inline void load_part(const Rows<Off> &A, const Rows<Off> &B,
                                 int q, int t, char *stage, int wave) {
  const Rows<Off> &r = q < 2 ? A : B;
  __builtin_amdgcn_global_load_lds(
      (const void *)((const char *)(r.p + (int64_t)t * (2 * BK)) +
                     r.off[q & 1]),
      (lds_void *)(stage + (q >> 1) * OPB +
                   (wave * 32 + (q & 1) * 16) * ROWB),
      16, 0, 0);
}

__device__ inline bf8_t lds_frag(const char *lds_op, int row, int c) {
  return *(const bf8_t *)(lds_op + row * ROWB + (lds_slot(row, c) << 4));
}

// blocks of 32 in n rows of a last tile
__host__ __device__ inline int edge_blocks(int n) { return (n + 31) / 32; }
// tiles before a last one of at most EDGE blocks
constexpr int EDGE = 6;
inline int full_tiles(int n, int tile) {
  const int r = n % tile;
  return r > 0 && edge_blocks(r) <= EDGE ? n / tile : (n + tile - 1) / tile;
}

// the fragments, hi and lo, of RT row and CT column blocks of one 16-deep K
// step (chunk c: 0 or 2, plus the lane's half)
template <int RT, int CT> struct Frag {
  bf8_t ah[RT], al[RT], bh[CT], bl[CT];
};
// fragment q of the 2 (RT + CT) of a step
template <int RT, int CT>
__device__ inline void read_frag(Frag<RT, CT> &f, int q, const char *stage,
                                 int wm, int wn, int li, int lg) {
  const int h = q & 1, b = q >> 1;
  if (b < CT) {
    const bf8_t v =
        lds_frag(stage + OPB, (wn * CT + b) * 32 + li, 2 * h + lg);
    if (h) f.bl[b] = v;
    else f.bh[b] = v;
  } else {
    const bf8_t v =
        lds_frag(stage, (wm * RT + b - CT) * 32 + li, 2 * h + lg);
    if (h) f.al[b - CT] = v;
    else f.ah[b - CT] = v;
  }
}
// The MFMAs of one K step, lo*hi + hi*lo + hi*hi in that order for every
// accumulator, two accumulators in turn; other(q), q < n, is what is issued
// between them.
template <int RT, int CT, typename Other>
__device__ __forceinline__ void mfma_step(f16_t (&acc)[RT][CT],
                                          const Frag<RT, CT> &f, int n,
                                          Other other) {
  constexpr int NA = RT * CT, G = (NA + 1) / 2;
  int done = 0;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int upto = ((g + 1) * n + G - 1) / G;
#pragma unroll
    for (int q = done; q < upto; ++q) other(q);
    done = upto;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int a = 2 * g; a < (2 * g + 2 < NA ? 2 * g + 2 : NA); ++a) {
        const int rt = a / CT, ct = a % CT;
        acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            t == 0 ? f.al[rt] : f.ah[rt], t == 1 ? f.bl[ct] : f.bh[ct],
            acc[rt][ct], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One tile of C, RT x CT blocks of 32x32 a wave at block row wm RT, column
// wn CT: 4x2 blocks on 2x4 waves for a whole tile; for a last tile with nr
// (nc) <= 6 blocks of rows (columns), nr x 1 blocks on 1x8 waves (1 x nc on
// 8x1), whose matrix work is nr / 8 of a whole tile's.
template <int RT, int CT, typename Off = unsigned>
__device__ __forceinline__ void tile_product(const SbDev &p, const SbProb &pr,
                                             int bt, int m0, int n0, char *lds,
                                             int wm, int wn) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 31, lg = lane >> 5;
  // the tile's output rows and columns after the scatter maps (-1: past
  // the end or dropped), one of them a thread, read here ahead of the loop
  const int t = threadIdx.x, e = t < BM ? m0 + t : n0 + t - BM;
  const int *map = t < BM ? pr.rmap : pr.cmap;
  const int mapped = e < (t < BM ? pr.M : pr.N) ? (map ? map[e] : e) : -1;
  const int nstep = pr.Kp / BK;   // even
  const Rows<Off> A =
      tile_rows<Off>(pr.A + 2 * bt * pr.sAb, pr.lda, m0, pr.M, wave, lane);
  const Rows<Off> B =
      tile_rows<Off>(pr.B + 2 * bt * pr.sBb, pr.ldb, n0, pr.N, wave, lane);

  f16_t acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // an empty K (a spin class without pairs) only writes beta * C
  constexpr int NF = 2 * (RT + CT);
  Frag<RT, CT> f0, f1;
  if (nstep > 0) {
#pragma unroll
    for (int s = 0; s < NST; ++s)
#pragma unroll
      for (int q = 0; q < NL; ++q)
        load_part(A, B, q, min(s, nstep - 1), lds + s * STAGEB, wave);
    __builtin_amdgcn_s_waitcnt(wait_for((NST - 1) * NL, 15));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < NF; ++q) read_frag(f0, q, lds, wm, wn, li, lg);
  }
  char *cur = lds;
  // step s: its fragments are in f, those of step s + 1 go to g
  auto step = [&](int s, const Frag<RT, CT> &f, Frag<RT, CT> &g) {
    // step s + 1 has landed (every wave's loads) and every wave holds its
    // fragments of step s, whose stage takes step s + NST.  Past the last
    // step that one is loaded again, into stages that are not read any
    // more, which keeps the count of loads in flight constant.
    __builtin_amdgcn_s_waitcnt(wait_for((NST - 2) * NL, 0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    char *const nxt =
        cur == lds + (NST - 1) * STAGEB ? lds : cur + STAGEB;
    const int ahead = min(s + NST, nstep - 1);
    mfma_step(acc, f, NF + NL, [&](int q) {
      // reads and loads in turn, then what is left of either (NF >= NL)
      if (q < 2 * NL && (q & 1)) load_part(A, B, q >> 1, ahead, cur, wave);
      else read_frag(g, q < 2 * NL ? q >> 1 : q - NL, nxt, wm, wn, li, lg);
    });
    cur = nxt;
  };
  for (int s = 0; s < nstep; s += 2) {
    step(s, f0, f1);
    step(s + 1, f1, f0);
  }
  // no load may still be writing LDS when the maps take its place
  __builtin_amdgcn_s_waitcnt(wait_for(0, 0));
  __syncthreads();
  int *const emap = (int *)lds;   // rows, then columns
  emap[t] = mapped;
  __syncthreads();

  // lane holds column li, rows 8*(v/4) + 4*lg + v%4 of each 32x32 block.
  // Per block, the reads of C (beta != 0) are unconditional (a dropped
  // element reads element 0) and every value is formed before the first
  // store: reads or stores under divergent branches make the compiler wait
  // for all outstanding memory operations before each store.
  double *C = p.C + bt * p.sCb;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int cc = emap[BM + (wn * CT + ct) * 32 + li];
      int64_t off[16];
      double res[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int rr =
            emap[(wm * RT + rt) * 32 + 8 * (v >> 2) + 4 * lg + (v & 3)];
        off[v] = (rr >= 0 && cc >= 0)
                     ? (int64_t)rr * p.sCm + (int64_t)cc * p.sCn
                     : (int64_t)-1;
        res[v] = p.alpha * (double)acc[rt][ct][v];
      }
      if (p.beta != 0.0) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
          res[v] += p.beta * C[off[v] >= 0 ? off[v] : (int64_t)0];
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (off[v] >= 0) C[off[v]] = res[v];
    }
}

__global__ __launch_bounds__(512, 1) void sbgemm_kernel(SbDev p) {
  extern __shared__ char lds[];   // [NST stages][A | B][256 rows][64 B]
  int bt, tm, tn;
  const SbProb pr = tile_of(p, bt, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int wave = threadIdx.x >> 6;
  const int nr = tm < pr.fullM ? 8 : edge_blocks(pr.M - m0);
  const int nc = tn < pr.fullN ? 8 : edge_blocks(pr.N - n0);
#define FTCC_EDGE(NB)                                                      \
  if (nr <= nc) tile_product<NB, 1>(p, pr, bt, m0, n0, lds, 0, wave); \
  else tile_product<1, NB>(p, pr, bt, m0, n0, lds, wave, 0)
  switch (min(nr, nc)) {
    case 1: FTCC_EDGE(1); break;
    case 2: FTCC_EDGE(2); break;
    case 3: FTCC_EDGE(3); break;
    case 4: FTCC_EDGE(4); break;
    case 5:
    case 6: FTCC_EDGE(6); break;
    default:
      tile_product<4, 2>(p, pr, bt, m0, n0, lds, wave >> 2, wave & 3);
  }
#undef FTCC_EDGE
}

// The same for longer rows, whose offsets take 64 bits (whole tiles only:
// the launch has no edge tiles)
__global__ __launch_bounds__(512, 1) void sbgemm_long_kernel(SbDev p) {
  extern __shared__ char lds[];
  int bt, tm, tn;
  const SbProb pr = tile_of(p, bt, tm, tn);
  const int wave = threadIdx.x >> 6;
  tile_product<4, 2, uint64_t>(p, pr, bt, tm * BM, tn * BN, lds, wave >> 2,
                               wave & 3);
}

__device__ inline void split1(double v, __bf16 &hi, __bf16 &lo) {
  const float f = (float)v;
  hi = (__bf16)f;
  lo = (__bf16)(f - (float)hi);
}

// Destination writers of the gather kernels: split into (hi, lo) bf16, or
// plain FP64 or FP32 (the spin-blocked operands of those modes).
// store4 writes four consecutive elements (o a multiple of 4).
struct SplitOut {
  __bf16 *p;
  __device__ void operator()(int64_t o, double v) const {
    __bf16 h, l;
    split1(v, h, l);
    const int64_t q = SplitMat::place(o);
    p[q] = h;
    p[q + 16] = l;
  }
  __device__ void store4(int64_t o, const double v[4]) const {
    typedef __bf16 b4_t __attribute__((ext_vector_type(4)));
    b4_t h, l;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      __bf16 hk, lk;
      split1(v[k], hk, lk);
      h[k] = hk;
      l[k] = lk;
    }
    const int64_t q = SplitMat::place(o);
    *(b4_t *)(p + q) = h;
    *(b4_t *)(p + q + 16) = l;
  }
};
struct F32Out {
  float *p;
  __device__ void operator()(int64_t o, double v) const { p[o] = (float)v; }
  __device__ void store4(int64_t o, const double v[4]) const {
    typedef float f4_t __attribute__((ext_vector_type(4)));
    *(f4_t *)(p + o) =
        f4_t{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  }
};
struct F64Out {
  double *p;
  __device__ void operator()(int64_t o, double v) const { p[o] = v; }
  __device__ void store4(int64_t o, const double v[4]) const {
    typedef double d2_t __attribute__((ext_vector_type(2)));
    *(d2_t *)(p + o) = d2_t{v[0], v[1]};
    *(d2_t *)(p + o + 2) = d2_t{v[2], v[3]};
  }
};

// source row / column of destination index i: map[i] (-1: zero) or i itself
// below the bound n
__device__ inline int src_index(const int *map, int i, int n) {
  return map ? map[i] : (i < n ? i : -1);
}

// The source columns of columns c0, c0 + step, ... (NQ of them): -1 past W
// or where the map drops them.  The map test is hoisted (it is uniform) and
// the map reads are unconditional, so they are in flight together.
template <int NQ>
__device__ inline void map_cols(const int *map, int n, int W, int c0,
                                int step, int out[NQ]) {
  if (map) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = c0 + q * step;
      const int m = map[c < W ? c : 0];
      out[q] = c < W ? m : -1;
    }
  } else {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = c0 + q * step;
      out[q] = (c < W && c < n) ? c : -1;
    }
  }
}

// Sources of the gather kernels: value of the dense matrix at (slice b,
// row pair rr, column pair cc).  Plain: a strided FP64 tensor.
struct PlainSrc {
  const double *src;
  int64_t sr, sc, sb;
  __device__ double operator()(int64_t b, int rr, int cc) const {
    return src[b * sb + (int64_t)rr * sr + (int64_t)cc * sc];
  }
};
// Ring tensor W[e][m][b][j] (slice stride sb) of a spin-flip symmetric
// problem whose rows of an alpha e are stored (alpha runs [0, hv), [0, ho),
// beta runs after them), read by rows (b,j) and columns (e,m) (pair indices
// x * no + y): an element of a beta e is read from its image
// W[e - hv][fl m][fl b][fl j].
struct FlipRingSrc {
  const double *src;
  int64_t sb;
  int nv, no, hv, ho;
  __device__ double operator()(int64_t b, int rr, int cc) const {
    int e = cc / no, m = cc - e * no;
    int q = rr / no, l = rr - q * no;
    if (e >= hv) {
      e -= hv;
      m = m < ho ? m + ho : m - ho;
      q = q < hv ? q + hv : q - hv;
      l = l < ho ? l + ho : l - ho;
    }
    return src[b * sb + ((int64_t)e * no + m) * ((int64_t)nv * no) +
               (int64_t)q * no + l];
  }
};
// Amplitude-derived operands computed from t1 [V][O] and t2 [V][V][O][O]
// of each slice as they are gathered (nothing is materialised):
//   AMP_TAU_AB: rows (a,b), columns (i,j): tau = t2 + t1 t1 - t1 t1
//   AMP_TAU_IJ: rows (i,j), columns (a,b): the same tau
//   AMP_T2R:    rows (a,i), columns (e,m): t2[a,e,i,m]
//   AMP_ARING:  rows (b,j), columns (f,n): -1/2 t2[f,b,n,j] + t1[f,j] t1[b,n]
// (pair indices x * ny + y of the pair maps), one kind per instantiation (no
// branch on the kind inside the gathers' loads).
template <int KIND>
struct AmpSrc {
  const double *t1, *t2;
  int nv, no;
  __device__ double operator()(int64_t b, int rr, int cc) const {
    const int64_t VO = (int64_t)nv * no;
    const double *x1 = t1 + b * VO, *x2 = t2 + b * VO * VO;
    auto T2 = [&](int a, int e, int i, int m) {
      return x2[(((int64_t)a * nv + e) * no + i) * no + m];
    };
    auto T1 = [&](int a, int i) { return x1[(int64_t)a * no + i]; };
    if (KIND == AMP_TAU_AB || KIND == AMP_TAU_IJ) {
      const int ab = KIND == AMP_TAU_AB ? rr : cc;
      const int ij = KIND == AMP_TAU_AB ? cc : rr;
      const int a = ab / nv, bb = ab % nv, i = ij / no, j = ij % no;
      return T2(a, bb, i, j) + T1(a, i) * T1(bb, j) - T1(bb, i) * T1(a, j);
    } else if (KIND == AMP_T2R) {
      const int a = rr / no, i = rr % no, e = cc / no, m = cc % no;
      return T2(a, e, i, m);
    } else {   // AMP_ARING
      const int bb = rr / no, j = rr % no, f = cc / no, n = cc % no;
      return -0.5 * T2(f, bb, n, j) + T1(f, j) * T1(bb, n);
    }
  }
};

// dst[b][r][c] (row stride os) = src(b, R(r), C(c)) for r < R, c < W, zero
// where a map gives -1 (or, without maps, for c >= C); threads run along c
// (use when the source is contiguous along columns).
// Each thread takes four consecutive columns (W, os and db multiples of 4,
// destinations aligned to four elements).
template <typename Src, typename Out>
__global__ void gather_rows_kernel(Src src, const int *rmap, int R,
                                   const int *cmap, int C, int W, int64_t os,
                                   int64_t db, Out out, int nb) {
  const int W4 = W / 4;
  const int64_t per = (int64_t)R * W4;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
       idx < per * nb; idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = idx / per, e = idx % per;
    const int r = (int)(e / W4);
    const int c = 4 * (int)(e % W4);
    const int rr = src_index(rmap, r, R);
    int cc[4];
    map_cols<4>(cmap, C, W, c, 1, cc);
    double v[4];
    // branch-free loads (out of range reads element (0, 0), then zero)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double x = src(b, rr < 0 ? 0 : rr, cc[k] < 0 ? 0 : cc[k]);
      v[k] = (rr >= 0 && cc[k] >= 0) ? x : 0.0;
    }
    out.store4(b * db + (int64_t)r * os + c, v);
  }
}

// Same map through a GT x GT LDS tile: reads run along r (the source is
// contiguous along rows), writes along c, four columns per thread.  32x32
// tiles measured faster than 64x64 at n = 114 (24.2 against 30.0 ms of
// gathers per iteration: more workgroups in flight).
constexpr int GT = 32;
template <typename Src, typename Out>
__global__ void gather_transpose_kernel(Src src, const int *rmap, int R,
                                        const int *cmap, int C, int W,
                                        int64_t os, int64_t db, Out out) {
  __shared__ double tile[GT][GT + 1];
  const int b = blockIdx.z;
  const int r0 = blockIdx.y * GT, c0 = blockIdx.x * GT;
  const int tx = threadIdx.x % GT, ty = threadIdx.x / GT;   // 256 threads
  // a fixed trip count with branch-free loads (an out-of-range element
  // reads element (0, 0) and is replaced by zero): every row's map and
  // source loads are in flight together instead of one round trip each
  constexpr int NQ = GT / (256 / GT);
  const int r = r0 + tx;
  const int rr = r < R ? src_index(rmap, r, R) : -1;
  int cc[NQ];
  map_cols<NQ>(cmap, C, W, c0 + ty, 256 / GT, cc);
  double v[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const double x = src(b, rr < 0 ? 0 : rr, cc[q] < 0 ? 0 : cc[q]);
    v[q] = (rr >= 0 && cc[q] >= 0) ? x : 0.0;
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) tile[ty + q * (256 / GT)][tx] = v[q];
  __syncthreads();
  const int cq = threadIdx.x % (GT / 4), rq = threadIdx.x / (GT / 4);
  for (int i = rq; i < GT; i += 1024 / GT) {
    const int r = r0 + i, c = c0 + 4 * cq;
    if (r < R && c < W) {
      double v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = tile[4 * cq + k][i];
      out.store4(b * db + (int64_t)r * os + c, v);
    }
  }
}

template <typename Src, typename Out>
void gather_launch(Src src, bool along_rows, const int *rmap, int R,
                   const int *cmap, int C, int W, int64_t os, int64_t db,
                   Out out, int nb, hipStream_t s) {
  if ((int64_t)R * W == 0 || nb <= 0) return;
  require(W % 4 == 0 && os % 4 == 0 && db % 4 == 0,
          "gather: widths and strides must be multiples of 4");
  if (along_rows) {
    const int gx = (W + GT - 1) / GT, gy = (R + GT - 1) / GT;
    require(gy < 65536 && nb < 65536, "gather grid too large");
    hipLaunchKernelGGL((gather_transpose_kernel<Src, Out>), dim3(gx, gy, nb),
                       dim3(256), 0, s, src, rmap, R, cmap, C, W, os, db,
                       out);
  } else {
    const int64_t total = (int64_t)R * (W / 4) * nb;
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 1 << 20);
    hipLaunchKernelGGL((gather_rows_kernel<Src, Out>), dim3(blocks),
                       dim3(256), 0, s, src, rmap, R, cmap, C, W, os, db, out,
                       nb);
  }
  FTCC_CHECK_HIP(hipGetLastError());
}

// a plain source is read along rows when its row stride is the unit one
PlainSrc plain(const double *src, int64_t sr, int64_t sc, int64_t sb,
               bool &along_rows) {
  along_rows = (sr == 1 && sc != 1);
  return PlainSrc{src, sr, sc, sb};
}
// gather_launch over the amplitude source of `kind` (tau by (i,j) rows and
// aring by (b,j) rows are contiguous along rows)
template <typename Out>
void amp_launch(int kind, const double *t1, const double *t2, int nv, int no,
                const int *rmap, int R, const int *cmap, int W, int64_t os,
                int64_t db, Out out, int nb, hipStream_t s) {
  const bool ar = (kind == AMP_TAU_IJ || kind == AMP_ARING);
  switch (kind) {
    case AMP_TAU_AB:
      gather_launch(AmpSrc<AMP_TAU_AB>{t1, t2, nv, no}, ar, rmap, R, cmap, W,
                    W, os, db, out, nb, s);
      break;
    case AMP_TAU_IJ:
      gather_launch(AmpSrc<AMP_TAU_IJ>{t1, t2, nv, no}, ar, rmap, R, cmap, W,
                    W, os, db, out, nb, s);
      break;
    case AMP_T2R:
      gather_launch(AmpSrc<AMP_T2R>{t1, t2, nv, no}, ar, rmap, R, cmap, W, W,
                    os, db, out, nb, s);
      break;
    default:
      gather_launch(AmpSrc<AMP_ARING>{t1, t2, nv, no}, ar, rmap, R, cmap, W,
                    W, os, db, out, nb, s);
  }
}

}  // namespace

int64_t split_ld(int K) { return ((int64_t)K + 63) / 64 * 64; }

void split_convert(const double *src, int64_t sr, int64_t sc, int64_t sb,
                   int R, int C, const SplitMat &d, int nb, hipStream_t s) {
  require(d.ld >= C && d.ld % 32 == 0, "split operand leading dimension");
  if ((int64_t)R * C == 0) return;
  bool ar;
  const PlainSrc src_ = plain(src, sr, sc, sb, ar);
  gather_launch(src_, ar, nullptr, R, nullptr, C, (int)d.ld, d.ld, d.bstride,
                SplitOut{d.p}, nb, s);
}

void split_gather(const double *src, int64_t sr, int64_t sc, int64_t sb,
                  const int *rmap, int R, const int *cmap, int W,
                  const SplitMat &d, int nb, hipStream_t s) {
  require(d.ld % 32 == 0 && W <= d.ld, "split operand leading dimension");
  bool ar;
  const PlainSrc src_ = plain(src, sr, sc, sb, ar);
  gather_launch(src_, ar, rmap, R, cmap, W, W, d.ld, d.bstride,
                SplitOut{d.p}, nb, s);
}

void split_rows(const double *src, int64_t sr, int64_t sb, int R, int W,
                const SplitMat &d, int nb, hipStream_t s) {
  require(d.ld % 32 == 0 && W <= d.ld, "split operand leading dimension");
  gather_launch(PlainSrc{src, sr, 1, sb}, false, nullptr, R, nullptr, W, W,
                d.ld, d.bstride, SplitOut{d.p}, nb, s);
}

void amp_split_gather(int kind, const double *t1, const double *t2, int nv,
                      int no, const int *rmap, int R, const int *cmap, int W,
                      const SplitMat &d, int nb, hipStream_t s) {
  require(d.ld % 32 == 0 && W <= d.ld, "split operand leading dimension");
  require(rmap && cmap, "amplitude operands are gathered through pair maps");
  amp_launch(kind, t1, t2, nv, no, rmap, R, cmap, W, d.ld, d.bstride,
             SplitOut{d.p}, nb, s);
}

void amp_gather_plain(int kind, const double *t1, const double *t2, int nv,
                      int no, const int *rmap, int R, const int *cmap, int W,
                      int64_t os, void *dst, bool f32, int64_t db, int nb,
                      hipStream_t s) {
  require(rmap && cmap, "amplitude operands are gathered through pair maps");
  if (f32)
    amp_launch(kind, t1, t2, nv, no, rmap, R, cmap, W, os, db,
               F32Out{(float *)dst}, nb, s);
  else
    amp_launch(kind, t1, t2, nv, no, rmap, R, cmap, W, os, db,
               F64Out{(double *)dst}, nb, s);
}

void flip_ring_gather(const double *src, int nv, int no, int hv, int ho,
                      int64_t sb, const int *rmap, int R, const int *cmap,
                      int W, const SplitMat *d, int64_t os, void *dst,
                      bool f32, int64_t db, int nb, hipStream_t s) {
  require(2 * hv == nv && 2 * ho == no, "flip gather needs equal spin halves");
  require(rmap && cmap, "flip gather reads through pair maps");
  const FlipRingSrc src_{src, sb, nv, no, hv, ho};
  if (d) {
    require(d->ld % 32 == 0 && W <= d->ld, "split operand leading dimension");
    gather_launch(src_, true, rmap, R, cmap, W, W, d->ld, d->bstride,
                  SplitOut{d->p}, nb, s);
  } else if (f32) {
    gather_launch(src_, true, rmap, R, cmap, W, W, os, db,
                  F32Out{(float *)dst}, nb, s);
  } else {
    gather_launch(src_, true, rmap, R, cmap, W, W, os, db,
                  F64Out{(double *)dst}, nb, s);
  }
}

void gather_plain(const double *src, int64_t sr, int64_t sc, int64_t sb,
                  const int *rmap, int R, const int *cmap, int W, int64_t os,
                  void *dst, bool f32, int64_t db, int nb, hipStream_t s) {
  bool ar;
  const PlainSrc src_ = plain(src, sr, sc, sb, ar);
  if (f32)
    gather_launch(src_, ar, rmap, R, cmap, W, W, os, db,
                  F32Out{(float *)dst}, nb, s);
  else
    gather_launch(src_, ar, rmap, R, cmap, W, W, os, db,
                  F64Out{(double *)dst}, nb, s);
}

void sbgemm_grouped(int nprob, const SbProblem *prob, int nb, double alpha,
                    double beta, double *C, int64_t sCm, int64_t sCn,
                    int64_t sCb, hipStream_t s) {
  require(nprob >= 1 && nprob <= MAXP, "1 to 3 problems per grouped launch");
  static std::once_flag attr, attr_long;
  set_max_lds_once(attr, (const void *)sbgemm_kernel, (int)LDS_BYTES);
  set_max_lds_once(attr_long, (const void *)sbgemm_long_kernel,
                   (int)LDS_BYTES);
  // band height of the launch order (FTCC_SB_GROUP_M tunes it)
  static const int group_m = [] {
    const char *e = getenv("FTCC_SB_GROUP_M");
    const int v = e ? atoi(e) : GROUP_M;
    return v >= 1 && v <= 64 ? v : GROUP_M;
  }();
  SbDev p;
  p.nb = nb;
  p.group_m = group_m;
  p.C = C;
  p.sCm = sCm;
  p.sCn = sCn;
  p.sCb = sCb;
  p.alpha = alpha;
  p.beta = beta;
  p.nprob = 0;
  int64_t tiles = 0, whole = 0, ld = 0;
  for (int k = 0; k < nprob; ++k)
    ld = std::max(ld, std::max(prob[k].A.ld, prob[k].B.ld));
  // a tile's rows beyond 32-bit byte offsets
  const bool far = ld >= (1LL << 32) / (4 * BM);
  for (int k = 0; k < nprob; ++k) {
    const SbProblem &q = prob[k];
    if (q.M <= 0 || q.N <= 0) continue;
    require(q.A.ld % 32 == 0 && q.B.ld % 32 == 0 && q.A.ld >= q.K &&
                q.B.ld >= q.K,
            "split operands need K padded to 32");
    SbProb &d = p.pr[p.nprob++];
    d.M = q.M;
    d.N = q.N;
    d.Kp = (int)((q.K + 31) / 32 * 32);
    d.tilesM = (q.M + BM - 1) / BM;
    d.tilesN = (q.N + BN - 1) / BN;
    d.fullM = far ? d.tilesM : full_tiles(q.M, BM);
    d.fullN = far ? d.tilesN : full_tiles(q.N, BN);
    d.full0 = (int)whole;
    d.edge0 = (int)(tiles - whole);
    d.A = q.A.p;
    d.lda = q.A.ld;
    d.sAb = q.A.bstride;
    d.B = q.B.p;
    d.ldb = q.B.ld;
    d.sBb = q.B.bstride;
    d.rmap = q.rmap;
    d.cmap = q.cmap;
    tiles += (int64_t)d.tilesM * d.tilesN * nb;
    whole += (int64_t)d.fullM * d.fullN * nb;
  }
  if (p.nprob == 0 || nb <= 0) return;
  require(tiles < (1LL << 31), "too many GEMM tiles");
  p.nfull = (int)whole;
  hipLaunchKernelGGL(far ? sbgemm_long_kernel : sbgemm_kernel,
                     dim3((unsigned)tiles), dim3(512), LDS_BYTES, s, p);
  FTCC_CHECK_HIP(hipGetLastError());
}

void sbgemm(int M, int N, int K, int nb, double alpha, const SplitMat &A,
            const SplitMat &B, double beta, double *C, int64_t sCm,
            int64_t sCn, int64_t sCb, hipStream_t s, const int *rmap,
            const int *cmap) {
  if (M <= 0 || N <= 0 || nb <= 0) return;
  SbProblem q{M, N, K, A, B, rmap, cmap};
  sbgemm_grouped(1, &q, nb, alpha, beta, C, sCm, sCn, sCb, s);
}

}  // namespace ftcc
