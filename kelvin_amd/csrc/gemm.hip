// Batched strided GEMM on the CDNA4 matrix cores.
//
// One workgroup = 4 wave64s computes a tile of C of 128x128 to 64x64; each
// wave owns a quadrant as 16x16 MFMA blocks.  K advances in slabs of 16 staged
// through LDS (the largest tile double buffered, one barrier per slab) with
// the next slab prefetched into registers while the current one feeds the
// MFMAs.  Tile and splits of K: plan_of.  A launch takes up to GEMM_GROUP
// products (the spin blocks of a contraction), and products that add into
// one output leave partial sums for one reduction.
//
// LDS holds both operands "K-inner": As[m][k], Bs[n][k], rows padded so the
// 16 lanes that share a k-group hit distinct banks.  Inside a slab the
// physical k index used by lane group g (= lane/16) in MFMA step s is 4g+s, so
// each lane fetches its four k values for the four MFMA steps with one
// 128-bit (FP32) or two 128-bit (FP64) LDS reads; A and B use the same map, so
// the contraction is unchanged.
//
// Global loads are scalar and coalesced along whichever operand dimension is
// contiguous in memory (template flags), so every stride pattern is legal and
// the common layouts (A k-contiguous or m-contiguous, B n-contiguous or
// k-contiguous) stream whole cache lines.
//
// Precisions: FP64 (v_mfma_f64_16x16x4_f64) and FP32 (v_mfma_f32_16x16x4_f32,
// FP64 operands rounded to FP32 on load).  Split-BF16 products run in
// sbgemm.hip on operands split ahead of time.
//
// The output may be scattered through row and column maps (spin-blocked
// products write their blocks straight into the caller's layout).
#include "ftcc_internal.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace ftcc {
namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef double d2_t __attribute__((ext_vector_type(2)));

constexpr int BK = 16, NT = 256;

// Output tile: 128x128, 128x64, 64x128 or 64x64
struct Tile {
  int m, n;
};

struct GemmDev {
  int M, N, K, nb1, nb2, splits, kchunk, tilesM, tilesN;
  int m_inner;               // tile rows vary fastest (fewer of them)
  double alpha, beta;
  const double *A;
  int64_t sAm, sAk, sA1, sA2;
  const double *B;
  int64_t sBk, sBn, sB1, sB2;
  double *C;
  int64_t sCm, sCn, sC1, sC2;
  // [R][nb1 * nb2][M][N] when R partial sums make up C, this product's
  // splits being rbase, rbase + 1, ... (nullptr: C is written directly)
  double *partial;
  int rbase, R;
  const int *rmap, *cmap;   // output scatter (nullptr: identity)
  const double *D;          // addend gamma*D laid out like C (or nullptr)
  double gamma;
  int64_t sDm, sDn, sD1, sD2;
  // rows m = (m0*M1 + m1)*M2 + m2 and columns likewise (one index: M1 = 1,
  // M2 = 2^30); the strides above belong to the innermost index
  int M1, M2, N1, N2;
  int64_t sAm0, sAm1, sCm0, sCm1, sDm0, sDm1;
  int64_t sBn0, sBn1, sCn0, sCn1, sDn0, sDn1;
  int K1, K2;                // K levels (kernels instantiated with KL)
  int64_t sAk0, sAk1, sBk0, sBk1;
  // optional map of one row level and one column level (level 0, 1 or 2;
  // -1: none): that level's index x becomes map[x] before the strides
  const int *mmap, *nmap;
  int mlvl, nlvl;
};

// Up to GEMM_GROUP products in one launch: the spin blocks of a contraction,
// each a product of a few tiles.  Launched one by one, the sixty of a step
// at n = 38 took 10 to 25 us each whatever their size.
struct GemmGroup {
  int n;
  int tile0[GEMM_GROUP];     // first workgroup of each product
  GemmDev pr[GEMM_GROUP];
};

struct Lvl {
  int x0, x1, x2;
};
__device__ inline Lvl map_level(Lvl l, const int *map, int lvl) {
  if (lvl == 0) l.x0 = map[l.x0];
  else if (lvl == 1) l.x1 = map[l.x1];
  else if (lvl == 2) l.x2 = map[l.x2];
  return l;
}
__device__ inline Lvl levels(int x, int n1, int n2) {
  Lvl l;
  l.x2 = x % n2;
  const int t = x / n2;
  l.x1 = t % n1;
  l.x0 = t / n1;
  return l;
}
__device__ inline int64_t at(const Lvl &l, int64_t s0, int64_t s1,
                             int64_t s2) {
  return l.x0 * s0 + l.x1 * s1 + l.x2 * s2;
}

template <typename T> struct Mma;
template <> struct Mma<double> {
  using acc_t = d4_t;
  static constexpr int LDK = BK + 2;   // 36-dword rows: conflict-free reads
  // output element v of lane group lg sits in row lg + 4v of the 16x16 block
  __device__ static int crow(int lg, int v) { return lg + 4 * v; }
  __device__ static acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<float> {
  using acc_t = f4_t;
  static constexpr int LDK = BK + 4;   // 20-dword rows: conflict-free reads
  // output element v of lane group lg sits in row 4*lg + v of the block
  __device__ static int crow(int lg, int v) { return 4 * lg + v; }
  __device__ static acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// The flat block index regrouped per XCD: workgroups are dispatched to the
// eight XCDs round robin and each XCD has its own L2; the hardware ids x,
// x + 8, x + 16, ... of XCD x take a contiguous range of tiles (a bijection
// on [0, gridDim.x)).
__device__ inline int64_t xcd_block() {
  const int64_t G = gridDim.x, hw = blockIdx.x;
  const int64_t q8 = G / 8, r8 = G % 8, x = hw % 8, loc = hw / 8;
  return x < r8 ? x * (q8 + 1) + loc : r8 * (q8 + 1) + (x - r8) * q8 + loc;
}
// Decode a product's block into (tile n, tile m, split, b2, b1), the tiles
// along the dimension with fewer of them innermost: those tiles share one
// panel of the operand with more panels, which is then read from HBM once
// instead of once per tile row (an O(n^5) term of 456 x 185193 x 57 read
// 1.72 GB with columns innermost against 0.84 GB of distinct data).
struct BlockPos {
  int tn, tm, ks, b1, b2;
};
__device__ inline BlockPos decode(const GemmDev &p, int bid) {
  BlockPos q;
  if (p.m_inner) {
    q.tm = bid % p.tilesM;
    bid /= p.tilesM;
    q.tn = bid % p.tilesN;
    bid /= p.tilesN;
  } else {
    q.tn = bid % p.tilesN;
    bid /= p.tilesN;
    q.tm = bid % p.tilesM;
    bid /= p.tilesM;
  }
  q.ks = bid % p.splits;
  bid /= p.splits;
  q.b2 = bid % p.nb2;
  q.b1 = bid / p.nb2;
  return q;
}

// Element offsets of the tile's rows of A and columns of B, one table entry
// per row/column of the tile (-1 past the end), kept in LDS so they hold no
// registers through the K loop.
template <int TM, int TN>
__device__ inline void tile_offsets(const GemmDev &p, int m0, int n0,
                                    int64_t *aoff, int64_t *boff) {
  const int t = threadIdx.x;
  if (t < TM) {
    const int m = m0 + t;
    aoff[t] = m < p.M ? at(map_level(levels(m, p.M1, p.M2), p.mmap, p.mlvl),
                           p.sAm0, p.sAm1, p.sAm)
                      : -1;
  } else if (t < TM + TN) {
    const int n = n0 + t - TM;
    boff[t - TM] =
        n < p.N ? at(map_level(levels(n, p.N1, p.N2), p.nmap, p.nlvl),
                     p.sBn0, p.sBn1, p.sBn)
                : -1;
  }
}

// One K slab (16 deep) of the TM-row A tile and the TN-column B tile: each
// of the 256 threads loads TM/16 values of A and TN/16 of B.  Along the
// contiguous index: m = t % TM, k = t / TM + (256 / TM) r; otherwise
// m = t / 16 + 16 r, k = t % 16.
// KL (K over several indices, both operands K-fastest): every load of a
// thread shares k = k0 + t % 16, decoded once per slab.
template <typename T, bool A_MFAST, bool B_NFAST, int TM, int TN, bool KL>
__device__ inline void load_slab(const GemmDev &p, const double *A,
                                 const double *B, const int64_t *aoff,
                                 const int64_t *boff, int k0, int kend,
                                 double ra[TM / 16], double rb[TN / 16]) {
  static_assert(!KL || (!A_MFAST && !B_NFAST), "K levels need K-fast loads");
  const int t = threadIdx.x;
  int64_t ka = 0, kb = 0;
  bool kin = true;
  if (KL) {
    const int k = k0 + (t & 15);
    kin = k < kend;
    const Lvl l = levels(kin ? k : 0, p.K1, p.K2);
    ka = at(l, p.sAk0, p.sAk1, p.sAk);
    kb = at(l, p.sBk0, p.sBk1, p.sBk);
  }
#pragma unroll
  for (int r = 0; r < TM / 16; ++r) {
    const int64_t off = aoff[A_MFAST ? (t % TM) : (t >> 4) + 16 * r];
    double v = 0.0;
    if (KL) {
      if (off >= 0 && kin) v = A[off + ka];
    } else {
      const int k = A_MFAST ? k0 + t / TM + (NT / TM) * r : k0 + (t & 15);
      if (off >= 0 && k < kend) v = A[off + (int64_t)k * p.sAk];
    }
    ra[r] = v;
  }
#pragma unroll
  for (int r = 0; r < TN / 16; ++r) {
    const int64_t off = boff[B_NFAST ? (t % TN) : (t >> 4) + 16 * r];
    double v = 0.0;
    if (KL) {
      if (off >= 0 && kin) v = B[kb + off];
    } else {
      const int k = B_NFAST ? k0 + t / TN + (NT / TN) * r : k0 + (t & 15);
      if (off >= 0 && k < kend) v = B[(int64_t)k * p.sBk + off];
    }
    rb[r] = v;
  }
}

template <typename T, bool A_MFAST, bool B_NFAST, int TM, int TN>
// (the prefetched values stay FP64 until here, so that the FP32 form's
// rounding does not wait for the loads right where they are issued)
__device__ inline void store_slab(T *As, T *Bs, const double ra[TM / 16],
                                  const double rb[TN / 16]) {
  constexpr int LDK = Mma<T>::LDK;
  const int t = threadIdx.x;
#pragma unroll
  for (int r = 0; r < TM / 16; ++r) {
    if (A_MFAST)
      As[(t % TM) * LDK + t / TM + (NT / TM) * r] = (T)ra[r];
    else
      As[((t >> 4) + 16 * r) * LDK + (t & 15)] = (T)ra[r];
  }
#pragma unroll
  for (int r = 0; r < TN / 16; ++r) {
    if (B_NFAST)
      Bs[(t % TN) * LDK + t / TN + (NT / TN) * r] = (T)rb[r];
    else
      Bs[((t >> 4) + 16 * r) * LDK + (t & 15)] = (T)rb[r];
  }
}

template <typename T>
__device__ inline void load4(const T *src, T out[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) out[s] = src[s];
}

// TM x TN output tile per workgroup (128x128 down to 64x64): the four
// waves form a 2x2 grid, each owning (TM/2) x (TN/2) as RT x CT MFMA blocks.
template <typename T, bool A_MFAST, bool B_NFAST, int TM, int TN, bool KL>
__global__ __launch_bounds__(NT, 2) void gemm_mfma_kernel(GemmGroup grp) {
  using acc_t = typename Mma<T>::acc_t;
  constexpr int LDK = Mma<T>::LDK;
  constexpr int RT = TM / 32, CT = TN / 32;
  // the 128x128 tile is register-bound at two workgroups per CU and double
  // buffers its slabs; the narrow tiles single-buffer so that three
  // workgroups fit the LDS (two barriers per slab)
  constexpr bool DB = (TM == 128 && TN == 128);
  constexpr int NBUF = DB ? 2 : 1;
  static_assert(TM + TN <= NT, "one offset-table entry per thread");
  __shared__ T As[NBUF][TM * LDK];
  __shared__ T Bs[NBUF][TN * LDK];
  __shared__ int64_t aoff[TM], boff[TN], drow[TM], dcol[TN];

  const int64_t bid = xcd_block();
  int item = 0;
  for (int k = 1; k < grp.n; ++k)
    if (bid >= grp.tile0[k]) item = k;
  const GemmDev &p = grp.pr[item];
  const BlockPos q = decode(p, (int)(bid - grp.tile0[item]));
  const double *A = p.A + q.b1 * p.sA1 + q.b2 * p.sA2;
  const double *B = p.B + q.b1 * p.sB1 + q.b2 * p.sB2;
  const int m0 = q.tm * TM, n0 = q.tn * TN;
  const int kbeg = q.ks * p.kchunk;
  const int kend = min(p.K, kbeg + p.kchunk);
  const int nslab = (kend - kbeg + BK - 1) / BK;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lg = lane >> 4;

  acc_t acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  // FP32 sums run over at most FOLD_K of K and are added up in FP64 (not on
  // the wide tiles: plan_of)
  constexpr bool FOLD = sizeof(T) == 4 && TM == 64 && TN == 64;
  d4_t sum[FOLD ? RT : 1][FOLD ? CT : 1];
  if (FOLD) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) sum[i][j] = d4_t{0, 0, 0, 0};
  }
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[i][j][v] += (double)acc[i][j][v];
        acc[i][j] = acc_t{0, 0, 0, 0};
      }
  };

  double ra[TM / 16], rb[TN / 16];
  tile_offsets<TM, TN>(p, m0, n0, aoff, boff);
  __syncthreads();
  if (nslab > 0) {
    load_slab<T, A_MFAST, B_NFAST, TM, TN, KL>(p, A, B, aoff, boff, kbeg,
                                               kend, ra, rb);
    store_slab<T, A_MFAST, B_NFAST, TM, TN>(As[0], Bs[0], ra, rb);
  }
  __syncthreads();
  for (int s = 0; s < nslab; ++s) {
    const int buf = DB ? (s & 1) : 0;
    if (s + 1 < nslab)
      load_slab<T, A_MFAST, B_NFAST, TM, TN, KL>(p, A, B, aoff, boff,
                                                 kbeg + (s + 1) * BK, kend,
                                                 ra, rb);
    T a[RT][4], b[CT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      load4<T>(&As[buf][(wm * (TM / 2) + rt * 16 + li) * LDK + 4 * lg],
               a[rt]);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      load4<T>(&Bs[buf][(wn * (TN / 2) + ct * 16 + li) * LDK + 4 * lg],
               b[ct]);
    // single buffer: every wave has its fragments before the slab is
    // overwritten
    if (!DB) __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
          acc[rt][ct] = Mma<T>::op(a[rt][kk], b[ct][kk], acc[rt][ct]);
    if (FOLD && (s + 1) % (FOLD_K / BK) == 0) fold();
    if (s + 1 < nslab)
      store_slab<T, A_MFAST, B_NFAST, TM, TN>(As[DB ? buf ^ 1 : 0],
                                              Bs[DB ? buf ^ 1 : 0], ra, rb);
    __syncthreads();
  }

  if (FOLD) fold();
  auto result = [&](int rt, int ct, int v) {
    return FOLD ? sum[rt][ct][v] : (double)acc[rt][ct][v];
  };

  // epilogue: lane holds column li of each 16x16 block, rows Mma<T>::crow.
  // Output offsets of the tile's rows and columns (after the scatter maps;
  // -1 where dropped or past the end) go to LDS first, so the unrolled
  // stores below only look them up.  The K loop ended on a barrier, so the
  // offset tables of A and B are free.
  const bool direct = (p.partial == nullptr);
  double *C = p.C + q.b1 * p.sC1 + q.b2 * p.sC2;
  const double *D = p.D ? p.D + q.b1 * p.sD1 + q.b2 * p.sD2 : nullptr;
  int64_t *crow = aoff, *ccol = boff;
  if (direct) {
    const int t = threadIdx.x;
    if (t < TM) {
      const int row = m0 + t;
      const int rr = row < p.M ? (p.rmap ? p.rmap[row] : row) : -1;
      const Lvl l =
          map_level(levels(rr < 0 ? 0 : rr, p.M1, p.M2), p.mmap, p.mlvl);
      crow[t] = rr < 0 ? -1 : at(l, p.sCm0, p.sCm1, p.sCm);
      drow[t] = rr < 0 ? -1 : at(l, p.sDm0, p.sDm1, p.sDm);
    } else if (t < TM + TN) {
      const int col = n0 + t - TM;
      const int cc = col < p.N ? (p.cmap ? p.cmap[col] : col) : -1;
      const Lvl l =
          map_level(levels(cc < 0 ? 0 : cc, p.N1, p.N2), p.nmap, p.nlvl);
      ccol[t - TM] = cc < 0 ? -1 : at(l, p.sCn0, p.sCn1, p.sCn);
      dcol[t - TM] = cc < 0 ? -1 : at(l, p.sDn0, p.sDn1, p.sDn);
    }
    __syncthreads();
  }
  double *P = direct ? nullptr
                     : p.partial + ((int64_t)(p.rbase + q.ks) * p.nb1 * p.nb2 +
                                    q.b1 * p.nb2 + q.b2) *
                                       (int64_t)p.M * p.N;
  // Direct stores go one 16-row block at a time: all its reads of D and C
  // are issued before any store (a store may alias them as far as the
  // compiler knows, which would otherwise serialise every element on a
  // round trip to memory).
  // The reads of D and C are unconditional (a dropped element reads
  // element 0 and is not stored) and every value is formed before the first
  // store: with reads or stores under divergent branches the compiler can
  // no longer count which memory operations are outstanding and waits for
  // all of them before each store, serialising the stores one round trip
  // at a time.
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    if (direct) {
      int64_t oc[CT][4];
      double res[CT][4];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int lc = wn * (TN / 2) + ct * 16 + li;
          const int lr = wm * (TM / 2) + rt * 16 + Mma<T>::crow(lg, v);
          const bool ok = crow[lr] >= 0 && ccol[lc] >= 0;
          oc[ct][v] = ok ? crow[lr] + ccol[lc] : -1;
          res[ct][v] = p.alpha * result(rt, ct, v);
        }
      if (D) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int lc = wn * (TN / 2) + ct * 16 + li;
            const int lr = wm * (TM / 2) + rt * 16 + Mma<T>::crow(lg, v);
            const double dv =
                D[oc[ct][v] >= 0 ? drow[lr] + dcol[lc] : (int64_t)0];
            res[ct][v] += p.gamma * dv;
          }
      }
      if (p.beta != 0.0) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double cv = C[oc[ct][v] >= 0 ? oc[ct][v] : (int64_t)0];
            res[ct][v] += p.beta * cv;
          }
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (oc[ct][v] >= 0) C[oc[ct][v]] = res[ct][v];
    } else {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int lc = wn * (TN / 2) + ct * 16 + li;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int lr = wm * (TM / 2) + rt * 16 + Mma<T>::crow(lg, v);
          if (m0 + lr < p.M && n0 + lc < p.N)
            P[(int64_t)(m0 + lr) * p.N + n0 + lc] = result(rt, ct, v);
        }
      }
    }
  }
}

// The same product for K of one index and at most KP (16 to 64): the O(n^5)
// terms over one spin run of an orbital index, whose time is the passes over
// their outputs.  In the kernel above a workgroup takes its slabs and then
// its C one after another, each at the latency of memory: 20 us in all for
// the Z -= t1.u term at n = 66, of which 1.3 us is the matrix cores'.  Here
// everything a workgroup reads (both whole panels, C and the addend) is in
// flight together before the first use.  RT x CT MFMA blocks per wave, WM x
// WN waves: 16 RT rows where the rows are one orbital run (33 take 48, not
// 64), likewise for columns, 64x64 otherwise.  MFMA step s takes the k from
// 4s to 4s + 3, steps past K are left out; row stride KP + 2 doubles, so
// that the 32 lanes of a read (16 rows, two k) hit distinct banks.
template <int RT, int CT, int WM, int WN, int KP>
__global__ __launch_bounds__(NT, KP > 48 ? 2 : 3) void gemm_short_kernel(
    GemmGroup grp, int amf, int bnf) {
  constexpr int TM = 16 * RT * WM, TN = 16 * CT * WN, LDK = KP + 2;
  constexpr int EA = TM * KP / NT, EB = TN * KP / NT;
  static_assert(WM * WN == 4 && TM + TN <= NT / 2, "four waves, 128 offsets");
  extern __shared__ double sm[];   // A [TM][LDK], B [TN][LDK]
  double *As = sm, *Bs = sm + TM * LDK;
  __shared__ int64_t aoff[TM], boff[TN], crow[TM], ccol[TN], drow[TM],
      dcol[TN];
  const int64_t bid = xcd_block();
  int item = 0;
  for (int k = 1; k < grp.n; ++k)
    if (bid >= grp.tile0[k]) item = k;
  const GemmDev &p = grp.pr[item];
  const BlockPos q = decode(p, (int)(bid - grp.tile0[item]));
  const int t = threadIdx.x, m0 = q.tm * TM, n0 = q.tn * TN, K = p.K;
  // offsets: of A and B by the first half of the threads, of C and D (after
  // the scatter maps; -1: dropped or past the end) by the second
  if (t < NT / 2) {
    tile_offsets<TM, TN>(p, m0, n0, aoff, boff);
  } else {
    const int u = t - NT / 2;
    if (u < TM) {
      const int row = m0 + u;
      const int rr = row < p.M ? (p.rmap ? p.rmap[row] : row) : -1;
      const Lvl l =
          map_level(levels(rr < 0 ? 0 : rr, p.M1, p.M2), p.mmap, p.mlvl);
      crow[u] = rr < 0 ? -1 : at(l, p.sCm0, p.sCm1, p.sCm);
      drow[u] = rr < 0 ? -1 : at(l, p.sDm0, p.sDm1, p.sDm);
    } else if (u < TM + TN) {
      const int col = n0 + u - TM;
      const int cc = col < p.N ? (p.cmap ? p.cmap[col] : col) : -1;
      const Lvl l =
          map_level(levels(cc < 0 ? 0 : cc, p.N1, p.N2), p.nmap, p.nlvl);
      ccol[u - TM] = cc < 0 ? -1 : at(l, p.sCn0, p.sCn1, p.sCn);
      dcol[u - TM] = cc < 0 ? -1 : at(l, p.sDn0, p.sDn1, p.sDn);
    }
  }
  __syncthreads();
  // both panels: threads along the index that is contiguous in memory;
  // loads past an edge read element 0 and count as zero
  const double *A = p.A + q.b1 * p.sA1 + q.b2 * p.sA2;
  const double *B = p.B + q.b1 * p.sB1 + q.b2 * p.sB2;
  double ra[EA], rb[EB];
#pragma unroll
  for (int r = 0; r < EA; ++r) {
    const int e = t + NT * r;
    const int m = amf ? e % TM : e / KP, k = amf ? e / TM : e % KP;
    const int64_t off = aoff[m];
    const bool ok = off >= 0 && k < K;
    const double v = A[ok ? off + (int64_t)k * p.sAk : (int64_t)0];
    ra[r] = ok ? v : 0.0;
  }
#pragma unroll
  for (int r = 0; r < EB; ++r) {
    const int e = t + NT * r;
    const int n = bnf ? e % TN : e / KP, k = bnf ? e / TN : e % KP;
    const int64_t off = boff[n];
    const bool ok = off >= 0 && k < K;
    const double v = B[ok ? off + (int64_t)k * p.sBk : (int64_t)0];
    rb[r] = ok ? v : 0.0;
  }
  // the old C and the addend of this lane's elements
  const int lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 15, lg = lane >> 4;
  double *C = p.C + q.b1 * p.sC1 + q.b2 * p.sC2;
  const double *D = p.D ? p.D + q.b1 * p.sD1 + q.b2 * p.sD2 : nullptr;
  double cv[RT][CT][4];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v) cv[rt][ct][v] = 0.0;
  if (p.beta != 0.0) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t r = crow[(wm * RT + rt) * 16 + lg + 4 * v];
          const int64_t c = ccol[(wn * CT + ct) * 16 + li];
          cv[rt][ct][v] = p.beta * C[r >= 0 && c >= 0 ? r + c : (int64_t)0];
        }
  }
  if (D) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int x = (wm * RT + rt) * 16 + lg + 4 * v;
          const int z = (wn * CT + ct) * 16 + li;
          cv[rt][ct][v] +=
              p.gamma *
              D[crow[x] >= 0 && ccol[z] >= 0 ? drow[x] + dcol[z] : (int64_t)0];
        }
  }
#pragma unroll
  for (int r = 0; r < EA; ++r) {
    const int e = t + NT * r;
    As[(amf ? e % TM : e / KP) * LDK + (amf ? e / TM : e % KP)] = ra[r];
  }
#pragma unroll
  for (int r = 0; r < EB; ++r) {
    const int e = t + NT * r;
    Bs[(bnf ? e % TN : e / KP) * LDK + (bnf ? e / TN : e % KP)] = rb[r];
  }
  __syncthreads();
  d4_t acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = d4_t{0, 0, 0, 0};
#pragma unroll
  for (int st = 0; st < KP / 4; ++st) {
    if (4 * st >= K) break;
    double a[RT], b[CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      a[rt] = As[((wm * RT + rt) * 16 + li) * LDK + 4 * st + lg];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      b[ct] = Bs[((wn * CT + ct) * 16 + li) * LDK + 4 * st + lg];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        acc[rt][ct] = Mma<double>::op(a[rt], b[ct], acc[rt][ct]);
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t r = crow[(wm * RT + rt) * 16 + lg + 4 * v];
        const int64_t c = ccol[(wn * CT + ct) * 16 + li];
        if (r >= 0 && c >= 0)
          C[r + c] = p.alpha * acc[rt][ct][v] + cv[rt][ct][v];
      }
}

// Epilogue of one element of a split product: C[b][m,n] = alpha * s + gamma
// * D + beta * C through the scatter maps.
__device__ inline void put_sum(const GemmDev &p, int64_t cb, int64_t mn,
                               double s) {
  const int m0 = (int)(mn / p.N), n0 = (int)(mn % p.N);
  const int m = p.rmap ? p.rmap[m0] : m0, n = p.cmap ? p.cmap[n0] : n0;
  if (m < 0 || n < 0) return;
  const int64_t b1 = cb / p.nb2, b2 = cb % p.nb2;
  const Lvl lr = map_level(levels(m, p.M1, p.M2), p.mmap, p.mlvl),
            lc = map_level(levels(n, p.N1, p.N2), p.nmap, p.nlvl);
  double *c = p.C + b1 * p.sC1 + b2 * p.sC2 +
              at(lr, p.sCm0, p.sCm1, p.sCm) + at(lc, p.sCn0, p.sCn1, p.sCn);
  double y = p.alpha * s;
  if (p.D)
    y += p.gamma * p.D[b1 * p.sD1 + b2 * p.sD2 +
                       at(lr, p.sDm0, p.sDm1, p.sDm) +
                       at(lc, p.sDn0, p.sDn1, p.sDn)];
  if (p.beta != 0.0) y += p.beta * *c;
  *c = y;
}

// C[b][m,n] = alpha * sum_r partial[r][b][m][n] + beta*C  (fixed order), for
// the outputs of a group (tile0: the first workgroup of each).
// A block of RG x 64 threads takes 64 consecutive elements (coalesced rows
// of the partial buffer); its RG groups sum interleaved partials (several
// loads in flight per thread) and combine in LDS, so that even a small
// output (a few thousand elements) spreads its R-deep sums over the chip.
constexpr int RG = 16;
__global__ __launch_bounds__(64 * RG) void reduce_partial_kernel(
    GemmGroup grp) {
  __shared__ double part[RG][64];
  int item = 0;
  for (int k = 1; k < grp.n; ++k)
    if ((int)blockIdx.x >= grp.tile0[k]) item = k;
  const GemmDev &p = grp.pr[item];
  const int64_t MN = (int64_t)p.M * p.N;
  const int64_t total = MN * p.nb1 * p.nb2;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6, R = p.R;
  const int64_t idx =
      (int64_t)((int)blockIdx.x - grp.tile0[item]) * 64 + lane;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  if (idx < total) {
    const double *src = p.partial + idx;
    int r = g;
    for (; r + 3 * RG < R; r += 4 * RG) {
      s0 += src[(int64_t)r * total];
      s1 += src[(int64_t)(r + RG) * total];
      s2 += src[(int64_t)(r + 2 * RG) * total];
      s3 += src[(int64_t)(r + 3 * RG) * total];
    }
    for (; r < R; r += RG) s0 += src[(int64_t)r * total];
  }
  part[g][lane] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (g == 0 && idx < total) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < RG; ++q) s += part[q][lane];
    put_sum(p, idx / MN, idx % MN, s);
  }
}

// The same for few partials: one thread per element, which sums them in
// order with all its loads in flight (the form above leaves RG - R of its
// RG groups idle).
constexpr int FEW = 12;
__global__ __launch_bounds__(256) void reduce_few_kernel(GemmGroup grp) {
  int item = 0;
  for (int k = 1; k < grp.n; ++k)
    if ((int)blockIdx.x >= grp.tile0[k]) item = k;
  const GemmDev &p = grp.pr[item];
  const int64_t MN = (int64_t)p.M * p.N;
  const int64_t total = MN * p.nb1 * p.nb2;
  const int R = p.R;
  const int64_t idx =
      (int64_t)((int)blockIdx.x - grp.tile0[item]) * 256 + threadIdx.x;
  if (idx >= total) return;
  double v[FEW];
#pragma unroll
  for (int r = 0; r < FEW; ++r)
    v[r] = p.partial[(int64_t)(r < R ? r : 0) * total + idx];
  double s = v[0];
#pragma unroll
  for (int r = 1; r < FEW; ++r) s += r < R ? v[r] : 0.0;
  put_sum(p, idx / MN, idx % MN, s);
}

// Tile shape and K splits of a group: 64x64 tiles (policy 0), and the K per
// split with the least estimated time.  64x64 is the fastest tile of launches
// that do not fill the chip (TFLOP/s FP64, 64x64 | 128x64 | 128x128: 11 of
// 1458^3 51 | 48 | 42; 15 of 722^3 42 | 36 | 30) and of the short-K terms,
// whose groups it shortens by 4% of a step at n = 66; the wider ones are left
// to the autotuner, but for one product of K >= 1024 and at least 1024
// 128x128 tiles with at most 6% of padding, which takes those (FP64, 64x64 |
// 128x128: 3 of 3249^3 46 | 51, 4096^3 50 | 55, 4356^3 46 | 48, 6561^3 43 |
// 51, 8192^3 47 | 55; with 11% of padding, 8 of 1089x2178x2178, 46 | 42).
//   Per CU a workgroup's slab takes the time of its MFMAs, and a CU works
// through its workgroups of a launch at that rate or at that of the load
// latency of its resident ones, whichever is longer; partial sums (splits of
// K, and products of one output) add their write and read.  (Splitting every
// launch of fewer than 1024 workgroups, as this rule did before, spent half
// of an FP64 step at n = 54 in the sums of partials: 7.4 of 14.4 ms.)
//   FP32: the same; under policies 1 and 2 wide tiles (2: the narrower one by
// the aspect) only where one product has 1024 of them.  A wide tile has no
// registers for the FP64 sums of its accumulators, which at that many tiles
// run over all of K (TFLOP/s and error of the result, 128x128 | 64x64: 4096^3
// 82 1.1e-6 | 76 2.0e-7; 4356^3 78 1.2e-6 | 72 2.0e-7; four of 2178^3, 11% of
// padding, 64 8.3e-7 | 64 2.0e-7; the sums cost a 64x64 tile 2 to 4%).
struct Plan {
  Tile t;
  int kc;   // K of a split, whole slabs
};
int64_t tiles_of(const Gemm &g, Tile t) {
  return (int64_t)((g.M + t.m - 1) / t.m) * ((g.N + t.n - 1) / t.n) * g.nb1 *
         g.nb2;
}
int splits_of(const Gemm &g, int kc) {
  return g.K <= kc ? 1 : (g.K + kc - 1) / kc;
}
double estimate_us(const Gemm *g, const int *cblk, int n, Tile t, int kc) {
  const int occ = t.m * t.n >= 128 * 128 ? 2 : (t.m * t.n >= 8192 ? 3 : 4);
  // one slab of the tile on a CU's four matrix cores, us, and the time
  // from a slab's loads to its use
  const double ts = 1.9 * t.m * t.n / (128.0 * 128.0), lat = 1.2;
  double b = 0.0, sum = 0.0;
  for (int k = 0; k < n; ++k) {
    const int sp = splits_of(g[k], kc);
    // the last split of a product is shorter than the others
    b += tiles_of(g[k], t) * (double)std::min(kc, std::max(g[k].K, BK)) / kc *
         sp;
    bool shared = false;
    for (int q = 0; q < n; ++q) shared |= q != k && cblk[q] == cblk[k];
    if (sp > 1 || shared)
      sum += (double)g[k].M * g[k].N * g[k].nb1 * g[k].nb2 * 8e-6 *   // MB
             (sp * 2.0 + 1.0) / 3.0;
  }
  const double us =
      (kc / BK + 2.0) * std::max(std::ceil(b / 256.0) * ts,
                                 std::ceil(b / (256.0 * occ)) * lat);
  return us + (sum > 0.0 ? 4.0 + sum : 0.0);
}
Plan plan_of(const Gemm *g, const int *cblk, int n, bool f32) {
  const int pol = g[0].tile_policy;
  const Tile cand[4] = {{128, 128}, {128, 64}, {64, 128}, {64, 64}};
  int M = 0, N = 0, K = 0;
  for (int k = 0; k < n; ++k) {
    M = std::max(M, g[k].M);
    N = std::max(N, g[k].N);
    K = std::max(K, g[k].K);
  }
  const int whole = std::max(1, (K + BK - 1) / BK) * BK;
  Plan best{{64, 64}, whole};
  if (n == 1 && M > 64 && N > 64 && (pol == 0 ? K >= 1024 : f32)) {
    const Tile t = pol != 2 ? cand[0] : M >= N ? cand[1] : cand[2];
    const int64_t tiles = tiles_of(g[0], t);
    const bool tight = (double)M * N * g[0].nb1 * g[0].nb2 >=
                       0.94 * (double)tiles * t.m * t.n;
    // (a larger split_target asks FP32 for more partial sums)
    const int fill = f32 ? std::max(1024, g[0].split_target) : 1024;
    if (tiles >= fill && (pol != 0 || tight)) return Plan{t, whole};
  }
  double us = 1e300;
  for (const Tile &t : cand) {
    if (f32 && t.m * t.n > 64 * 64) continue;
    // the wide policies take no 128-wide tile for a side of at most 64
    if ((M <= 64 && t.m > 64) || (N <= 64 && t.n > 64)) continue;
    const bool full = t.m >= std::min(128, (M + 63) / 64 * 64) &&
                      t.n >= std::min(128, (N + 63) / 64 * 64);
    if (pol == 0 && t.m * t.n > 64 * 64) continue;
    if (pol == 1 && !f32 && !full) continue;
    if (pol == 2 && t.m * t.n == 128 * 128) continue;
    int64_t blocks = 0;
    for (int k = 0; k < n; ++k) blocks += tiles_of(g[k], t);
    const int64_t want =
        (std::max(1, g[0].split_target) + blocks - 1) / blocks;
    const int maxs = (int)std::max<int64_t>(
        1, std::min<int64_t>(std::min<int64_t>(want, 2048), K / (4 * BK)));
    for (int sp = 1; sp <= maxs; sp += 1 + sp / 8) {
      const int kc = ((K + sp - 1) / sp + BK - 1) / BK * BK;
      const double e =
          estimate_us(g, cblk, n, t, std::max(BK, std::min(kc, whole)));
      if (e < us * 0.98) {
        us = e;
        best = Plan{t, std::max(BK, std::min(kc, whole))};
      }
    }
  }
  return best;
}

template <typename K3>
void launch(K3 kernel, const GemmGroup &d, int64_t blocks, hipStream_t s) {
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(NT), 0, s, d);
  FTCC_CHECK_HIP(hipGetLastError());
}

template <typename T, int TM, int TN>
void launch_tile(bool amf, bool bnf, bool kl, const GemmGroup &d, int64_t nb,
                 hipStream_t s) {
  if (kl) launch(gemm_mfma_kernel<T, false, false, TM, TN, true>, d, nb, s);
  else if (amf && bnf)
    launch(gemm_mfma_kernel<T, true, true, TM, TN, false>, d, nb, s);
  else if (amf)
    launch(gemm_mfma_kernel<T, true, false, TM, TN, false>, d, nb, s);
  else if (bnf)
    launch(gemm_mfma_kernel<T, false, true, TM, TN, false>, d, nb, s);
  else launch(gemm_mfma_kernel<T, false, false, TM, TN, false>, d, nb, s);
}

template <typename T>
void launch_layout(Tile tl, bool amf, bool bnf, bool kl, const GemmGroup &d,
                   int64_t nb, hipStream_t s) {
  if (tl.m == 64 && tl.n == 64)
    launch_tile<T, 64, 64>(amf, bnf, kl, d, nb, s);
  else if (tl.m == 64) launch_tile<T, 64, 128>(amf, bnf, kl, d, nb, s);
  else if (tl.n == 64) launch_tile<T, 128, 64>(amf, bnf, kl, d, nb, s);
  else launch_tile<T, 128, 128>(amf, bnf, kl, d, nb, s);
}

template <int RT, int CT, int WM, int WN, int KP>
void launch_short(const GemmGroup &d, int64_t nb, bool amf, bool bnf,
                  hipStream_t s) {
  constexpr int LDS =
      (16 * RT * WM + 16 * CT * WN) * (KP + 2) * (int)sizeof(double);
  static std::once_flag attr;
  set_max_lds_once(attr, (const void *)gemm_short_kernel<RT, CT, WM, WN, KP>,
                   LDS);
  hipLaunchKernelGGL((gemm_short_kernel<RT, CT, WM, WN, KP>),
                     dim3((unsigned)nb), dim3(NT), LDS, s, d, amf ? 1 : 0,
                     bnf ? 1 : 0);
  FTCC_CHECK_HIP(hipGetLastError());
}
template <int RT, int CT, int WM, int WN>
void launch_short_k(int K, const GemmGroup &d, int64_t nb, bool amf, bool bnf,
                    hipStream_t s) {
  if (K <= 32) launch_short<RT, CT, WM, WN, 32>(d, nb, amf, bnf, s);
  else if (K <= 48) launch_short<RT, CT, WM, WN, 48>(d, nb, amf, bnf, s);
  else launch_short<RT, CT, WM, WN, 64>(d, nb, amf, bnf, s);
}
// Most 64x64 tiles of a launch of the short-K kernel, some five for each of
// its places on the chip.  Below it the latencies count, above it the passes
// over memory, which its three workgroups a CU hide less well than the four
// of the kernel above (n = 66: 162 -> 185 us at 28 000 tiles; the narrow
// forms are faster at any count, their tiles hold no empty rows: 492 -> 468
// us for the Z -= t1.u term).  n = 38, bf16x3 step: 1572 -> 1505 us.
constexpr int64_t SHORT_TILES = 4096;
// tile of the short-K kernel: as few 16-wide blocks as hold a side of at
// most 64 (the other side 64), else 64x64
Tile short_tile(int M, int N) {
  if (M <= 64) return Tile{std::max(2, (M + 15) / 16) * 16, 64};
  if (N <= 64) return Tile{64, std::max(2, (N + 15) / 16) * 16};
  return Tile{64, 64};
}
void launch_short_tile(Tile t, bool rows, int K, const GemmGroup &d,
                       int64_t nb, bool amf, bool bnf, hipStream_t s) {
  if (rows && t.m == 32) launch_short_k<2, 1, 1, 4>(K, d, nb, amf, bnf, s);
  else if (rows && t.m == 48)
    launch_short_k<3, 1, 1, 4>(K, d, nb, amf, bnf, s);
  else if (t.n == 32) launch_short_k<1, 2, 4, 1>(K, d, nb, amf, bnf, s);
  else if (t.n == 48) launch_short_k<1, 3, 4, 1>(K, d, nb, amf, bnf, s);
  else launch_short_k<2, 2, 2, 2>(K, d, nb, amf, bnf, s);
}

// operand layouts of the kernel instantiations
bool a_mfast(const Gemm &g) { return g.sAm == 1 && g.sAk != 1; }
bool b_nfast(const Gemm &g) { return g.sBn == 1 && g.sBk != 1; }

GemmDev device_form(const Gemm &g) {
  GemmDev d;
  d.M = g.M;
  d.N = g.N;
  d.K = g.K;
  d.nb1 = g.nb1;
  d.nb2 = g.nb2;
  d.alpha = g.alpha;
  d.beta = g.beta;
  d.A = g.A;
  d.sAm = g.sAm;
  d.sAk = g.sAk;
  d.sA1 = g.sA1;
  d.sA2 = g.sA2;
  d.B = g.B;
  d.sBk = g.sBk;
  d.sBn = g.sBn;
  d.sB1 = g.sB1;
  d.sB2 = g.sB2;
  d.C = g.C;
  d.sCm = g.sCm;
  d.sCn = g.sCn;
  d.sC1 = g.sC1;
  d.sC2 = g.sC2;
  d.rmap = g.rmap;
  d.cmap = g.cmap;
  d.D = g.D;
  d.gamma = g.gamma;
  d.sDm = g.sDm;
  d.sDn = g.sDn;
  d.sD1 = g.sD1;
  d.sD2 = g.sD2;
  // index levels of rows and columns (one index: everything in the last)
  require(g.M2 >= 0 && g.N2 >= 0 && g.M1 >= 1 && g.N1 >= 1,
          "GEMM index levels must be positive");
  if (g.M2 > 0)
    require(g.M % ((int64_t)g.M1 * g.M2) == 0,
            "GEMM rows are not a product of their index levels");
  if (g.N2 > 0)
    require(g.N % ((int64_t)g.N1 * g.N2) == 0,
            "GEMM columns are not a product of their index levels");
  d.M1 = g.M2 > 0 ? g.M1 : 1;
  d.M2 = g.M2 > 0 ? g.M2 : (1 << 30);
  d.N1 = g.N2 > 0 ? g.N1 : 1;
  d.N2 = g.N2 > 0 ? g.N2 : (1 << 30);
  d.sAm0 = g.sAm0;
  d.sAm1 = g.sAm1;
  d.sCm0 = g.sCm0;
  d.sCm1 = g.sCm1;
  d.sDm0 = g.sDm0;
  d.sDm1 = g.sDm1;
  d.sBn0 = g.sBn0;
  d.sBn1 = g.sBn1;
  d.sCn0 = g.sCn0;
  d.sCn1 = g.sCn1;
  d.sDn0 = g.sDn0;
  d.sDn1 = g.sDn1;
  require(g.K2 >= 0 && g.K1 >= 1, "GEMM K levels must be positive");
  if (g.K2 > 0)
    require(g.K % ((int64_t)g.K1 * g.K2) == 0,
            "GEMM K is not a product of its index levels");
  d.K1 = g.K2 > 0 ? g.K1 : 1;
  d.K2 = g.K2 > 0 ? g.K2 : (1 << 30);
  d.sAk0 = g.sAk0;
  d.sAk1 = g.sAk1;
  d.sBk0 = g.sBk0;
  d.sBk1 = g.sBk1;
  require((g.mlvl < 0 || (g.mmap && g.mlvl <= 2)) &&
              (g.nlvl < 0 || (g.nmap && g.nlvl <= 2)),
          "GEMM level map without a map or level");
  d.mmap = g.mmap;
  d.nmap = g.nmap;
  d.mlvl = g.mmap ? g.mlvl : -1;
  d.nlvl = g.nmap ? g.nlvl : -1;
  require(g.K2 == 0 || (!a_mfast(g) && !b_nfast(g)),
          "K over several indices needs both operands K-fastest");
  d.partial = nullptr;
  d.rbase = 0;
  d.R = 1;
  return d;
}

}  // namespace

bool gemm_groupable(const Gemm &x, const Gemm &y) {
  return a_mfast(x) == a_mfast(y) && b_nfast(x) == b_nfast(y) &&
         (x.K2 > 0) == (y.K2 > 0) && x.nb1 == y.nb1 && x.nb2 == y.nb2;
}

size_t gemm_group_scratch(const Gemm *g, const int *cblk, int n,
                          int precision) {
  const Plan pl = plan_of(g, cblk, n, precision == FTCC_PREC_FP32);
  size_t need = 0;
  for (int k = 0; k < n; ++k) {
    const int sp = splits_of(g[k], pl.kc);
    bool shared = false;
    for (int q = 0; q < n; ++q) shared |= q != k && cblk[q] == cblk[k];
    if (sp > 1 || shared)
      need += (size_t)sp * g[k].M * g[k].N * g[k].nb1 * g[k].nb2;
  }
  return need;
}

void gemm_run_group(const Gemm *g, const int *cblk, int n, int precision,
                    Scratch &scr, hipStream_t s) {
  require(precision == FTCC_PREC_FP64 || precision == FTCC_PREC_FP32,
          "the generic GEMM runs FP64 or FP32 (bf16x3 uses sbgemm)");
  require(n >= 1 && n <= GEMM_GROUP, "GEMM group size");
  const Plan pl = plan_of(g, cblk, n, precision == FTCC_PREC_FP32);
  // K of one index and at most 64, each output of one product: the short-K
  // kernel (in FP64, the precision of those terms, and under the default
  // launch plan)
  int Mx = 0, Nx = 0, Kx = 0;
  bool brief = precision == FTCC_PREC_FP64 && g[0].tile_policy == 0;
  for (int k = 0; k < n; ++k) {
    Mx = std::max(Mx, g[k].M);
    Nx = std::max(Nx, g[k].N);
    Kx = std::max(Kx, g[k].K);
    brief = brief && g[k].K >= 1 && g[k].K <= 64 && g[k].K2 == 0;
    for (int q = 0; q < k; ++q) brief = brief && cblk[q] != cblk[k];
  }
  const Tile st = short_tile(Mx, Nx);
  if (brief && st.m * st.n == 64 * 64) {
    int64_t tiles = 0;
    for (int k = 0; k < n; ++k) tiles += tiles_of(g[k], st);
    brief = tiles <= SHORT_TILES;
  }
  const Tile tl = brief ? st : pl.t;
  GemmGroup grp, red;
  grp.n = red.n = 0;
  int64_t blocks = 0, rblocks = 0, elems = 0;
  size_t used = 0;
  int maxR = 1;
  for (int k = 0; k < n; ++k) {
    if (g[k].M <= 0 || g[k].N <= 0 || g[k].nb1 <= 0 || g[k].nb2 <= 0) continue;
    require(gemm_groupable(g[0], g[k]), "GEMM group of different layouts");
    GemmDev &d = grp.pr[grp.n];
    d = device_form(g[k]);
    d.tilesM = (g[k].M + tl.m - 1) / tl.m;
    d.tilesN = (g[k].N + tl.n - 1) / tl.n;
    d.m_inner = d.tilesM < d.tilesN ? 1 : 0;
    d.splits = splits_of(g[k], pl.kc);
    d.kchunk = pl.kc;
    grp.tile0[grp.n++] = (int)blocks;
    blocks += (int64_t)d.tilesM * d.tilesN * d.splits * d.nb1 * d.nb2;
  }
  if (grp.n == 0) return;
  require(blocks < (1LL << 31), "GEMM grid too large");
  // partial sums: each output of several products, or of a split K, in the
  // order the products are given
  int q = 0;
  std::vector<int> blk(grp.n);
  for (int k = 0; k < n; ++k)
    if (!(g[k].M <= 0 || g[k].N <= 0 || g[k].nb1 <= 0 || g[k].nb2 <= 0))
      blk[q++] = cblk[k];
  for (int k = 0; k < grp.n; ++k) {
    int R = 0;
    bool first = true;
    for (int j = 0; j < grp.n; ++j)
      if (blk[j] == blk[k]) {
        if (j < k) first = false;
        R += grp.pr[j].splits;
      }
    if (R == 1 || !first) continue;
    GemmDev &d = grp.pr[k];
    const int64_t per = (int64_t)d.M * d.N * d.nb1 * d.nb2;
    double *part = scr.partial + used;
    used += (size_t)R * per;
    require(used <= scr.partial_elems, "GEMM split-K scratch too small",
            FTCC_ENOMEM);
    int rb = 0;
    for (int j = k; j < grp.n; ++j)
      if (blk[j] == blk[k]) {
        GemmDev &e = grp.pr[j];
        require(e.M == d.M && e.N == d.N, "GEMM group: outputs differ");
        e.partial = part;
        e.rbase = rb;
        rb += e.splits;
      }
    d.R = R;
    red.pr[red.n++] = d;
    maxR = std::max(maxR, R);
    elems += per;
  }
  const bool amf = a_mfast(g[0]), bnf = b_nfast(g[0]), kl = g[0].K2 > 0;
  if (brief) {
    launch_short_tile(tl, Mx <= 64, Kx, grp, blocks, amf, bnf, s);
    return;
  }
  if (precision == FTCC_PREC_FP64)
    launch_layout<double>(tl, amf, bnf, kl, grp, blocks, s);
  else
    launch_layout<float>(tl, amf, bnf, kl, grp, blocks, s);
  if (red.n == 0) return;
  // few partials of a large output: a thread for each element
  const bool few = maxR <= FEW && elems >= 32 * 1024;
  const int unit = few ? 256 : 64;
  for (int k = 0; k < red.n; ++k) {
    const GemmDev &d = red.pr[k];
    red.tile0[k] = (int)rblocks;
    rblocks += ((int64_t)d.M * d.N * d.nb1 * d.nb2 + unit - 1) / unit;
  }
  require(rblocks < (1LL << 31), "GEMM grid too large");
  if (few)
    hipLaunchKernelGGL(reduce_few_kernel, dim3((unsigned)rblocks), dim3(256),
                       0, s, red);
  else
    hipLaunchKernelGGL(reduce_partial_kernel, dim3((unsigned)rblocks),
                       dim3(64 * RG), 0, s, red);
  FTCC_CHECK_HIP(hipGetLastError());
}

}  // namespace ftcc
