// FP64 and FP32 GEMM for the O(n^6) products: operands already gathered into
// contiguous K-fast copies (A as [M][ld], B transposed as [N][ld], K padded
// with zeros to a multiple of 32), FP64 output through scatter maps.
//
// Bound: the matrix cores (v_mfma_f64_16x16x4_f64, v_mfma_f32_16x16x4_f32).
// A workgroup of 4 wave64s owns a TM x TM tile of C, each wave a quadrant of
// 16x16 blocks.  K advances in slabs of 128 bytes a row (16 doubles, 32
// floats).  Slabs go from memory straight into LDS
// (global_load_lds_dwordx4), NST - 1 slabs ahead, through a ring of NST
// stages with one barrier per slab; a row's eight 16-byte chunks are stored
// at slot c ^ (row & 7), so that the eight lanes that read one chunk of
// eight rows hit distinct banks.  In a slab, lane group g (= lane / 16)
// holds the k of chunks 2g and 2g + 1 of its row and MFMA step s takes its
// element s; A and B use the same map, so the contraction is unchanged.
//
// Against the general engine of gemm.hip (strided loads through registers,
// an offset lookup and a bounds test for each element): 15 of 1089x2178x2178
// FP64 49 TFLOP/s there, 64 here, FP32 66 and 115.
#include "ftcc_internal.h"

#include <algorithm>

namespace ftcc {
namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

template <typename T> struct Mma;
template <> struct Mma<double> {
  using acc_t = d4_t;
  static constexpr int STEPS = 4;   // MFMA steps (of 4 k each) per slab
  // output element v of lane group lg sits in row lg + 4v of the block
  __device__ static int crow(int lg, int v) { return lg + 4 * v; }
  __device__ static acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<float> {
  using acc_t = f4_t;
  static constexpr int STEPS = 8;
  // output element v of lane group lg sits in row 4*lg + v of the block
  __device__ static int crow(int lg, int v) { return 4 * lg + v; }
  __device__ static acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

constexpr int MAXP = 3;
constexpr int ROWB = 128;      // bytes of a row in a slab
template <typename T> struct Prob {
  int M, N, nslab, tilesM, tilesN;
  int tile0;                   // first linear tile of this problem
  const T *A, *B;
  int64_t lda, sAb, ldb, sBb;
  const int *rmap, *cmap;      // output scatter (nullptr: identity)
};
template <typename T> struct Dev {
  int nprob;
  Prob<T> pr[MAXP];
  double *C;
  int64_t sCm, sCn, sCb;
  double alpha, beta;
};

// Workgroup -> (problem, batch, tile m, tile n): ids regrouped per XCD
// (consecutive ones go to different XCDs), tiles in bands of GROUP_M rows so
// that an XCD's concurrent tiles share operand panels in its L2.
constexpr int GROUP_M = 8;
template <typename T>
__device__ inline Prob<T> tile_of(const Dev<T> &p, int &bt, int &tm, int &tn) {
  const int nblk = gridDim.x, b = blockIdx.x;
  const int q = nblk / 8, r = nblk % 8, x = b % 8, j = b / 8;
  const int lid = (x < r) ? x * (q + 1) + j : r * (q + 1) + (x - r) * q + j;
  Prob<T> pr = p.pr[0];
  if (p.nprob > 1 && lid >= p.pr[1].tile0) pr = p.pr[1];
  if (p.nprob > 2 && lid >= p.pr[2].tile0) pr = p.pr[2];
  const int local = lid - pr.tile0;
  const int per = pr.tilesM * pr.tilesN;
  bt = local / per;
  const int t = local % per;
  const int span = GROUP_M * pr.tilesN;
  const int first_m = (t / span) * GROUP_M;
  const int gsz = min(pr.tilesM - first_m, GROUP_M);
  tm = first_m + (t % span) % gsz;
  tn = (t % span) / gsz;
  return pr;
}

// One wave's share of a slab of one operand: its quarter of the TM rows,
// eight rows x eight chunks a load.  Rows past the end read the last one
// (their products are never stored).
template <typename T, int TM>
__device__ inline void load_slab(const T *src, int64_t ld, int row0, int rows,
                                 int slab, char *op, int wave, int lane) {
  const int r8 = lane >> 3, slot = lane & 7;
#pragma unroll
  for (int j = 0; j < TM / 32; ++j) {
    const int rl0 = (wave * (TM / 32) + j) * 8;
    const int g = min(row0 + rl0 + r8, rows - 1);
    const char *a = (const char *)(src + (int64_t)g * ld) +
                    (int64_t)slab * ROWB + 16 * (slot ^ r8);
    __builtin_amdgcn_global_load_lds((const void *)a,
                                     (lds_void *)(op + rl0 * ROWB), 16, 0, 0);
  }
}

// the 32 bytes (chunks 2 lg, 2 lg + 1) of one row
template <typename T>
__device__ inline void frag(const char *op, int row, int lg, T *out) {
  typedef T v_t __attribute__((ext_vector_type(16 / sizeof(T))));
  constexpr int E = 16 / sizeof(T);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const v_t v =
        *(const v_t *)(op + row * ROWB + (((2 * lg + h) ^ (row & 7)) << 4));
#pragma unroll
    for (int e = 0; e < E; ++e) out[h * E + e] = v[e];
  }
}

template <typename T, int TM, int NST>
__global__ __launch_bounds__(256, 2) void pgemm_kernel(Dev<T> p) {
  using acc_t = typename Mma<T>::acc_t;
  constexpr int RT = TM / 32;            // 16x16 blocks of a wave per side
  constexpr int STEPS = Mma<T>::STEPS;
  constexpr int OPB = TM * ROWB, STAGEB = 2 * OPB;
  constexpr int LOADS = 2 * (TM / 32);   // loads of a wave per slab
  extern __shared__ char lds[];          // [NST][A | B][TM rows][128 B]
  __shared__ int emap[2 * TM];
  int bt, tm, tn;
  const Prob<T> pr = tile_of(p, bt, tm, tn);
  const int m0 = tm * TM, n0 = tn * TM;
  for (int t = threadIdx.x; t < 2 * TM; t += 256) {
    const bool row = t < TM;
    const int x = row ? m0 + t : n0 + t - TM;
    const int *map = row ? pr.rmap : pr.cmap;
    emap[t] = x < (row ? pr.M : pr.N) ? (map ? map[x] : x) : -1;
  }
  const T *A = pr.A + bt * pr.sAb, *B = pr.B + bt * pr.sBb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lg = lane >> 4;

  acc_t acc[RT][RT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < RT; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  // FP32: the sums folded so far
  constexpr bool FOLD = sizeof(T) == 4;
  d4_t sum[FOLD ? RT : 1][FOLD ? RT : 1];
  if (FOLD) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < RT; ++j) sum[i][j] = d4_t{0, 0, 0, 0};
  }
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < RT; ++j) {
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[i][j][v] += (double)acc[i][j][v];
        acc[i][j] = acc_t{0, 0, 0, 0};
      }
  };

  // the maps above are read after a barrier even when K is empty, and their
  // loads are not counted by the waits below
  __syncthreads();
  const int nslab = pr.nslab;
  if (nslab > 0) {
#pragma unroll
    for (int q = 0; q < NST - 1; ++q) {
      char *st = lds + q * STAGEB;
      load_slab<T, TM>(A, pr.lda, m0, pr.M, min(q, nslab - 1), st, wave, lane);
      load_slab<T, TM>(B, pr.ldb, n0, pr.N, min(q, nslab - 1), st + OPB, wave,
                       lane);
    }
  }
  int cur = 0, nxt = NST - 1;   // stages of slab s and of slab s + NST - 1
  for (int s = 0; s < nslab; ++s) {
    // slab s has landed (this wave's loads, then every wave's), and every
    // wave has its fragments of slab s - 1, whose stage is loaded next.
    // Past the last slab the last one is loaded again into a stage that is
    // not read any more, which keeps the count of loads in flight constant.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NST - 2) * LOADS)
                 : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    {
      const int sl = min(s + NST - 1, nslab - 1);
      char *st = lds + nxt * STAGEB;
      load_slab<T, TM>(A, pr.lda, m0, pr.M, sl, st, wave, lane);
      load_slab<T, TM>(B, pr.ldb, n0, pr.N, sl, st + OPB, wave, lane);
    }
    const char *As = lds + cur * STAGEB, *Bs = As + OPB;
    T a[RT][STEPS], b[RT][STEPS];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      frag<T>(As, wm * (TM / 2) + rt * 16 + li, lg, a[rt]);
#pragma unroll
    for (int ct = 0; ct < RT; ++ct)
      frag<T>(Bs, wn * (TM / 2) + ct * 16 + li, lg, b[ct]);
#pragma unroll
    for (int k = 0; k < STEPS; ++k)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < RT; ++ct)
          acc[rt][ct] = Mma<T>::op(a[rt][k], b[ct][k], acc[rt][ct]);
    if (FOLD && (s + 1) % (FOLD_K / (ROWB / (int)sizeof(T))) == 0) fold();
    cur = cur + 1 == NST ? 0 : cur + 1;
    nxt = nxt + 1 == NST ? 0 : nxt + 1;
  }
  // no load may still be writing LDS when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (FOLD) fold();

  // lane holds column li of each block.  Reads of C (beta != 0) are
  // unconditional (a dropped element reads element 0) and every value is
  // formed before the first store, so that no store waits for a read.
  double *C = p.C + bt * p.sCb;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int64_t off[RT][4];
    double res[RT][4];
#pragma unroll
    for (int ct = 0; ct < RT; ++ct) {
      const int cc = emap[TM + wn * (TM / 2) + ct * 16 + li];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int rr = emap[wm * (TM / 2) + rt * 16 + Mma<T>::crow(lg, v)];
        off[ct][v] = (rr >= 0 && cc >= 0)
                         ? (int64_t)rr * p.sCm + (int64_t)cc * p.sCn
                         : (int64_t)-1;
        res[ct][v] = p.alpha * (FOLD ? sum[rt][ct][v] : (double)acc[rt][ct][v]);
      }
    }
    if (p.beta != 0.0) {
#pragma unroll
      for (int ct = 0; ct < RT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          res[ct][v] += p.beta * C[off[ct][v] >= 0 ? off[ct][v] : (int64_t)0];
    }
#pragma unroll
    for (int ct = 0; ct < RT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (off[ct][v] >= 0) C[off[ct][v]] = res[ct][v];
  }
}

// 64x64 tiles, 32x32 where those would be fewer than two per CU.  Measured
// (TFLOP/s, FP64 | FP32, 64x64 against 32x32): 15 of 1120x2240x2240 64 to 50
// | 115 to 102; 11 of 736^3 46 to 42 | 81 to 81; 11 of 352^3 31 to 32 | 50
// to 52; one 384x768x768 14 to 20 | 23 to 36; 9 of 64x128x128 2.2 to 3.5 |
// 2.8 to 4.2.  128x128 tiles reach 69 | 119 at 4096^3 against 67 | 118, but
// leave more of the chip idle at every size above (11 of 736x1472x1472: 46
// against 57).
bool small_tiles(const PgProblem *prob, int nprob, int nb) {
  int64_t tiles = 0;
  for (int k = 0; k < nprob; ++k)
    tiles += (int64_t)((prob[k].M + 63) / 64) * ((prob[k].N + 63) / 64) * nb;
  return tiles < 512;
}

template <typename T, int TM, int NST>
void launch(Dev<T> &p, const PgProblem *prob, int nprob, int nb,
            hipStream_t s) {
  constexpr size_t LDS = (size_t)NST * 2 * TM * ROWB;
  static std::once_flag attr;
  set_max_lds_once(attr, (const void *)pgemm_kernel<T, TM, NST>, (int)LDS);
  int64_t tiles = 0;
  p.nprob = 0;
  for (int k = 0; k < nprob; ++k) {
    const PgProblem &q = prob[k];
    if (q.M <= 0 || q.N <= 0) continue;
    Prob<T> &d = p.pr[p.nprob++];
    d.M = q.M;
    d.N = q.N;
    d.nslab = (int)((q.K * sizeof(T) + ROWB - 1) / ROWB);
    d.tilesM = (q.M + TM - 1) / TM;
    d.tilesN = (q.N + TM - 1) / TM;
    d.tile0 = (int)tiles;
    d.A = (const T *)q.A;
    d.B = (const T *)q.B;
    d.lda = q.lda;
    d.ldb = q.ldb;
    d.sAb = q.sAb;
    d.sBb = q.sBb;
    d.rmap = q.rmap;
    d.cmap = q.cmap;
    tiles += (int64_t)d.tilesM * d.tilesN * nb;
  }
  if (p.nprob == 0 || nb <= 0) return;
  require(tiles < (1LL << 31), "too many GEMM tiles");
  hipLaunchKernelGGL((pgemm_kernel<T, TM, NST>), dim3((unsigned)tiles),
                     dim3(256), LDS, s, p);
  FTCC_CHECK_HIP(hipGetLastError());
}

template <typename T>
void grouped(const PgProblem *prob, int nprob, int nb, double alpha,
             double beta, double *C, int64_t sCm, int64_t sCn, int64_t sCb,
             hipStream_t s) {
  constexpr int KSTEP = ROWB / sizeof(T);
  for (int k = 0; k < nprob; ++k) {
    const PgProblem &q = prob[k];
    if (q.M <= 0 || q.N <= 0) continue;
    // whole slabs are read: K padded to a slab inside the rows, and every
    // row aligned for the 16-byte loads
    const int64_t kp = (q.K + KSTEP - 1) / KSTEP * KSTEP;
    const int64_t el = 16 / sizeof(T);
    require(q.lda >= kp && q.ldb >= kp && q.lda % el == 0 &&
                q.ldb % el == 0 && q.sAb % el == 0 && q.sBb % el == 0 &&
                ((uintptr_t)q.A & 15) == 0 && ((uintptr_t)q.B & 15) == 0,
            "product operands need K padded to a slab and aligned rows");
  }
  Dev<T> p;
  p.C = C;
  p.sCm = sCm;
  p.sCn = sCn;
  p.sCb = sCb;
  p.alpha = alpha;
  p.beta = beta;
  if (small_tiles(prob, nprob, nb)) launch<T, 32, 6>(p, prob, nprob, nb, s);
  else launch<T, 64, 3>(p, prob, nprob, nb, s);
}

}  // namespace

void pgemm_grouped(int nprob, const PgProblem *prob, int nb, bool f32,
                   double alpha, double beta, double *C, int64_t sCm,
                   int64_t sCn, int64_t sCb, hipStream_t s) {
  require(nprob >= 1 && nprob <= MAXP, "1 to 3 problems per grouped launch");
  if (f32) grouped<float>(prob, nprob, nb, alpha, beta, C, sCm, sCn, sCb, s);
  else grouped<double>(prob, nprob, nb, alpha, beta, C, sCm, sCn, sCb, s);
}

}  // namespace ftcc
