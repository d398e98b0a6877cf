// df.hip -- density-fitted J/K on the device.
//
// Set-up (lai_dev_df_create): the auxiliary metric through the raw ERI
// kernels ((P u|Q u) with the unit function u) or the overlap kernel, its
// Cholesky factor and triangular inverse on the host (n_aux^3 / 3 flops each,
// once), the three-centre integrals (ab|P u) of every orbital shell pair in
// bounded batches through the raw ERI kernels, scattered into
// T[a][P][b], and B[a] = L^-1 T[a] for every orbital function a (one batched
// FP64 MFMA GEMM).  B stays in HBM in the layout [a][P][b]: row a of B is a
// contiguous n_aux x n matrix, so both exchange products are single GEMMs.
//
// Per build (lai_dev_df_jk): J in two HBM-bound passes over B (gamma_P, then
// J_ab = sum_P B[a][P][b] gamma_P); K = sum_P B_P D B_P^T as
// X[a][P][:] = B[a][P][:] D (one GEMM, rows (a, P)) and
// K[a][c] = sum_(P,b) X[a][P][b] B[c][P][b] (one GEMM over the summation
// index n_aux n, split into slices that are summed by a last kernel).
// A symmetric D that is positive semidefinite of low rank, as the density of
// occupied orbitals is, is factored first (df_factor, D = L L^T with r
// columns, corrected and checked against D): then X = B L has r columns instead
// of n and K[a][c] = sum_(P,i) X[a][P][i] X[c][P][i], r/n of the work (16 waters
// / cc-pVDZ, n 400, r 80: 7.6 -> 2.24 ms; X = B L 0.84, K beside the Coulomb
// passes 0.75, df_factor 0.34 and its correction 0.2 ms are what is left).
// Relative error of K (40 rows against long double, B as it is) by the general
// products and factored, 225 / 300 / 400 functions, in 1e-16: localised orbitals
// 6.1 8.0 11.0 and 5.6 7.5 9.0, delocalised 6.2 7.6 11.7 and 5.8 7.3 8.0, graded
// 7.5 8.0 14.6 and 6.2 6.1 10.5; without the correction (6 rows) 5.8 4.8 10.0,
// 9.2 11.0 12.3 and 18.7 29.8 33.6.
// The device decides (Factor::ok); the launches of the other form return at
// once.
#include "lai_device.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "api_internal.hpp"

namespace {

using lai::set_error;

#define DF_HIP(call)                                                                             \
  do {                                                                                           \
    hipError_t e_ = (call);                                                                      \
    if (e_ != hipSuccess)                                                                        \
      return set_error(LAI_ERR_BACKEND, std::string(#call) + ": " + hipGetErrorString(e_));     \
  } while (0)

constexpr int ncart_of(int L) { return (L + 1) * (L + 2) / 2; }

// ---------------------------------------------------------------------------
// FP64 GEMM on the matrix cores: C = A B with A row-major M x K and B either
// row-major K x N (bt = 0) or given as its transpose, row-major N x K
// (bt = 1).  A workgroup of four wavefronts computes a (64 BM) x (16 BN) tile
// of C, the wavefronts stacked along M, each a (16 BM) x (16 BN) strip as
// BM x BN blocks of v_mfma_f64_16x16x4f64.  The summation runs in steps of
// 16 through two LDS buffers: the next step's global loads are in flight
// (in registers) while the current step multiplies, then land in the other
// buffer; one workgroup barrier per step.  BN = 5 makes the 80-column tiles
// that divide the 400-function orbital dimension of the exchange products.
// blockIdx.z is a batch index (split = 0: A, B, C offset by sA, sB, sC) or a
// slice of the summation index (split = 1: columns [z kchunk, (z+1) kchunk)
// of A and rows of B, written to C + z sC).
// Lane layout of v_mfma_f64_16x16x4f64 on gfx950 (measured with one
// wavefront of marked inputs): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[l / 16 + 4 r][l % 16] in accumulator element r.
// ---------------------------------------------------------------------------
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int KT = 16;  // summation step

// What the factorisation of a density found out (factor_density).
struct Factor {
  int ok;    // 1: D = L L^T to rounding, rank columns
  int rank;
  double dmax;  // largest diagonal element of D
  double e2, d2;  // ||D - L L^T||^2 and ||D||^2 (Frobenius) over dmax^2
  int low;      // 0 until pivoting has ended, then 1 (the general product under way
                // may end) or -1 (D has no factor of at most n/2 columns)
};
constexpr double kEps = 2.220446049250313e-16;
// df_factor takes columns while a diagonal element of D - L L^T exceeds half of
// this, relative to dmax, and refuses a D of which one falls below minus this:
// what is left of a D of rank r after r pivots is D's own rounding, amplified by
// the pivots, which grows with n (random columns, n/5 of them, eps of dmax: 10
// at 225, 15 at 400, 22 at 800).
__host__ __device__ constexpr double factor_tol(int n) { return 32 * kEps * (n > 300 ? n / 300.0 : 1.0); }
// Bound of the corrected factor: ||D - L L^T|| <= kResidTol ||D||.  The
// exchange averages over D - L L^T: at 225 to 400 functions the relative error
// of K from it is a quarter of this or less, at most one eps, where the rounding
// of the general products gives K 2.5 to 4.5 eps.
constexpr double kResidTol = 4 * kEps;

// which sizes of a product are the rank (GemmArgs::low, SmallArgs::low)
enum : int { kRankM = 1, kRankN = 2, kRankK = 4, kRankLda = 8, kRankLdb = 16, kRankLdc = 32, kRankSlices = 64 };

struct GemmArgs {
  const Factor* fac;  // null: run; else run only when fac->ok == want
  int want;           // (-1: beside the factorisation, workgroups begin until fac->low)
  // with fac and want = 1, the sizes that are the rank r (kRank*);
  // kRankSlices: K = lda = ldb = naux r in kslices slices (K = X X^T)
  int low, naux, kslices;
  // with want = 1 and not null: the right factor (row-major, bt = 0) and sizes
  // as given where the D was refused after fac->low, so that want = -1 left
  // the product undone
  const double* Blate;
  const double* A;
  const double* B;
  double* C;
  long long lda, ldb, ldc;
  long long sA, sB, sC;
  int M, N, K;
  int bt, split, kchunk;
  int skip_lower;  // 1: tiles whose every row is below every column of C are not computed
  // 1: one-dimensional grid in an XCD-aware order.  Workgroups go to the 8
  // XCDs (each with its own L2) round-robin by block id, so block b runs on
  // XCD b % 8: split = 1 puts every tile of slice z on XCD z % 8 (the slice's
  // rows of A and B are read into one L2), split = 0 every column tile of row
  // tile m on XCD m % 8 (the row tile of A is read once).  mt, nt: tiles
  // along M and N; nz: slices.
  int xcd, mt, nt, nz;
  // 1 (NCOLS): one workgroup takes every column tile of its row tile, one after another
  // (the number of columns is the rank, which the host does not know: a
  // workgroup that finds nothing to do still takes its 55 KB of LDS, some 70 ns
  // on each XCD; X = B L of 300 functions and rank 60 0.52 -> 0.38 ms)
  int ncols;
};

template <int BM, int BN, bool NCOLS = false>
__global__ __launch_bounds__(256, 2) void dgemm_mfma(GemmArgs g) {
  if (g.fac) {  // uniform over the grid
    const int r = g.fac->rank;
    if (g.want == -1) {  // one answer for the workgroup: low may be set meanwhile
      __shared__ int low;
      if (threadIdx.x == 0) low = __hip_atomic_load(&g.fac->low, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (low > 0) return;
    } else if (g.Blate && !g.fac->ok) {
      if (g.fac->low < 0) return;
      g.B = g.Blate;
      g.bt = 0;
      g.low = 0;
    } else if (g.fac->ok != g.want)
      return;
    if (g.low & kRankN) g.N = r;
    if (g.low & kRankLdc) g.ldc = r;
    if (g.low & kRankSlices) {
      g.K = g.naux * r;
      g.lda = g.ldb = g.K;
      g.kchunk = ((g.K + g.kslices - 1) / g.kslices + KT - 1) / KT * KT;
    }
  }
  constexpr int TM = 64 * BM, TN = 16 * BN;
  constexpr int NA = TM * KT / 256;              // A entries per thread per step
  constexpr int NB = (KT * TN + 255) / 256;      // B entries per thread per step
  __shared__ double As[2][TM][KT + 1];
  __shared__ double Bs[2][KT][TN + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int mi = blockIdx.x, ni = blockIdx.y, z = blockIdx.z;
  if (g.xcd) {  // every return below is uniform over the workgroup, before any barrier
    const int b = blockIdx.x;
    if (g.split) {
      const int T = g.mt * g.nt;
      const int grp = b / (8 * T), w = b - grp * 8 * T;
      const int t = w / 8;
      z = grp * 8 + (w - t * 8);
      if (z >= g.nz) return;
      mi = t / g.nt;
      ni = t - mi * g.nt;
    } else {
      const int grp = b / (8 * g.nt), w = b - grp * 8 * g.nt;
      ni = w / 8;
      mi = grp * 8 + (w - ni * 8);
      if (mi >= g.mt) return;
      z = 0;
    }
  }
  const int m0 = mi * TM;
  int n0 = ni * TN;
  if (!NCOLS && n0 >= g.N) return;
  if (g.skip_lower && m0 > n0 + TN - 1) return;  // uniform over the workgroup, before any barrier
  const double* A = g.A;
  const double* B = g.B;
  double* C = g.C + z * g.sC;
  int kb = 0, ke = g.K;
  if (g.split) {
    kb = z * g.kchunk;
    ke = min(g.K, kb + g.kchunk);
  } else {
    A += z * g.sA;
    B += z * g.sB;
  }
  const int wm = wave * 16 * BM;
  v4d acc[BM][BN];
  double ra[NA], rb[NB];
  auto load = [&](int k0) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {  // 16 lanes per row of A
      const int e = tid + 256 * r;
      const int gm = m0 + e / KT, gk = k0 + e % KT;
      ra[r] = (gm < g.M && gk < ke) ? A[(long long)gm * g.lda + gk] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int e = tid + 256 * r;
      double x = 0.0;
      if (e < KT * TN) {
        if (g.bt) {  // rows of B^T: contiguous along the summation index
          const int gn = n0 + e / KT, gk = k0 + e % KT;
          if (gn < g.N && gk < ke) x = B[(long long)gn * g.ldb + gk];
        } else {  // rows of B: contiguous along N
          const int gk = k0 + e / TN, gn = n0 + e % TN;
          if (gn < g.N && gk < ke) x = B[(long long)gk * g.ldb + gn];
        }
      }
      rb[r] = x;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int e = tid + 256 * r;
      As[buf][e / KT][e % KT] = ra[r];
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int e = tid + 256 * r;
      if (e < KT * TN) {
        if (g.bt)
          Bs[buf][e % KT][e / KT] = rb[r];
        else
          Bs[buf][e / TN][e % TN] = rb[r];
      }
    }
  };
  do {
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  if (kb < ke) {
    load(kb);
    store(0);
  }
  __syncthreads();
  int cur = 0;
  for (int k0 = kb; k0 < ke; k0 += KT) {
    const bool more = k0 + KT < ke;
    if (more) load(k0 + KT);
#pragma unroll
    for (int kk = 0; kk < KT; kk += 4) {
      double a[BM], b[BN];
#pragma unroll
      for (int i = 0; i < BM; ++i) a[i] = As[cur][wm + 16 * i + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
      for (int j = 0; j < BN; ++j) b[j] = Bs[cur][kk + (lane >> 4)][16 * j + (lane & 15)];
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (more) store(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + (lane >> 4) + 4 * r;
        const int col = n0 + 16 * j + (lane & 15);
        if (row < g.M && col < g.N) C[(long long)row * g.ldc + col] = acc[i][j][r];
      }
  n0 += TN;
  } while (NCOLS && n0 < g.N);
}

// K[r][c] = K[c][r] for r > c (n x n, row-major)
__global__ __launch_bounds__(256) void mirror_lower(double* __restrict__ K, int n) {
  const long long nn = (long long)n * n;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < nn; i += 256ll * gridDim.x) {
    const int r = int(i / n), c = int(i - (long long)r * n);
    if (r > c) K[i] = K[(long long)c * n + r];
  }
}

// out[i] = sum over the ns slices part[z slice + i]
__global__ __launch_bounds__(256) void sum_slices(const double* __restrict__ part, long long slice, int ns,
                                                  long long n, double* __restrict__ out) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += 256ll * gridDim.x) {
    double s = 0.0;
    for (int z = 0; z < ns; ++z) s += part[z * slice + i];
    out[i] = s;
  }
}

// ---------------------------------------------------------------------------
// Coulomb passes over B[a][P][b] (both HBM-bound: one read of B each).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// part[a][P] = sum_b B[a][P][b] D[a][b]: workgroup (a, 32 rows of P), each
// wavefront 8 rows at a time (eight loads in flight per lane, lanes along b),
// then eight wavefront sums.  sym: D is symmetric, as each B_P is, so only the
// columns b >= a are read, those above a with twice the weight.
constexpr int kGammaRows = 32;
__global__ __launch_bounds__(256) void df_gamma_part(const double* __restrict__ B, const double* __restrict__ D,
                                                     int n, int naux, int sym, double* __restrict__ part) {
  const int a = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int P0 = blockIdx.y * kGammaRows + wave * 8;
  const double* Da = D + (long long)a * n;
  const double* Ba = B + ((long long)a * naux + P0) * n;
  double s[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) s[r] = 0.0;
  for (int b = (sym ? a & ~63 : 0) + lane; b < n; b += 64) {
    const double d = sym ? (b < a ? 0.0 : b == a ? Da[b] : 2.0 * Da[b]) : Da[b];
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (P0 + r < naux) s[r] = fma(Ba[(long long)r * n + b], d, s[r]);
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) s[r] = wave_sum(s[r]);
  if (lane < 8 && P0 + lane < naux) {
    double v = s[0];
#pragma unroll
    for (int r = 1; r < 8; ++r)
      if (lane == r) v = s[r];
    part[(long long)a * naux + P0 + lane] = v;
  }
}

// gamma[P] = sum_a part[a][P]: workgroup of 64 P (lanes) and 16 wavefronts,
// each summing every 16th a, then a fixed-order sum of the 16 partials.
__global__ __launch_bounds__(1024) void df_gamma_sum(const double* __restrict__ part, int n, int naux,
                                                     double* __restrict__ gamma) {
  __shared__ double red[16][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int P = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (P < naux)
    for (int a = wave; a < n; a += 16) s += part[(long long)a * naux + P];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && P < naux) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += red[w][lane];
    gamma[P] = t;
  }
}

// gamma[P] = sum_a X[a][P][a] with X[a][P][c] = sum_b B[a][P][b] D[b][c]:
// each B_P is symmetric in (a, b), so sum_ab B_P,ab D_ab = sum_ab B_P,ab D_ba =
// sum_a (B_P D)_aa for any D.  Reads the n n_aux diagonal entries of X
// instead of all of B; workgroup shape and summation order as df_gamma_sum.
__global__ __launch_bounds__(1024) void df_gamma_diag(const double* __restrict__ X, int n, int naux,
                                                      double* __restrict__ gamma) {
  __shared__ double red[16][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int P = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (P < naux)
    for (int a = wave; a < n; a += 16) s += X[((long long)a * naux + P) * n + a];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && P < naux) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) t += red[w][lane];
    gamma[P] = t;
  }
}

// The same where the device decided which X there is: part[a][P] = sum_i
// X[a][P][i] L[a][i] of X = B L (r columns; a fifth of the bytes of a pass over
// half of B; Lt holds rows of L, rmax apart), or X[a][P][a] of X = B D;
// df_gamma_sum sums over a.  A wavefront takes 32 rows, 16 lanes each.  0.37 ms
// beside the K product of 400 functions and rank 80 (with a cache line of L per
// lane 0.45 to 0.61; in the epilogue of X = B L it costs that product 0.13 ms).
__global__ __launch_bounds__(256) void df_gamma_x(const double* __restrict__ X, const double* __restrict__ Lt, int rmax,
                                                  int n, int naux, const Factor* __restrict__ fac,
                                                  double* __restrict__ part) {
  const int a = blockIdx.x, lane = threadIdx.x & 63, l16 = lane & 15;
  const int Pw = blockIdx.y * 128 + (threadIdx.x >> 6) * 32;
  const long long row0 = (long long)a * naux;
  if (!fac->ok) {
    if (lane < 32 && Pw + lane < naux) part[row0 + Pw + lane] = X[(row0 + Pw + lane) * n + a];
    return;
  }
  const int rank = fac->rank, P0 = Pw + (lane >> 4);
  double s[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) s[t] = 0.0;
  for (int i = l16; i < rank; i += 16) {
    const double l = Lt[(long long)a * rmax + i];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (P0 + 4 * t < naux) s[t] = fma(X[(row0 + P0 + 4 * t) * rank + i], l, s[t]);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) s[t] += __shfl_xor(s[t], o, 64);
    if (l16 == 0 && P0 + 4 * t < naux) part[row0 + P0 + 4 * t] = s[t];
  }
}

// J[a][b] = sum_P B[a][P][b] gamma[P] for b >= a, and J[b][a] (each B_P is
// symmetric: half of B is read, 0.45 -> 0.25 ms for 400 x 1536 x 400):
// workgroup (64 columns b, a), the four wavefronts take every fourth P (lanes
// along b, two accumulators each) and meet in LDS.
__global__ __launch_bounds__(256) void df_coulomb(const double* __restrict__ B, const double* __restrict__ gamma,
                                                  int n, int naux, double* __restrict__ J) {
  __shared__ double red[4][64];
  const int a = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.x * 64 + lane;
  if (int(blockIdx.x) * 64 + 63 < a) return;  // uniform over the workgroup
  double s0 = 0.0, s1 = 0.0;
  if (b < n && b >= a) {
    const double* Ba = B + (long long)a * naux * n + b;
    int P = wave;
    for (; P + 4 < naux; P += 8) {
      s0 = fma(Ba[(long long)P * n], gamma[P], s0);
      s1 = fma(Ba[(long long)(P + 4) * n], gamma[P + 4], s1);
    }
    if (P < naux) s0 = fma(Ba[(long long)P * n], gamma[P], s0);
  }
  red[wave][lane] = s0 + s1;
  __syncthreads();
  if (wave == 0 && b < n && b >= a) {
    const double v = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
    J[(long long)a * n + b] = v;
    J[(long long)b * n + a] = v;
  }
}

// ---------------------------------------------------------------------------
// D = L L^T by pivoted Cholesky in one workgroup: Lc[k][i] holds column k,
// Lh[k][i] the column over its pivot element dk[k].  Columns are taken while the largest diagonal element of D - L L^T exceeds
// factor_tol/2 times the largest of D, at most rmax; any order of pivots gives
// a semidefinite D of rank r in r columns.  They are taken in panels: up to
// kPanel rows whose diagonal element is at least half of the largest are the
// candidates, their columns of D - L L^T are formed in registers (a lane per
// row reads each earlier column of L once for the whole panel), and the
// candidates become pivots, largest first, until the rest of them has dropped
// below a quarter.  (Random D of rank 81 in 200: residual 11 eps; with a tenth
// and a hundredth instead 125 eps in as many panels, since small pivots amplify
// the rounding of the earlier ones.)  A step is bound by latency (two barriers and
// a few LDS reads): 0.35 ms for 80 columns of 400.
// RP rows per lane: n at most RP kFactorNT.
// ---------------------------------------------------------------------------
// From kFactorMinN functions on: J and K in ms by the general products alone,
// with a factor (a fifth of the functions), and where D is refused as indefinite
// and for its rank, water / cc-pVDZ:
//   225: 1.13 0.80 1.19 1.22   250: 1.82 0.92 1.86 1.89   300: 3.07 1.30 3.09 3.12
//   400: 7.63 2.24 7.76 7.85   600: 43.1 11.4 43.2 43.6
// (the step from 400 to 600 is B, 2.2 GB, outgrowing the cache; what a refused D
// loses are 30 us of launches that do nothing, and under 300 functions the pivoting
// beside a short X = B D).  Up to kFactorMaxN rows stay in registers.
constexpr int kFactorMaxN = 2048, kFactorMinN = 224, kFactorNT = 1024, kPanel = 16, kPanelK = 32;
template <int RP>
__global__ __launch_bounds__(kFactorNT) void df_factor(const double* __restrict__ D, int n, int rmax,
                                                       double* __restrict__ Lc, double* __restrict__ Lh,
                                                       double* __restrict__ dk, Factor* __restrict__ fac) {
  __shared__ double prow[kPanelK][kPanel];  // L[candidate][k] of a block of earlier columns
  __shared__ double pd[kPanel];             // diagonal elements of the candidates
  __shared__ double prw[kPanel];            // the pivot row of the panel
  __shared__ int cand[kPanel];
  __shared__ double wv[kFactorNT / 64];
  __shared__ int wc[kFactorNT / 64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  double diag[RP];  // of D - L L^T
  bool open[RP];    // not yet a pivot
#pragma unroll
  for (int q = 0; q < RP; ++q) {
    const int i = tid + kFactorNT * q;
    open[q] = i < n;
    diag[q] = open[q] ? D[(long long)i * n + i] : 0.0;
  }
  const double eps = factor_tol(n);
  double dmax = -1.0;
  int k = 0;
  bool low = true, full = false;
  for (;;) {
    // largest diagonal element
    double m = -1.0;
#pragma unroll
    for (int q = 0; q < RP; ++q)
      if (open[q] && diag[q] > m) m = diag[q];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if (lane == 0) wv[wave] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kFactorNT / 64; ++w) m = fmax(m, wv[w]);
    if (dmax < 0.0) dmax = m;
    // (also ends where dmax is not a positive number)
    if (!(m > 0.5 * eps * dmax) || !(dmax > 0.0)) break;
    // a negative diagonal element: indefinite (a difference of densities ends
    // here, at the first panel or soon after)
    bool neg = false;
#pragma unroll
    for (int q = 0; q < RP; ++q) neg |= open[q] && diag[q] < -eps * dmax;
    if (__syncthreads_or(neg)) {
      low = false;
      break;
    }
    // candidates, in row order: each of them may become a pivot, so every panel
    // takes at least one column and the loop ends after at most rmax panels
    const double tol = 0.5 * eps * dmax;
    const int k_panel = k;
    int nc = 0;
    for (int q = 0; q < RP; ++q) {
      const bool take = open[q] && diag[q] >= 0.5 * m && diag[q] > tol;
      const unsigned long long bal = __ballot(take);
      if (lane == 0) wc[wave] = __popcll(bal);
      __syncthreads();
      int at = nc + __popcll(bal & ((1ull << lane) - 1));
      for (int w = 0; w < kFactorNT / 64; ++w) {
        if (w < wave) at += wc[w];
        nc += wc[w];
      }
      if (take && at < kPanel) {
        cand[at] = tid + kFactorNT * q;
        pd[at] = diag[q];
      }
      __syncthreads();
    }
    nc = min(nc, kPanel);
    // their columns of D - L L^T (D is symmetric: row `candidate` of D)
    double c[RP][kPanel];
#pragma unroll
    for (int q = 0; q < RP; ++q) {
      const int i = tid + kFactorNT * q;
#pragma unroll
      for (int p = 0; p < kPanel; ++p) c[q][p] = p < nc && i < n ? D[(long long)cand[p] * n + i] : 0.0;
    }
    for (int k0 = 0; k0 < k; k0 += kPanelK) {
      const int kb = min(kPanelK, k - k0);
      for (int e = tid; e < kPanelK * kPanel; e += kFactorNT) {
        const int kk = e / kPanel, p = e - kk * kPanel;
        prow[kk][p] = kk < kb && p < nc ? Lc[(long long)(k0 + kk) * n + cand[p]] : 0.0;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < RP; ++q) {
        const int i = tid + kFactorNT * q;
        if (i < n) {
          const double* col = Lc + (long long)k0 * n + i;
#pragma unroll 4
          for (int kk = 0; kk < kb; ++kk) {
            const double l = col[(long long)kk * n];
#pragma unroll
            for (int p = 0; p < kPanel; ++p) c[q][p] = fma(-l, prow[kk][p], c[q][p]);
          }
        }
      }
      __syncthreads();
    }
    // pivots among them, largest first
    const double floor_v = fmax(tol, 0.25 * m);
    unsigned left = (1u << nc) - 1;
    for (;;) {
      double v = -1.0;
      int best = 0;
#pragma unroll
      for (int p = 0; p < kPanel; ++p) {
        const double x = pd[p];
        if ((left >> p & 1) && x > v) {
          v = x;
          best = p;
        }
      }
      if (!(v > floor_v)) break;  // uniform: every lane read the same values
      if (k == rmax) {  // (rounding left of a D of rank rmax: the residual decides)
        low = v <= 4.0 * eps * dmax;
        full = true;
        break;
      }
      const int at = cand[best];
#pragma unroll
      for (int q = 0; q < RP; ++q)
        if (at == tid + kFactorNT * q)
#pragma unroll
          for (int p = 0; p < kPanel; ++p) prw[p] = c[q][p];
      __syncthreads();
      const double inv = 1.0 / sqrt(v);
      double rp[kPanel];
#pragma unroll
      for (int p = 0; p < kPanel; ++p) rp[p] = prw[p] * inv;
#pragma unroll
      for (int q = 0; q < RP; ++q) {
        const int i = tid + kFactorNT * q;
        double x = 0.0;
#pragma unroll
        for (int p = 0; p < kPanel; ++p)
          if (p == best) x = c[q][p];
        x *= inv;
        if (i == at) {
          x = v * inv;
          open[q] = false;
        } else if (!open[q]) {
          x = 0.0;
        }
        if (i < n) {
          Lc[(long long)k * n + i] = x;
          Lh[(long long)k * n + i] = x * inv;
        }
        diag[q] -= x * x;
#pragma unroll
        for (int p = 0; p < kPanel; ++p) c[q][p] = fma(-x, rp[p], c[q][p]);
      }
      if (tid < kPanel) pd[tid] -= prw[tid] * prw[tid] / v;
      if (tid == 0) dk[k] = v * inv;
      left &= ~(1u << best);
      ++k;
      __syncthreads();  // pd is updated, prw is read
    }
    __syncthreads();  // every lane has read pd before the next panel
    if (full || k == k_panel) break;  // (no column: a diagonal element that is not finite)
  }
  if (tid == 0) {
    fac->ok = low && dmax > 0.0 && dmax < HUGE_VAL ? 1 : 0;
    fac->rank = k;
    fac->dmax = dmax;
    fac->e2 = 0.0;
    fac->d2 = 0.0;
    // (the general product ends here, not after the correction, whose small
    // kernels would wait for its workgroups: 400 functions 2.59 -> 2.34 ms)
    __hip_atomic_store(&fac->low, fac->ok ? 1 : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------------------
// Correction of the factor.  What pivoting leaves of D is small on the pivot
// rows and holds D's own rounding, amplified, everywhere else: 4 to 20 eps of
// ||D|| at 400 functions, 40 at 800, whatever precision the pivoting runs in,
// and K inherits it (relative error of K, 400 functions, graded orbital sizes:
// 3.4e-15, the general products 1.0e-15).  The nearest L L^T of the same rank
// takes E = D - L L^T to first order to (1 - P) E (1 - P), P the projection on
// the columns of L:
//   L += E Z - L (Z^T E Z) / 2,  Z = L (L^T L)^-1,
// with E summed in two doubles (df_resid).  Computed with the columns scaled
// to pivots of one (Lh), whose L^T L has a condition of 10 to 1e3; two digits
// of the correction are enough.  One step brings ||E|| to 0.8-2 eps of ||D||
// up to 400 functions; where the pivots took columns of D's rounding as well
// the second order counts and a second step is needed (800 functions: 4 and
// 8 eps after one, 1.7 and 2.7 after two).
// ---------------------------------------------------------------------------
// hi + lo -= a b, the product and the sum exact
__device__ __forceinline__ void sub_product(double& hi, double& lo, double a, double b) {
#pragma clang fp contract(off)
  const double p = a * b, e = __builtin_fma(a, b, -p);
  const double t = hi - p, v = t - hi;
  const double err = (hi - (t - v)) - (p + v);
  hi = t;
  lo += err - e;
}

// E = D - L L^T (D's upper triangle, both of E), or with LAST its norm and D's
// into fac.  32 x 32 elements per workgroup, 2 x 2 per lane, columns of L
// through LDS; 15 operations a term, 5 us of 400 functions and 80 columns.
template <bool LAST>
__global__ __launch_bounds__(256) void df_resid(const double* __restrict__ D, const double* __restrict__ Lc, int n,
                                                double* __restrict__ E, Factor* fac) {
  if (!fac->ok || blockIdx.x < blockIdx.y) return;
  constexpr int KB = 16;
  __shared__ double La[KB][32], Lb[KB][32];
  const int tid = threadIdx.x, ti = tid / 16, tj = tid % 16;
  const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32, r = fac->rank;
  double hi[2][2], lo[2][2], d[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int i = i0 + ti + 16 * x, j = j0 + tj + 16 * y;
      d[x][y] = i < n && j < n ? D[(long long)min(i, j) * n + max(i, j)] : 0.0;
      hi[x][y] = d[x][y];
      lo[x][y] = 0.0;
    }
  for (int k0 = 0; k0 < r; k0 += KB) {
    for (int e = tid; e < KB * 32; e += 256) {
      const int k = e / 32, i = e - k * 32;
      La[k][i] = k0 + k < r && i0 + i < n ? Lc[(long long)(k0 + k) * n + i0 + i] : 0.0;
      Lb[k][i] = k0 + k < r && j0 + i < n ? Lc[(long long)(k0 + k) * n + j0 + i] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KB; ++k)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) sub_product(hi[x][y], lo[x][y], La[k][ti + 16 * x], Lb[k][tj + 16 * y]);
    __syncthreads();
  }
  double e2 = 0.0, d2 = 0.0;
  const double inv = 1.0 / fac->dmax;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int i = i0 + ti + 16 * x, j = j0 + tj + 16 * y;
      if (i >= n || j >= n) continue;
      const double v = hi[x][y] + lo[x][y];
      if constexpr (LAST) {  // (tiles on the diagonal hold both triangles)
        const double w = i0 == j0 ? 1.0 : 2.0, ev = v * inv, dv = d[x][y] * inv;
        e2 += w * ev * ev;
        d2 += w * dv * dv;
      } else {
        E[(long long)i * n + j] = v;
        E[(long long)j * n + i] = v;
      }
    }
  if constexpr (LAST) {
    e2 = wave_sum(e2);
    d2 = wave_sum(d2);
    if ((tid & 63) == 0) {
      __hip_atomic_fetch_add(&fac->e2, e2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(&fac->d2, d2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// G = G^-1 in place (r x r, symmetric positive definite: Gauss-Jordan without
// pivoting) in one workgroup.  Up to 128 columns a lane holds 4 x 4 elements
// and a step costs one barrier; beyond, the matrix stays in the cache, two
// barriers and a pass over it a step.
constexpr int kInvReg = 128;
__global__ __launch_bounds__(1024) void df_invert(double* G, const Factor* __restrict__ fac) {
  if (!fac->ok) return;
  const int r = fac->rank, tid = threadIdx.x, ty = tid >> 5, tx = tid & 31;
  if (r <= kInvReg) {
    __shared__ double col[2][kInvReg], row[2][kInvReg];
    double A[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int i = ty + 32 * a, j = tx + 32 * b;
        A[a][b] = i < r && j < r ? G[i * r + j] : 0.0;
      }
    for (int k = 0; k < r; ++k) {
      const int u = k & 1;
      // row k and column k, the pivot less one in the column: with row k over
      // the pivot q, and 1 + 1/q at k, A - col row is then the step for every
      // element, row and column k among them
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (tx + 32 * m == k)
#pragma unroll
          for (int a = 0; a < 4; ++a) col[u][ty + 32 * a] = ty + 32 * a == k ? A[a][m] - 1.0 : A[a][m];
        if (ty + 32 * m == k)
#pragma unroll
          for (int b = 0; b < 4; ++b) row[u][tx + 32 * b] = A[m][b];
      }
      __syncthreads();  // (the other buffer was read before this)
      const double q = row[u][k];
      double p = __builtin_amdgcn_rcp(q);
      p = fma(p, fma(-q, p, 1.0), p);
      double c[4], x[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) c[a] = col[u][ty + 32 * a];
#pragma unroll
      for (int b = 0; b < 4; ++b) x[b] = tx + 32 * b == k ? 1.0 + p : row[u][tx + 32 * b] * p;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) A[a][b] = fma(-c[a], x[b], A[a][b]);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int i = ty + 32 * a, j = tx + 32 * b;
        if (i < r && j < r) G[i * r + j] = A[a][b];
      }
  } else {
    __shared__ double col[kFactorMaxN / 2], row[kFactorMaxN / 2];
    for (int k = 0; k < r; ++k) {
      if (tid < r) {
        col[tid] = G[(long long)tid * r + k];
        row[tid] = G[(long long)k * r + tid];
      }
      __syncthreads();
      const double p = 1.0 / row[k];
      for (int i = ty; i < r; i += 32) {
        const double c = col[i];
        double* Gi = G + (long long)i * r;
        for (int j = tx; j < r; j += 32) {
          const double x = row[j] * p;
          Gi[j] = i == k ? (j == k ? p : x) : j == k ? -c * p : fma(-c, x, Gi[j]);
        }
      }
      __syncthreads();
    }
  }
}

// The products of the correction: C = A B (BT: A B^T) of at most some hundred
// rows, rows and columns from the rank where low says so.  A workgroup computes
// 16 x 16 elements, its four wavefronts a quarter of the summation each, with
// the operands straight from the cache (dgemm_mfma has 7 tiles for 80 x 400
// and takes 40 us for a summation over 400, this 10).  UPDATE: instead of C,
// L += (F - C / 2) / dk by rows.
struct SmallArgs {
  const Factor* fac;
  int low;
  const double *A, *B;
  double* C;
  int M, N, K;
  int lda, ldb, ldc;
  const double *F, *dk;  // UPDATE: F laid out as C
  double* Lt;            // and L by columns too, column j at Lt + j ldt
  int ldt;
};
template <bool BT, bool UPDATE>
__global__ __launch_bounds__(256) void df_small(SmallArgs g) {
  if (!g.fac->ok) return;
  const int r = g.fac->rank;
  if (g.low & kRankM) g.M = r;
  if (g.low & kRankN) g.N = r;
  if (g.low & kRankK) g.K = r;
  if (g.low & kRankLda) g.lda = r;
  if (g.low & kRankLdc) g.ldc = r;
  const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
  if (m0 >= g.M || n0 >= g.N) return;
  __shared__ double part[4][16][17];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  // lane (l16, q) holds elements k0 + 4 q .. + 3 of its row of A and column of B
  // (any order of the summation index will do, if it is the same in both)
  const bool am = m0 + l16 < g.M, bn = n0 + l16 < g.N;
  const double* A = g.A + (long long)(m0 + l16) * g.lda;
  const double* B = BT ? g.B + (long long)(n0 + l16) * g.ldb : g.B + n0 + l16;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
  for (int k0 = 16 * wave; k0 < g.K; k0 += 64) {
    double a[4], b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int k = k0 + 4 * q + t;
      a[t] = am && k < g.K ? A[k] : 0.0;
      b[t] = bn && k < g.K ? (BT ? B[k] : B[(long long)k * g.ldb]) : 0.0;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[t], acc, 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) part[wave][q + 4 * t][l16] = acc[t];
  __syncthreads();
  const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
  if (m0 + i >= g.M || n0 + j >= g.N) return;
  const double v = (part[0][i][j] + part[1][i][j]) + (part[2][i][j] + part[3][i][j]);
  const long long at = (long long)(m0 + i) * g.ldc + n0 + j;
  if constexpr (UPDATE) {
    const double x = g.C[at] + (g.F[at] - 0.5 * v) / g.dk[m0 + i];
    g.C[at] = x;
    g.Lt[(long long)(n0 + j) * g.ldt + m0 + i] = x;
  } else {
    g.C[at] = v;
  }
}

// Before a factorisation: the general product may begin.
__global__ void df_open(Factor* fac) {
  __hip_atomic_store(&fac->low, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// After it: the decision.  (An e2 that is not finite refuses.)
__global__ void df_decide(Factor* fac) {
  if (!(fac->e2 < HUGE_VAL && fac->e2 <= kResidTol * kResidTol * fac->d2)) fac->ok = 0;
}

// ---------------------------------------------------------------------------
// Three-centre scatter: raw blocks of the quartets (a b|P u) of one orbital
// shell pair, P over all auxiliary shells in order, start at base; the block
// of auxiliary shell P starts na nb ps(P) further (ps = the shell's first
// auxiliary function) and is row-major [na][nb][nP].  Writes T[a][P][b] and,
// for a != b, T[b][P][a].
// ---------------------------------------------------------------------------
struct Pair3 {
  int fa, fb, na, nb;
  long long base;
  int same, pad;
};

__global__ __launch_bounds__(256) void df_scatter3(const double* __restrict__ blk, const Pair3* __restrict__ prs,
                                                   const int* __restrict__ pstart, const int* __restrict__ pn,
                                                   int naux, int n, double* __restrict__ T) {
  const Pair3 q = prs[blockIdx.x];
  const int tot = q.na * q.nb * naux;
  for (int e = threadIdx.x; e < tot; e += 256) {
    const int p = e % naux, ij = e / naux;
    const int i = ij / q.nb, j = ij - i * q.nb;
    const int ps = pstart[p], np = pn[p];
    const double v = blk[q.base + (long long)q.na * q.nb * ps + (long long)(i * q.nb + j) * np + (p - ps)];
    T[((long long)(q.fa + i) * naux + p) * n + q.fb + j] = v;
    if (!q.same) T[((long long)(q.fb + j) * naux + p) * n + q.fa + i] = v;
  }
}

template <typename T>
struct Dev {
  T* p = nullptr;
  ~Dev() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
  }
  hipError_t alloc(size_t n) {
    release();
    return hipMalloc(reinterpret_cast<void**>(&p), sizeof(T) * (n ? n : 1));
  }
  T* take() {
    T* q = p;
    p = nullptr;
    return q;
  }
};

// C tiles of 128 x 80 (BM = 2) for tall products, 64 x 80 (BM = 1) when M is
// small (the exchange product, M = n_orb).
int gemm(const GemmArgs& g0, int gz, hipStream_t st) {
  GemmArgs g = g0;
  if (g.M <= 0 || g.N <= 0 || gz <= 0) return LAI_OK;
  const bool tall = g.M >= 1024 || g.ncols;
  const int TM = tall ? 128 : 64, TN = 80;
  dim3 grid((g.M + TM - 1) / TM, (g.N + TN - 1) / TN, gz);
  if (g.ncols) grid.y = 1;
  if (g.xcd) {
    if (!g.split && gz != 1)
      return set_error(LAI_ERR_INVALID_ARGUMENT, "density fitting: XCD order needs one batch or a split product");
    g.mt = int(grid.x);
    g.nt = int(grid.y);
    g.nz = gz;
    const long long blocks = g.split ? (long long)(gz + 7) / 8 * 8 * g.mt * g.nt
                                     : (long long)(g.mt + 7) / 8 * 8 * g.nt;
    if (blocks > 0x7fffffffll)
      return set_error(LAI_ERR_INVALID_ARGUMENT, "density fitting: GEMM grid beyond the launch limits");
    grid = dim3(unsigned(blocks), 1, 1);
  }
  if (grid.y > 65535u || grid.z > 65535u)
    return set_error(LAI_ERR_INVALID_ARGUMENT, "density fitting: GEMM grid beyond the launch limits");
  if (g.ncols)
    hipLaunchKernelGGL((dgemm_mfma<2, 5, true>), grid, dim3(256), 0, st, g);
  else if (tall)
    hipLaunchKernelGGL((dgemm_mfma<2, 5>), grid, dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((dgemm_mfma<1, 5>), grid, dim3(256), 0, st, g);
  DF_HIP(hipGetLastError());
  return LAI_OK;
}

// Memory of a factorisation: factor_doubles(n) doubles at one address.
struct FactorBufs {
  double *Lc, *Lh, *Z, *F;  // [rmax][n]: L, its scaled columns, Z and E Z
  double* E;                // [n][n]: D - L L^T, and once L is corrected
  double* Lt;               // [n][rmax] in its place: the rows of L
  double *G, *H;            // [rmax][rmax]
  double* dk;               // [rmax]
  int rmax;
  FactorBufs(double* p, int n) : rmax(n / 2) {
    const size_t rn = size_t(rmax) * n, rr = size_t(rmax) * rmax;
    Lc = p;
    Lh = Lc + rn;
    Z = Lh + rn;
    F = Z + rn;
    E = Lt = F + rn;
    G = E + size_t(n) * n;
    H = G + rr;
    dk = H + rr;
  }
};
size_t factor_doubles(int n) {
  const size_t r = size_t(n / 2);
  return 4 * r * n + size_t(n) * n + 2 * r * r + r;
}

// Factors D into f.Lc and decides (fac->ok), all on st.
int factor_density(const double* D, int n, const FactorBufs& f, Factor* fac, hipStream_t st) {
  if (n <= kFactorNT)
    hipLaunchKernelGGL(df_factor<1>, dim3(1), dim3(kFactorNT), 0, st, D, n, f.rmax, f.Lc, f.Lh, f.dk, fac);
  else
    hipLaunchKernelGGL(df_factor<2>, dim3(1), dim3(kFactorNT), 0, st, D, n, f.rmax, f.Lc, f.Lh, f.dk, fac);
  DF_HIP(hipGetLastError());
  const unsigned t = unsigned((n + 31) / 32);
  const int r = f.rmax;
  // C = A B or A B^T, M rows and N columns of which the rank is as low says
  auto args = [&](const double* A, const double* B, double* C, int M, int N, int K, int low) {
    SmallArgs g{};
    g.fac = fac;
    g.low = low;
    g.A = A;
    g.B = B;
    g.C = C;
    g.M = M;
    g.N = N;
    g.K = K;
    g.lda = g.ldb = g.ldc = n;
    return g;
  };
  auto grid = [](const SmallArgs& g) { return dim3((g.N + 15) / 16, (g.M + 15) / 16); };
  const SmallArgs gram = args(f.Lh, f.Lh, f.G, r, r, n, kRankM | kRankN | kRankLdc);
  const SmallArgs z = args(f.G, f.Lh, f.Z, r, n, r, kRankM | kRankK | kRankLda);
  const SmallArgs ez = args(f.Z, f.E, f.F, r, n, n, kRankM);
  const SmallArgs h = args(f.Z, f.F, f.H, r, r, n, kRankM | kRankN | kRankLdc);
  SmallArgs up = args(f.H, f.Lh, f.Lc, r, n, r, kRankM | kRankK | kRankLda);
  up.F = f.F;
  up.dk = f.dk;
  up.Lt = f.Lt;
  up.ldt = r;
  for (int step = 0; step < (n <= 512 ? 1 : 2); ++step) {
    hipLaunchKernelGGL(df_resid<false>, dim3(t, t), dim3(256), 0, st, D, f.Lc, n, f.E, fac);
    DF_HIP(hipGetLastError());
    if (step == 0) {  // G = (Lh^T Lh)^-1, Z (the projection hardly changes)
      hipLaunchKernelGGL((df_small<true, false>), grid(gram), dim3(256), 0, st, gram);
      hipLaunchKernelGGL(df_invert, dim3(1), dim3(1024), 0, st, f.G, fac);
      hipLaunchKernelGGL((df_small<false, false>), grid(z), dim3(256), 0, st, z);
      DF_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL((df_small<false, false>), grid(ez), dim3(256), 0, st, ez);
    hipLaunchKernelGGL((df_small<true, false>), grid(h), dim3(256), 0, st, h);
    hipLaunchKernelGGL((df_small<false, true>), grid(up), dim3(256), 0, st, up);
    DF_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(df_resid<true>, dim3(t, t), dim3(256), 0, st, D, f.Lc, n, nullptr, fac);
  DF_HIP(hipGetLastError());
  hipLaunchKernelGGL(df_decide, dim3(1), dim3(1), 0, st, fac);
  DF_HIP(hipGetLastError());
  return LAI_OK;
}

// Lower Cholesky factor of the row-major SPD matrix A in place (upper part
// zeroed): the row-oriented algorithm of math::cholesky_decompose
// (include/libaccint/math/cholesky.hpp), which fails when a pivot is <= 0.
bool cholesky_lower(std::vector<double>& A, int n) {
  for (int i = 0; i < n; ++i) {
    double* Ai = &A[size_t(i) * n];
    double s = Ai[i];
    for (int k = 0; k < i; ++k) s -= Ai[k] * Ai[k];
    if (!(s > 0.0)) return false;
    Ai[i] = std::sqrt(s);
    for (int j = i + 1; j < n; ++j) {
      double* Aj = &A[size_t(j) * n];
      double t = Aj[i];
      for (int k = 0; k < i; ++k) t -= Aj[k] * Ai[k];
      Aj[i] = t / Ai[i];
    }
  }
  for (int i = 0; i < n; ++i)
    for (int j = i + 1; j < n; ++j) A[size_t(i) * n + j] = 0.0;
  return true;
}

// X = L^-1 for lower-triangular L (row-major), by forward substitution row by
// row: X[i][j] = (delta_ij - sum_{k=j}^{i-1} L[i][k] X[k][j]) / L[i][i], the
// sum taken in increasing k as in math::triangular_inverse.
void lower_inverse(const std::vector<double>& L, std::vector<double>& X, int n) {
  X.assign(size_t(n) * n, 0.0);
  std::vector<double> acc(n);
  for (int i = 0; i < n; ++i) {
    const double* Li = &L[size_t(i) * n];
    std::fill(acc.begin(), acc.begin() + i + 1, 0.0);
    acc[i] = 1.0;
    for (int k = 0; k < i; ++k) {
      const double l = Li[k];
      const double* Xk = &X[size_t(k) * n];
      for (int j = 0; j <= k; ++j) acc[j] -= l * Xk[j];
    }
    double* Xi = &X[size_t(i) * n];
    for (int j = 0; j <= i; ++j) Xi[j] = acc[j] / Li[i];
  }
}

}  // namespace

struct lai_df {
  int n = 0, naux = 0;
  int nsplit = 1, kchunk = 0;          // slices of the exchange product
  int nsplit_sym = 1, kchunk_sym = 0;  // the same over the tiles a symmetric D needs
  double* B = nullptr;     // [n][naux][n]
  double* X = nullptr;     // [n][naux][n]
  double* part = nullptr;   // nsplit * n * n: slices of the exchange product
  double* gpart = nullptr;  // [n][naux]: partial gamma
  double* gamma = nullptr;  // [naux]
  hipEvent_t ev[6] = {};
  bool have_ev = false;
  double* fbuf = nullptr;   // memory of the density's factor (FactorBufs), null where it is not tried
  Factor* fac = nullptr;
  // X = B D beside the factorisation, the Coulomb pass beside the K product
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};

namespace {
void df_release(lai_df* d) {
  if (!d) return;
  if (d->B) (void)hipFree(d->B);
  if (d->X) (void)hipFree(d->X);
  if (d->part) (void)hipFree(d->part);
  if (d->gpart) (void)hipFree(d->gpart);
  if (d->gamma) (void)hipFree(d->gamma);
  if (d->fbuf) (void)hipFree(d->fbuf);
  if (d->fac) (void)hipFree(d->fac);
  if (d->side) (void)hipStreamDestroy(d->side);
  if (d->fork) (void)hipEventDestroy(d->fork);
  if (d->join) (void)hipEventDestroy(d->join);
  if (d->have_ev)
    for (auto& e : d->ev) (void)hipEventDestroy(e);
  delete d;
}
}  // namespace

extern "C" int lai_dev_df_free(lai_df* df) {
  df_release(df);
  return LAI_OK;
}

extern "C" int lai_dev_df_dims(const lai_df* df, int* n_orb, int* n_aux) {
  if (!df) return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_dims: null handle");
  if (n_orb) *n_orb = df->n;
  if (n_aux) *n_aux = df->naux;
  return LAI_OK;
}

extern "C" int lai_dev_df_create(lai_basis* b, int n_orb_shells, int n_aux_shells, int metric,
                                 double cond_hard_limit, double* cond_estimate, lai_df** out) {
  if (!b || !out || n_orb_shells < 1 || n_aux_shells < 1)
    return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_create: invalid arguments");
  *out = nullptr;
  const lai::BasisView v = lai::basis_view(b);
  if (v.n_mol != 1 || v.ns != n_orb_shells + n_aux_shells + 1)
    return set_error(LAI_ERR_INVALID_ARGUMENT,
                     "lai_dev_df_create: the handle must hold one molecule of orbital shells, auxiliary shells "
                     "and one unit shell");
  const int u = v.ns - 1;
  if (v.L[u] != 0 || v.nprim[u] != 1 || v.exps[v.prim_off[u]] != 0.0 || v.coefs[v.prim_off[u]] != 1.0)
    return set_error(LAI_ERR_INVALID_ARGUMENT,
                     "lai_dev_df_create: the last shell must be the unit s function (exponent 0, coefficient 1)");
  if (metric == 2)
    return set_error(LAI_ERR_INVALID_ARGUMENT,
                     "AttenuatedCoulomb metric is not yet supported. Use Coulomb or Overlap metric instead.");
  if (metric != 0 && metric != 1) return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_create: unknown metric");
  const int n = v.func_off[n_orb_shells];
  const int naux = v.func_off[u] - n;
  const int a0 = n_orb_shells;  // first auxiliary shell

  // ---- metric V (host, naux x naux) ----
  std::vector<double> V(size_t(naux) * naux, 0.0);
  if (metric == 0) {
    std::vector<int> s4;
    for (int P = 0; P < n_aux_shells; ++P)
      for (int Q = P; Q < n_aux_shells; ++Q) {
        const int q[4] = {a0 + P, u, a0 + Q, u};
        s4.insert(s4.end(), q, q + 4);
      }
    const int64_t nq = int64_t(s4.size() / 4);
    std::vector<int64_t> off(nq + 1);
    int64_t tot = 0;
    for (int P = 0; P < n_aux_shells; ++P)
      for (int Q = P; Q < n_aux_shells; ++Q) tot += int64_t(ncart_of(v.L[a0 + P])) * ncart_of(v.L[a0 + Q]);
    std::vector<double> blk(static_cast<size_t>(tot));
    int rc = lai_dev_eri_quartets(b, nq, s4.data(), blk.data(), off.data());
    if (rc != LAI_OK) return rc;
    int64_t t = 0;
    for (int P = 0; P < n_aux_shells; ++P)
      for (int Q = P; Q < n_aux_shells; ++Q, ++t) {
        const int fP = v.func_off[a0 + P] - n, fQ = v.func_off[a0 + Q] - n;
        const int nP = ncart_of(v.L[a0 + P]), nQ = ncart_of(v.L[a0 + Q]);
        for (int i = 0; i < nP; ++i)
          for (int j = 0; j < nQ; ++j) {
            const double x = blk[size_t(off[t]) + size_t(i) * nQ + j];
            V[size_t(fP + i) * naux + fQ + j] = x;
            V[size_t(fQ + j) * naux + fP + i] = x;
          }
      }
  } else {
    Dev<double> dS;
    DF_HIP(dS.alloc(size_t(v.nbf) * v.nbf));
    int rc = lai_dev_onee(b, 0, 0, nullptr, nullptr, dS.p, nullptr);
    if (rc != LAI_OK) return rc;
    DF_HIP(hipDeviceSynchronize());
    std::vector<double> S(size_t(v.nbf) * v.nbf);
    DF_HIP(hipMemcpy(S.data(), dS.p, sizeof(double) * S.size(), hipMemcpyDeviceToHost));
    for (int i = 0; i < naux; ++i)
      for (int j = 0; j < naux; ++j) V[size_t(i) * naux + j] = S[size_t(n + i) * v.nbf + n + j];
  }
  double dmax = 0.0, dmin = HUGE_VAL;
  for (int i = 0; i < naux; ++i) {
    const double d = V[size_t(i) * naux + i];
    dmax = std::max(dmax, d);
    if (d > 0.0) dmin = std::min(dmin, d);
  }
  const double cond = dmin < HUGE_VAL ? dmax / dmin : HUGE_VAL;
  if (cond_estimate) *cond_estimate = cond;
  if (cond_hard_limit > 0.0 && cond > cond_hard_limit)
    return set_error(LAI_ERR_INVALID_ARGUMENT,
                     "DF metric matrix is severely ill-conditioned (condition estimate = " + std::to_string(cond) +
                         ", hard limit = " + std::to_string(cond_hard_limit) + ")");
  if (!cholesky_lower(V, naux))
    return set_error(LAI_ERR_NUMERIC, "Cholesky decomposition failed: matrix is not positive definite");
  std::vector<double> Linv;
  lower_inverse(V, Linv, naux);
  V.clear();
  V.shrink_to_fit();

  // ---- three-centre integrals T[a][P][b] ----
  std::vector<int> pstart(naux), pn(naux);
  for (int P = 0; P < n_aux_shells; ++P) {
    const int f = v.func_off[a0 + P] - n, m = ncart_of(v.L[a0 + P]);
    for (int i = 0; i < m; ++i) {
      pstart[f + i] = f;
      pn[f + i] = m;
    }
  }
  const size_t nB = size_t(n) * naux * n;
  Dev<double> dT, dLinv, dB;
  Dev<int> dps, dpn;
  DF_HIP(dT.alloc(nB));
  DF_HIP(dps.alloc(naux));
  DF_HIP(dpn.alloc(naux));
  DF_HIP(hipMemcpy(dps.p, pstart.data(), sizeof(int) * naux, hipMemcpyHostToDevice));
  DF_HIP(hipMemcpy(dpn.p, pn.data(), sizeof(int) * naux, hipMemcpyHostToDevice));
  {
    // orbital shell pairs in batches of at most ~4M quartets / 64M doubles
    const int64_t kMaxQ = int64_t(1) << 22, kMaxD = int64_t(1) << 26;
    std::vector<std::pair<int, int>> pairs;
    for (int i = 0; i < n_orb_shells; ++i)
      for (int j = i; j < n_orb_shells; ++j) pairs.emplace_back(i, j);
    size_t p0 = 0;
    Dev<double> dblk;
    Dev<Pair3> dpr;
    int64_t blk_cap = 0, pr_cap = 0;
    while (p0 < pairs.size()) {
      size_t p1 = p0;
      int64_t nq = 0, nd = 0;
      while (p1 < pairs.size()) {
        const int64_t d = int64_t(ncart_of(v.L[pairs[p1].first])) * ncart_of(v.L[pairs[p1].second]) * naux;
        if (p1 > p0 && (nq + n_aux_shells > kMaxQ || nd + d > kMaxD)) break;
        nq += n_aux_shells;
        nd += d;
        ++p1;
      }
      std::vector<int> s4;
      s4.reserve(size_t(nq) * 4);
      std::vector<Pair3> prs;
      int64_t base = 0;
      for (size_t p = p0; p < p1; ++p) {
        const int i = pairs[p].first, j = pairs[p].second;
        Pair3 r{};
        r.fa = v.func_off[i];
        r.fb = v.func_off[j];
        r.na = ncart_of(v.L[i]);
        r.nb = ncart_of(v.L[j]);
        r.base = base;
        r.same = (i == j);
        prs.push_back(r);
        base += int64_t(r.na) * r.nb * naux;
        for (int P = 0; P < n_aux_shells; ++P) {
          const int q[4] = {i, j, a0 + P, u};
          s4.insert(s4.end(), q, q + 4);
        }
      }
      if (nd > blk_cap) {
        DF_HIP(dblk.alloc(size_t(nd)));
        blk_cap = nd;
      }
      if (int64_t(prs.size()) > pr_cap) {
        DF_HIP(dpr.alloc(prs.size()));
        pr_cap = int64_t(prs.size());
      }
      std::vector<int64_t> off(size_t(nq) + 1);
      int rc = lai_dev_eri_quartets_device(b, nq, s4.data(), dblk.p, off.data(), nullptr);
      if (rc != LAI_OK) return rc;
      if (off[size_t(nq)] != nd)
        return set_error(LAI_ERR_BACKEND, "lai_dev_df_create: three-centre block layout mismatch");
      DF_HIP(hipMemcpy(dpr.p, prs.data(), sizeof(Pair3) * prs.size(), hipMemcpyHostToDevice));
      hipLaunchKernelGGL(df_scatter3, dim3(unsigned(prs.size())), dim3(256), 0, nullptr, dblk.p, dpr.p, dps.p, dpn.p,
                         naux, n, dT.p);
      DF_HIP(hipGetLastError());
      DF_HIP(hipDeviceSynchronize());
      p0 = p1;
    }
  }

  // ---- B[a] = L^-1 T[a] ----
  DF_HIP(dLinv.alloc(size_t(naux) * naux));
  DF_HIP(hipMemcpy(dLinv.p, Linv.data(), sizeof(double) * Linv.size(), hipMemcpyHostToDevice));
  DF_HIP(dB.alloc(nB));
  {
    GemmArgs g{};
    g.A = dLinv.p;
    g.B = dT.p;
    g.C = dB.p;
    g.lda = naux;
    g.ldb = n;
    g.ldc = n;
    g.sA = 0;
    g.sB = (long long)naux * n;
    g.sC = (long long)naux * n;
    g.M = naux;
    g.N = n;
    g.K = naux;
    int rc = gemm(g, n, nullptr);
    if (rc != LAI_OK) return rc;
    DF_HIP(hipDeviceSynchronize());
  }
  dT.release();
  dLinv.release();

  auto* d = new lai_df;
  d->n = n;
  d->naux = naux;
  // slices of the exchange GEMM: about 2048 workgroups (8 per CU) over its
  // tiles, all of them or those a symmetric D needs (gemm's tile rule)
  const int TMk = n >= 1024 ? 128 : 64, TNk = 80;
  long long tiles = 0, tiles_sym = 0;
  for (int mi = 0; mi < (n + TMk - 1) / TMk; ++mi)
    for (int ni = 0; ni < (n + TNk - 1) / TNk; ++ni) {
      ++tiles;
      if (!(mi * TMk > ni * TNk + TNk - 1)) ++tiles_sym;
    }
  const long long ksum = (long long)naux * n;
  auto slices = [&](long long t, int& ns_out, int& kc_out) {
    int ns = int(std::max(1ll, std::min(std::max(1ll, 2048ll / t), (ksum + 16 * KT - 1) / (16 * KT))));
    long long kc = (ksum + ns - 1) / ns;
    kc = (kc + KT - 1) / KT * KT;
    ns_out = int((ksum + kc - 1) / kc);
    kc_out = int(kc);
  };
  slices(tiles, d->nsplit, d->kchunk);
  slices(tiles_sym, d->nsplit_sym, d->kchunk_sym);
  const int ns = std::max(d->nsplit, d->nsplit_sym);
  Dev<double> dX, dpart, dgp, dg;
  hipError_t e;
  if ((e = dX.alloc(nB)) != hipSuccess || (e = dpart.alloc(size_t(ns) * n * n)) != hipSuccess ||
      (e = dgp.alloc(size_t(n) * naux)) != hipSuccess || (e = dg.alloc(size_t(naux))) != hipSuccess) {
    delete d;
    return set_error(LAI_ERR_MEMORY, std::string("lai_dev_df_create: ") + hipGetErrorString(e));
  }
  d->B = dB.take();
  d->X = dX.take();
  d->part = dpart.take();
  d->gpart = dgp.take();
  d->gamma = dg.take();
  // the density is factored where the exchange GEMMs are worth it: see the
  // times beside kFactorMinN
  if (n >= kFactorMinN && n <= kFactorMaxN) {
    Dev<double> dl;
    Dev<Factor> df;
    if ((e = dl.alloc(factor_doubles(n))) != hipSuccess || (e = df.alloc(1)) != hipSuccess ||
        (e = hipMemset(df.p, 0, sizeof(Factor))) != hipSuccess) {
      df_release(d);
      return set_error(LAI_ERR_MEMORY, std::string("lai_dev_df_create: ") + hipGetErrorString(e));
    }
    d->fbuf = dl.take();
    d->fac = df.take();
  }
  if ((e = hipStreamCreateWithFlags(&d->side, hipStreamNonBlocking)) != hipSuccess ||
      (e = hipEventCreateWithFlags(&d->fork, hipEventDisableTiming)) != hipSuccess ||
      (e = hipEventCreateWithFlags(&d->join, hipEventDisableTiming)) != hipSuccess) {
    df_release(d);
    return set_error(LAI_ERR_BACKEND, std::string("lai_dev_df_create: ") + hipGetErrorString(e));
  }
  *out = d;
  return LAI_OK;
}

namespace {
int df_run(lai_df* d, const double* D, double* J, double* K, int flags, hipStream_t st, double* ms) {
  const int n = d->n, naux = d->naux;
  auto mark = [&](int i) -> int {
    if (ms) DF_HIP(hipEventRecord(d->ev[i], st));
    return LAI_OK;
  };
  // ms[out] = time between events i0 and i1 (recorded on st, serial in the profiled runs)
  auto take = [&](int i0, int i1, int out) -> int {
    if (!ms) return LAI_OK;
    float t;
    DF_HIP(hipEventSynchronize(d->ev[i1]));
    DF_HIP(hipEventElapsedTime(&t, d->ev[i0], d->ev[i1]));
    ms[out] = t;
    return LAI_OK;
  };
  if (ms && !d->have_ev) {
    for (auto& e : d->ev) DF_HIP(hipEventCreate(&e));
    d->have_ev = true;
  }
  if (ms)
    for (int i = 0; i < 5; ++i) ms[i] = 0.0;
  const bool both = (flags & LAI_DF_J) && (flags & LAI_DF_K);
  const int sym = (flags & LAI_DF_SYMMETRIC) ? 1 : 0;
  const bool factor = (flags & LAI_DF_K) && sym && d->fbuf;  // the exchange from a factor of D, if there is one
  const FactorBufs fb(d->fbuf, n);
  auto coulomb = [&](hipStream_t s) -> int {
    hipLaunchKernelGGL(df_coulomb, dim3((n + 63) / 64, n), dim3(256), 0, s, d->B, d->gamma, n, naux, J);
    DF_HIP(hipGetLastError());
    return LAI_OK;
  };
  auto gamma_sum = [&](hipStream_t s) -> int {
    hipLaunchKernelGGL(df_gamma_sum, dim3((naux + 63) / 64), dim3(1024), 0, s, d->gpart, n, naux, d->gamma);
    DF_HIP(hipGetLastError());
    return LAI_OK;
  };
  auto gamma_pass = [&](hipStream_t s) -> int {
    hipLaunchKernelGGL(df_gamma_part, dim3(n, (naux + kGammaRows - 1) / kGammaRows), dim3(256), 0, s, d->B, D, n, naux,
                       sym, d->gpart);
    DF_HIP(hipGetLastError());
    return gamma_sum(s);
  };
  auto gamma_of_x = [&](hipStream_t s) -> int {  // the fitted density from X, whichever it is
    if (!factor) {
      hipLaunchKernelGGL(df_gamma_diag, dim3((naux + 63) / 64), dim3(1024), 0, s, d->X, n, naux, d->gamma);
      DF_HIP(hipGetLastError());
      return LAI_OK;
    }
    hipLaunchKernelGGL(df_gamma_x, dim3(n, (naux + 127) / 128), dim3(256), 0, s, d->X, fb.Lt, fb.rmax, n, naux, d->fac,
                       d->gpart);
    DF_HIP(hipGetLastError());
    return gamma_sum(s);
  };
  auto x_low = [&](const double* late = nullptr) -> int {  // X = B L (or B late: GemmArgs::Blate)
    GemmArgs g{};
    g.fac = d->fac;
    g.want = 1;
    g.low = kRankN | kRankLdc;
    g.A = d->B;
    g.B = fb.Lc;  // given transposed: rows i, columns b
    g.bt = 1;
    g.C = d->X;
    g.lda = n;
    g.ldb = n;
    g.M = n * naux;
    g.Blate = late;
    g.ncols = 1;
    g.N = n;
    g.ldc = n;
    g.K = n;
    g.xcd = 1;
    return gemm(g, 1, st);
  };
  auto x_gemm = [&](hipStream_t s, int want) -> int {  // X = B D
    GemmArgs g{};
    g.fac = factor ? d->fac : nullptr;
    g.want = want;
    g.A = d->B;  // rows (a, P), n columns
    g.B = D;
    g.C = d->X;
    g.lda = n;
    g.ldb = n;
    g.ldc = n;
    g.M = n * naux;
    g.N = n;
    g.K = n;
    g.xcd = 1;
    return gemm(g, 1, s);
  };
  auto k_product = [&]() -> int {  // K = X B^T over (P, b), then the slice sum
    int rc = mark(3);
    if (rc) return rc;
    const int nsym = d->nsplit_sym;
    if (factor) {  // K = X X^T over (P, i)
      GemmArgs h{};
      h.fac = d->fac;
      h.want = 1;
      h.low = kRankSlices;
      h.naux = naux;
      h.kslices = nsym;
      h.A = d->X;
      h.B = d->X;
      h.C = d->part;
      h.ldc = n;
      h.sC = (long long)n * n;
      h.M = n;
      h.N = n;
      h.bt = 1;
      h.split = 1;
      h.skip_lower = 1;
      h.xcd = 1;
      if ((rc = gemm(h, nsym, st))) return rc;
    }
    GemmArgs h{};
    h.fac = factor ? d->fac : nullptr;  // want = 0
    h.A = d->X;  // rows a, summation (P, b)
    h.B = d->B;  // given transposed: rows c, summation (P, b)
    h.C = d->part;
    h.lda = (long long)naux * n;
    h.ldb = (long long)naux * n;
    h.ldc = n;
    h.sC = (long long)n * n;
    h.M = n;
    h.N = n;
    h.K = naux * n;
    h.bt = 1;
    h.split = 1;
    h.skip_lower = (flags & LAI_DF_SYMMETRIC) ? 1 : 0;
    h.xcd = 1;
    h.kchunk = h.skip_lower ? d->kchunk_sym : d->kchunk;
    const int nsl = h.skip_lower ? d->nsplit_sym : d->nsplit;
    if ((rc = gemm(h, nsl, st))) return rc;
    if ((rc = mark(4))) return rc;
    const long long nn = (long long)n * n;
    hipLaunchKernelGGL(sum_slices, dim3(unsigned(std::min(2048ll, (nn + 255) / 256))), dim3(256), 0, st, d->part, nn,
                       nsl, nn, K);
    DF_HIP(hipGetLastError());
    if (flags & LAI_DF_SYMMETRIC) {  // the skipped tiles hold stale slices: take the upper triangle
      hipLaunchKernelGGL(mirror_lower, dim3(unsigned(std::min(2048ll, (nn + 255) / 256))), dim3(256), 0, st, K, n);
      DF_HIP(hipGetLastError());
    }
    if ((rc = mark(5))) return rc;
    if ((rc = take(3, 4, 3))) return rc;
    return take(4, 5, 4);
  };
  // st waits for the side stream, on error returns too
  auto join_side = [&](int rc) -> int {
    const hipError_t e1 = hipEventRecord(d->join, d->side);
    const hipError_t e2 = e1 == hipSuccess ? hipStreamWaitEvent(st, d->join, 0) : e1;
    if (e2 != hipSuccess) {
      (void)hipStreamSynchronize(d->side);  // no event edge: order by waiting on the host
      if (rc == LAI_OK)
        rc = set_error(LAI_ERR_BACKEND, std::string("lai_dev_df_jk: join: ") + hipGetErrorString(e2));
    }
    return rc;
  };
  auto fork_side = [&]() -> int {
    DF_HIP(hipEventRecord(d->fork, st));
    DF_HIP(hipStreamWaitEvent(d->side, d->fork, 0));
    return LAI_OK;
  };
  const bool overlap = !ms && d->side;  // not profiled
  // X: B D, or from a factor of D
  auto x_product = [&]() -> int {
    int r;
    if (!factor) return x_gemm(st, 0);
    if (!overlap) {
      if ((r = factor_density(D, n, fb, d->fac, st)) || (r = x_low())) return r;
      return x_gemm(st, 0);
    }
    // beside the factorisation, which is one workgroup, X = B D, whose
    // workgroups begin until pivoting has ended well: a density that is refused
    // loses little
    hipLaunchKernelGGL(df_open, dim3(1), dim3(1), 0, st, d->fac);
    DF_HIP(hipGetLastError());
    if ((r = fork_side())) return r;
    if ((r = factor_density(D, n, fb, d->fac, st)) == LAI_OK) r = x_gemm(d->side, -1);
    r = join_side(r);
    return r ? r : x_low(D);
  };
  int rc;
  if (both) {
    // X first: J's fitted density comes from it, so B is read twice per build
    // (X, Coulomb pass) plus, where there is no factor, once more with X by the
    // K product.  The Coulomb pass (HBM-bound) runs on the side stream beside
    // the K product (matrix cores), joined back into st.
    const hipStream_t sj = overlap ? d->side : st;
    if ((rc = mark(0))) return rc;
    if ((rc = x_product())) return rc;
    if ((rc = mark(1))) return rc;
    if ((rc = take(0, 1, 2))) return rc;
    if (overlap && (rc = fork_side())) return rc;
    // from here on st is joined to the side stream on every return path, so
    // that a failed launch never leaves work writing J or gamma unordered
    // with the caller's stream
    auto side_part = [&]() -> int {
      int r;
      if ((r = mark(0))) return r;
      if ((r = gamma_of_x(sj))) return r;
      if ((r = mark(1))) return r;
      if ((r = coulomb(sj))) return r;
      if ((r = mark(2))) return r;
      if ((r = take(0, 1, 0)) || (r = take(1, 2, 1))) return r;
      return k_product();
    };
    rc = side_part();
    return overlap ? join_side(rc) : rc;
  }
  if (flags & LAI_DF_J) {  // J alone: the fitted density from one pass over B
    if ((rc = mark(0))) return rc;
    if ((rc = gamma_pass(st))) return rc;
    if ((rc = mark(1))) return rc;
    if ((rc = coulomb(st))) return rc;
    if ((rc = mark(2))) return rc;
    if ((rc = take(0, 1, 0)) || (rc = take(1, 2, 1))) return rc;
  }
  if (flags & LAI_DF_K) {
    if ((rc = mark(0))) return rc;
    if ((rc = x_product())) return rc;
    if ((rc = mark(1))) return rc;
    if ((rc = take(0, 1, 2))) return rc;
    if ((rc = k_product())) return rc;
  }
  return LAI_OK;
}
}  // namespace

extern "C" int lai_dev_df_factor_info(const lai_df* df, int* accepted, int* rank) {
  if (!df || !accepted || !rank)
    return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_factor_info: invalid arguments");
  Factor f{};
  f.ok = -1;
  if (df->fac) {
    DF_HIP(hipDeviceSynchronize());
    DF_HIP(hipMemcpy(&f, df->fac, sizeof(f), hipMemcpyDeviceToHost));
  }
  *accepted = f.ok;
  *rank = f.rank;
  return LAI_OK;
}

extern "C" int lai_dev_df_factor(const double* d_D, int n, double* d_L, int* accepted, int* rank, double* residual) {
  if (!d_D || !d_L || !accepted || !rank || !residual || n < 2 || n > kFactorMaxN)
    return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_factor: invalid arguments");
  Dev<double> buf;
  Dev<Factor> fac;
  hipError_t e;
  if ((e = buf.alloc(factor_doubles(n))) != hipSuccess || (e = fac.alloc(1)) != hipSuccess)
    return set_error(LAI_ERR_MEMORY, std::string("lai_dev_df_factor: ") + hipGetErrorString(e));
  const FactorBufs f(buf.p, n);
  const int rc = factor_density(d_D, n, f, fac.p, nullptr);
  DF_HIP(hipDeviceSynchronize());
  if (rc != LAI_OK) return rc;
  Factor h{};
  DF_HIP(hipMemcpy(&h, fac.p, sizeof(h), hipMemcpyDeviceToHost));
  DF_HIP(hipMemcpy(d_L, f.Lc, sizeof(double) * size_t(f.rmax) * n, hipMemcpyDeviceToDevice));
  *accepted = h.ok;
  *rank = h.rank;
  *residual = std::sqrt(h.e2 / h.d2);
  return LAI_OK;
}

extern "C" int lai_dev_df_jk(lai_df* df, const double* d_D, double* d_J, double* d_K, int flags, void* stream) {
  if (!df || !d_D || (flags & ~(LAI_DF_J | LAI_DF_K | LAI_DF_SYMMETRIC)) || ((flags & LAI_DF_J) && !d_J) ||
      ((flags & LAI_DF_K) && !d_K))
    return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_jk: invalid arguments");
  return df_run(df, d_D, d_J, d_K, flags, hipStream_t(stream), nullptr);
}

extern "C" int lai_dev_df_jk_profile(lai_df* df, const double* d_D, double* d_J, double* d_K, int flags,
                                     void* stream, double* ms) {
  if (!df || !d_D || !ms || (flags & ~(LAI_DF_J | LAI_DF_K | LAI_DF_SYMMETRIC)) || ((flags & LAI_DF_J) && !d_J) ||
      ((flags & LAI_DF_K) && !d_K))
    return set_error(LAI_ERR_INVALID_ARGUMENT, "lai_dev_df_jk_profile: invalid arguments");
  return df_run(df, d_D, d_J, d_K, flags, hipStream_t(stream), ms);
}
