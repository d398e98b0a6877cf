// wl_kernels.hpp -- device passes over the implicit worklist: the pair records
// in list order, per-class
// statistics (quartet and ERI counts, the order-independent list checksum,
// the FLOP model of the reference recursion) with the same per-quartet
// selection the J/K kernels apply, and the J/K matrices from the accumulators.
#pragma once

#include "eri_kernels.hpp"

namespace lai {

struct WlStatsArgs {
  const JkChunk* __restrict__ chunks;
  int nchunks;
  const JkSegs* __restrict__ segs;
  const PairRec* __restrict__ pairs;  // in list order
  QuartetSel sel;
  const int* __restrict__ L;      // angular momentum per shell
  const double* __restrict__ fp;  // F_prim[La][Lb][Lc][Ld], 4^4 entries, reference orientation
  int cls;
  // outputs, accumulated: per class [count, fp32 count, ERIs] and
  // [model flops FP64, FP32, executed flops FP64, FP32]; the checksum
  unsigned long long* counts;  // [kNumClasses][3]
  double* flops;               // [kNumClasses][4]
  unsigned long long* checksum;
  // gradient work per primitive quartet, two models ([La][Lb][Lc][Ld], 4^4
  // each), and the per-class sums over the executed primitive pairs of every
  // selected quartet ([kNumClasses][2])
  const double* __restrict__ fg;
  double* gflops;
};

__global__ void worklist_stats_kernel(WlStatsArgs a);

// out[p] = pairs[order[p]]: the pair records in list order
__global__ void gather_pairs_kernel(const PairRec* __restrict__ pairs, const int* __restrict__ order, int n,
                                    PairRec* __restrict__ out);

// Where the functions of a handle lie, for finish_jk_kernel.
struct FinishArgs {
  const double* __restrict__ Jl;       // Coulomb blocks of the pairs in list order
  const long long* __restrict__ jloc;  // per pair (reference order): its block in Jl
  const double* __restrict__ Kt;
  double* __restrict__ J;
  double* __restrict__ K;
  const long long* __restrict__ moff;  // per molecule: its matrices
  const int* __restrict__ mnbf;
  const int* __restrict__ mpair;       // per molecule: first pair, first shell, first function
  const int* __restrict__ mshell;
  const int* __restrict__ mfunc;
  const int* __restrict__ fsh;         // per function: its shell within the molecule
  const int* __restrict__ L;           // per shell
  const int* __restrict__ func_off;    // per shell: first function within the molecule
};

// J[m] += (Jt[m] + Jt[m]^T)/2 from the pair blocks, K[m] += (Kt[m] +
// Kt[m]^T)/2, for every molecule block m (blockIdx.y = molecule); with anti !=
// 0 (an antisymmetric density) only K[m] += (Kt[m] - Kt[m]^T)/2
__global__ void finish_jk_kernel(FinishArgs a, int anti);

}  // namespace lai
