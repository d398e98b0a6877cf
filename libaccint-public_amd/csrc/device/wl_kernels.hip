// wl_kernels.hip -- worklist order, statistics and the last step of a J/K build.
#include "wl_kernels.hpp"

namespace lai {

__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One lane per quartet over the chunks of one class, 256 lanes per chunk.
__global__ __launch_bounds__(256) void worklist_stats_kernel(WlStatsArgs a) {
  const int tid = threadIdx.x;
  unsigned long long n = 0, n32 = 0, neri = 0, sum = 0;
  double fm64 = 0.0, fm32 = 0.0, fx64 = 0.0, fx32 = 0.0, g0 = 0.0, g1 = 0.0;
  for (int ci = blockIdx.x; ci < a.nchunks; ci += gridDim.x) {
    const JkChunk ch = a.chunks[ci];
    const PairRec bra = a.pairs[ch.bra];
    const JkSegs* sg = a.segs + ch.seg;
    for (int k = ch.k0 + tid; k < ch.k1; k += blockDim.x) {
      const int kp = chunk_ket(sg, k);
      const PairRec ket = a.pairs[kp];
      const int mode = quartet_select(a.sel, ch.bra, bra, kp, ket);
      if (mode == 0) continue;
      // reference orientation: each pair's shells in index order, and the pair
      // whose shells come first (in that order) first
      int i = min(bra.sa, bra.sb), j = max(bra.sa, bra.sb), kk = min(ket.sa, ket.sb), l = max(ket.sa, ket.sb);
      if (kk < i || (kk == i && l < j)) {
        int t = i;
        i = kk;
        kk = t;
        t = j;
        j = l;
        l = t;
      }
      const unsigned long long key =
          ((unsigned long long)(unsigned short)a.sel.sh_loc[i] << 48) |
          ((unsigned long long)(unsigned short)a.sel.sh_loc[j] << 32) |
          ((unsigned long long)(unsigned short)a.sel.sh_loc[kk] << 16) |
          (unsigned long long)(unsigned short)a.sel.sh_loc[l];
      sum += mix64(key);
      const int Li = a.L[i], Lj = a.L[j], Lk = a.L[kk], Ll = a.L[l];
      const double F = a.fp[((Li * 4 + Lj) * 4 + Lk) * 4 + Ll];
      const double fm = double(bra.npp) * ket.npp * F, fx = double(bra.npp_sig) * ket.npp_sig * F;
      const int gi = ((Li * 4 + Lj) * 4 + Lk) * 4 + Ll;
      g0 += double(bra.npp_sig) * ket.npp_sig * a.fg[gi];
      g1 += double(bra.npp_sig) * ket.npp_sig * a.fg[256 + gi];
      neri += (unsigned long long)(ncart(Li) * ncart(Lj)) * (ncart(Lk) * ncart(Ll));
      ++n;
      if (mode == 2) {
        ++n32;
        fm32 += fm;
        fx32 += fx;
      } else {
        fm64 += fm;
        fx64 += fx;
      }
    }
  }
  n = wave_sum_u64(n);
  n32 = wave_sum_u64(n32);
  neri = wave_sum_u64(neri);
  sum = wave_sum_u64(sum);
  fm64 = wave_sum(fm64);
  fm32 = wave_sum(fm32);
  fx64 = wave_sum(fx64);
  fx32 = wave_sum(fx32);
  g0 = wave_sum(g0);
  g1 = wave_sum(g1);
  if ((tid & 63) == 0 && n > 0) {
    atomic_add(&a.gflops[2 * a.cls], g0);
    atomic_add(&a.gflops[2 * a.cls + 1], g1);
    atomicAdd(&a.counts[3 * a.cls], n);
    atomicAdd(&a.counts[3 * a.cls + 1], n32);
    atomicAdd(&a.counts[3 * a.cls + 2], neri);
    atomicAdd(a.checksum, sum);  // modulo 2^64
    atomic_add(&a.flops[4 * a.cls], fm64);
    atomic_add(&a.flops[4 * a.cls + 1], fm32);
    atomic_add(&a.flops[4 * a.cls + 2], fx64);
    atomic_add(&a.flops[4 * a.cls + 3], fx32);
  }
}

__global__ void gather_pairs_kernel(const PairRec* __restrict__ pairs, const int* __restrict__ order, int n,
                                    PairRec* __restrict__ out) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) out[p] = pairs[order[p]];
}

// Element (i, j) of the symmetrised Coulomb matrix from the pair blocks: a
// pair of two shells holds its block once, a pair of a shell with itself the
// whole square.
__device__ __forceinline__ double finish_j(const FinishArgs& a, int m, int i, int j) {
  const int f0 = a.mfunc[m], s0 = a.mshell[m];
  const int si = a.fsh[f0 + i], sj = a.fsh[f0 + j];
  const int ns = a.mshell[m + 1] - s0;
  const int lo = min(si, sj), hi = max(si, sj);
  const double* blk = a.Jl + a.jloc[a.mpair[m] + lo * ns - lo * (lo - 1) / 2 + (hi - lo)];
  const int xi = i - a.func_off[s0 + si], xj = j - a.func_off[s0 + sj];
  if (si == sj) {
    const int nf = ncart(a.L[s0 + si]);
    return 0.5 * (blk[xi * nf + xj] + blk[xj * nf + xi]);
  }
  // class order: the shell of larger angular momentum first, the earlier one
  // where they are equal
  const bool i_first = a.L[s0 + si] != a.L[s0 + sj] ? a.L[s0 + si] > a.L[s0 + sj] : si < sj;
  return 0.5 * (i_first ? blk[xi * ncart(a.L[s0 + sj]) + xj] : blk[xj * ncart(a.L[s0 + si]) + xi]);
}

// Bound by the transposed reads of Kt and the gathered pair blocks (1010
// functions: 8 MB each, a few tens of microseconds of a 50 ms build).
__global__ void finish_jk_kernel(FinishArgs a, int anti) {
  const int m = blockIdx.y;
  const int n = a.mnbf[m];
  const size_t o = size_t(a.moff[m]);
  for (int i = blockIdx.x; i < n; i += gridDim.x)
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
      const size_t x = o + size_t(i) * n + j, t = o + size_t(j) * n + i;
      if (anti) {
        a.K[x] += 0.5 * (a.Kt[x] - a.Kt[t]);
      } else {
        a.J[x] += finish_j(a, m, i, j);
        a.K[x] += 0.5 * (a.Kt[x] + a.Kt[t]);
      }
    }
}

}  // namespace lai
