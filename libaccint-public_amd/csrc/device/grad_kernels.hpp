// grad_kernels.hpp -- nuclear gradient of E = 1/2 tr(DJ) - x/4 tr(DK) for a
// fixed AO density, contracted on the fly (derivative integrals are recomputed,
// never stored).
//
// For a canonical quartet q with orbit size deg(q) = s_ij s_kl s_bk, the
// contribution to dE/dR is
//   deg(q) sum_abcd d(ab|cd)/dR * W_abcd,
//   W_abcd = 1/2 D_ab D_cd - x/8 (D_ac D_bd + D_ad D_bc)
// (the orbit average of the J and K weights).  Per primitive quartet three
// derivatives are contracted, from which all four forces follow:
//   A  : d/dA_x phi_a = 2 alpha phi_{a+1x} - a_x phi_{a-1x}, from the Rys 2D
//        tables built one unit higher in a;
//   C  : likewise, one unit higher in c;
//   AB : moving A and B together moves P - Q alone.  A 2D integral depends on
//        it through exp(-rho u (P-Q)^2), PA_eff = PA - (rho/zeta) u (P-Q) and
//        QC_eff = QC + (rho/eta) u (P-Q), and d/dPA_eff lowers a or b,
//        d/dQC_eff lowers c or d:
//        dI = -2 rho u (P-Q) I - (rho/zeta) u (a I_{a-1} + b I_{b-1})
//             + (rho/eta) u (c I_{c-1} + d I_{d-1}),  nothing raised.
// B = AB - A, and by translational invariance D = -AB - C.  (Raising b as well
// instead of the AB derivative makes the tables (Lb+2)/(Lb+1) larger: 36
// instead of 22 entries an axis for (dp|ps), 8 instead of 3 for (ss|ss).)
// Shapes (GradPolicy): a lane per shell quartet and bra slice with tables and
// weights W in registers, for all classes but (dd|dp) and (dd|dd), which take a
// workgroup per quartet, (root, axis) tables and W in LDS, each lane a strided
// subset of the Cartesian components.
#pragma once

#include "eri_kernels.hpp"

namespace lai {

struct GradArgs {
  const PairRec* __restrict__ pairs;  // in list order
  const PrimPair* __restrict__ pp;
  const double2* __restrict__ ppab;  // exponents (alpha_a, alpha_b) of each primitive pair
  const double* __restrict__ rys;
  const double* __restrict__ D;
  int nbf;
  double xscale;
  const int* __restrict__ shell_atom;
  double* grad;
  int n_atoms;
  int glds;  // 1: each workgroup sums its quartets' forces in LDS ([3 * n_atoms])
  // the J/K worklist: bra-anchored chunks over ket segments
  const JkChunk* __restrict__ chunks;
  int nchunks;
  const JkSegs* __restrict__ segs;
  QuartetSel sel;
  const double* __restrict__ ppih;  // 1 / (2 zeta) of each primitive pair
  int chain, kmax;  // division of the kets' primitives over lanes (ket_split)
};

// Primitive quartets per step of the LDS-shape gradient kernel: 3 n_r lanes
// build the (root, axis) tables of one primitive quartet, as many primitive
// quartets at once as the lanes and 16 KB of tables allow (more would cost
// workgroups per CU).
template <int La, int Lb, int Lc, int Ld, int NT>
struct GradShape {
  static constexpr int NR = (La + Lb + Lc + Ld + 1) / 2 + 1;
  static constexpr int A1 = La + 2, B1 = Lb + 1, C1 = Lc + 2, D1 = Ld + 1;
  static constexpr int S = A1 * B1 * C1 * D1;
  static constexpr int HS = A1 * B1 * (Lc + 1 + Ld + 1);
  static constexpr int NPQ = [] {
    constexpr int by_lanes = NT / (3 * NR);
    constexpr int by_lds = int((16 * 1024) / (3 * NR * (S + HS) * sizeof(double)));
    constexpr int n = by_lanes < by_lds ? by_lanes : by_lds;
    return n < 1 ? 1 : n;
  }();
};

template <int La, int Lb, int Lc, int Ld, int NT>
__global__ __launch_bounds__(NT) void grad_kernel(GradArgs g) {
  using Sh = GradShape<La, Lb, Lc, Ld, NT>;
  constexpr int NR = Sh::NR, NPQ = Sh::NPQ;
  constexpr int B1 = Sh::B1, C1 = Sh::C1, D1 = Sh::D1;
  constexpr int S = Sh::S, HS = Sh::HS;
  constexpr int na = ncart(La), nb = ncart(Lb), nc = ncart(Lc), nd = ncart(Ld);
  constexpr int NOUT = na * nb * nc * nd;
  constexpr int SA = B1 * C1 * D1, SB = C1 * D1, SC = D1;
  __shared__ double tab[NPQ * NR * 3 * S];
  __shared__ double hs[NPQ * NR * 3 * HS];
  __shared__ double W[NOUT];
  __shared__ double ex2[NPQ][2];        // 2 alpha_a, 2 alpha_c of each primitive quartet
  __shared__ double kpq[NPQ * NR * 3];  // -2 rho u (P-Q) of each (primitive quartet, root, axis)
  __shared__ double sze[NPQ * NR][2];   // (rho/zeta) u, (rho/eta) u
  __shared__ int cbase[NOUT], cexpo[NOUT];
  __shared__ double nrm[NOUT];  // normalisation of each component, computed once
  __shared__ double red[NT / 64][9];
  extern __shared__ double gacc[];
  const int tid = threadIdx.x;
  const bool glds = g.glds != 0;
  if (glds)
    for (int e = tid; e < 3 * g.n_atoms; e += NT) gacc[e] = 0.0;

  // per component: table offsets (8 bits per axis) and exponents
  for (int o = tid; o < NOUT; o += NT) {
    const int d = o % nd, c = (o / nd) % nc, b = (o / (nd * nc)) % nb, a = o / (nd * nc * nb);
    int e = 0, bs = 0;
    for (int x = 0; x < 3; ++x) {
      const int ax = cart_comp(La, a, x), bx = cart_comp(Lb, b, x), cx = cart_comp(Lc, c, x),
                dx = cart_comp(Ld, d, x);
      bs |= (((ax * B1 + bx) * C1 + cx) * D1 + dx) << (8 * x);
      e |= (ax | (bx << 2) | (cx << 4) | (dx << 6)) << (8 * x);
    }
    cbase[o] = bs;
    cexpo[o] = e;
    nrm[o] = norm_corr(La, a) * norm_corr(Lb, b) * norm_corr(Lc, c) * norm_corr(Ld, d);
  }

  for (int ci = blockIdx.x; ci < g.nchunks; ci += gridDim.x) {
   const JkChunk ch = load_chunk_uniform(g.chunks, ci);
   const PairRec bra = load_pair_uniform(g.pairs, ch.bra);
   const JkSegs* sg = g.segs + ch.seg;
   // gridDim.y workgroups share a chunk (chunks of the register-shape J/K
   // classes hold up to 2048 quartets)
   const int len = ch.k1 - ch.k0;
   const int kb = ch.k0 + int((long long)len * blockIdx.y / gridDim.y);
   const int ke = ch.k0 + int((long long)len * (blockIdx.y + 1) / gridDim.y);
   for (int kq = kb; kq < ke; ++kq) {
    const int kp = chunk_ket(sg, kq);
    const PairRec ket = g.pairs[kp];
    if (quartet_select(g.sel, ch.bra, bra, kp, ket) == 0) continue;  // uniform over the workgroup
    const bool ij = bra.same, kl = ket.same, bk = (kp == ch.bra);
    const double deg = (ij ? 1.0 : 2.0) * (kl ? 1.0 : 2.0) * (bk ? 1.0 : 2.0);
    const size_t n = size_t(bra.mn);
    __syncthreads();  // W and the tables of the previous quartet are no longer read
    for (int o = tid; o < NOUT; o += NT) {
      const int d = o % nd, c = (o / nd) % nc, b = (o / (nd * nc)) % nb, a = o / (nd * nc * nb);
      const size_t mu = bra.fa + a, nu = bra.fb + b, la = ket.fa + c, si = ket.fb + d;
      const double* D = g.D + bra.moff;
      const double w = 0.5 * D[mu * n + nu] * D[la * n + si] -
                       0.125 * g.xscale * (D[mu * n + la] * D[nu * n + si] + D[mu * n + si] * D[nu * n + la]);
      W[o] = deg * w * nrm[o];
    }
    double gA[3] = {0, 0, 0}, gT[3] = {0, 0, 0}, gC[3] = {0, 0, 0};
    const int npp_b = bra.npp_sig, npp_k = ket.npp_sig;
    const int npt = npp_b * npp_k;
    for (int t0 = 0; t0 < npt; t0 += NPQ) {
      const int nq = min(NPQ, npt - t0);
      if (t0 > 0) __syncthreads();  // the previous step's tables are no longer read
      if (tid < 3 * NR * nq) {
        const int q = tid / (3 * NR), rr = tid - q * (3 * NR);
        const int r = rr / 3, ax = rr - 3 * r;
        const int t = t0 + q;
        const int ib = t / npp_k, ik = t - ib * npp_k;
        const PrimPair P = g.pp[bra.pp_off + ib];
        const PrimPair Q = g.pp[ket.pp_off + ik];
        const double zeta = P.zeta, eta = Q.zeta;
        const double izpe = 1.0 / (zeta + eta);
        const double rz = eta * izpe, re = zeta * izpe;
        const double PQx = P.Px - Q.Px, PQy = P.Py - Q.Py, PQz = P.Pz - Q.Pz;
        const double T = zeta * rz * (PQx * PQx + PQy * PQy + PQz * PQz);
        double ur, wr;
        rys_root_one<NR>(T, g.rys, r, ur, wr);
        const double h_z = 0.5 / zeta, h_e = 0.5 / eta;
        const double B00 = 0.5 * ur * izpe, B10 = h_z - h_z * rz * ur, B01 = h_e - h_e * re * ur;
        const double PQ = pick3(ax, PQx, PQy, PQz);
        const double PA = pick3(ax, P.PAx, P.PAy, P.PAz);
        const double QC = pick3(ax, Q.PAx, Q.PAy, Q.PAz);
        const double AB = pick3(ax, bra.ABx, bra.ABy, bra.ABz);
        const double CD = pick3(ax, ket.ABx, ket.ABy, ket.ABz);
        const double sc = ax == 2 ? P.Kc * Q.Kc * sqrt(izpe) * wr : 1.0;
        build_2d_lds<La + 1, Lb, Lc + 1, Ld, double>(tab + ((q * NR + r) * 3 + ax) * S,
                                                         hs + ((q * NR + r) * 3 + ax) * HS, PA - rz * ur * PQ,
                                                         QC + re * ur * PQ, AB, CD, B10, B01, B00, sc);
        kpq[(q * NR + r) * 3 + ax] = -2.0 * zeta * rz * ur * PQ;
        if (ax == 0) {
          sze[q * NR + r][0] = rz * ur;
          sze[q * NR + r][1] = re * ur;
        }
        if (rr == 0) {
          ex2[q][0] = 2.0 * g.ppab[bra.pp_off + ib].x;
          ex2[q][1] = 2.0 * g.ppab[ket.pp_off + ik].x;
        }
      }
      __syncthreads();
      // contraction: tasks (component o, primitive quartet q) over all lanes
      for (int tk = tid; tk < NOUT * nq; tk += NT) {
        const int q = tk / NOUT, o = tk - q * NOUT;
        const double w = W[o];
        const int bs = cbase[o], ee = cexpo[o];
        const double ta2 = ex2[q][0], tc2 = ex2[q][1];
        int i0[3], ea[3], eb[3], ec[3], ed[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          i0[x] = (bs >> (8 * x)) & 255;
          const int e = (ee >> (8 * x)) & 255;
          ea[x] = e & 3;
          eb[x] = (e >> 2) & 3;
          ec[x] = (e >> 4) & 3;
          ed[x] = (e >> 6) & 3;
        }
#pragma unroll 1
        for (int r = 0; r < NR; ++r) {
          const double* T3[3] = {tab + ((q * NR + r) * 3) * S, tab + ((q * NR + r) * 3 + 1) * S,
                                 tab + ((q * NR + r) * 3 + 2) * S};
          const double v0[3] = {T3[0][i0[0]], T3[1][i0[1]], T3[2][i0[2]]};
          const double sz = sze[q * NR + r][0], se = sze[q * NR + r][1];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const double* tx = T3[x];
            const double rest = w * v0[(x + 1) % 3] * v0[(x + 2) % 3];
            double dA = ta2 * tx[i0[x] + SA], dC = tc2 * tx[i0[x] + SC];
            double lo = 0.0, hi = 0.0;
            if (La > 0 && ea[x] > 0) {
              const double v = ea[x] * tx[i0[x] - SA];
              dA -= v;
              lo += v;
            }
            if (Lb > 0 && eb[x] > 0) lo += eb[x] * tx[i0[x] - SB];
            if (Lc > 0 && ec[x] > 0) {
              const double v = ec[x] * tx[i0[x] - SC];
              dC -= v;
              hi += v;
            }
            if (Ld > 0 && ed[x] > 0) hi += ed[x] * tx[i0[x] - 1];
            gA[x] += dA * rest;
            gT[x] += (kpq[(q * NR + r) * 3 + x] * v0[x] - sz * lo + se * hi) * rest;
            gC[x] += dC * rest;
          }
        }
      }
    }
    // workgroup reduction of the 9 components, then atomics per atom
    double v[9] = {gA[0], gA[1], gA[2], gT[0], gT[1], gT[2], gC[0], gC[1], gC[2]};
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      double x = v[k];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
      v[k] = x;
    }
    if ((tid & 63) == 0)
#pragma unroll
      for (int k = 0; k < 9; ++k) red[tid >> 6][k] = v[k];
    __syncthreads();
    if (tid < 9) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) s += red[w][tid];
      red[0][tid] = s;  // each lane owns its slot
    }
    __syncthreads();
    if (tid < 3) {
      const double a = red[0][tid], ab = red[0][3 + tid], c = red[0][6 + tid];
      double* out = glds ? gacc : g.grad;
      const int ia = 3 * g.shell_atom[bra.sa] + tid, ib = 3 * g.shell_atom[bra.sb] + tid;
      const int ic = 3 * g.shell_atom[ket.sa] + tid, id = 3 * g.shell_atom[ket.sb] + tid;
      if (glds) {
        lds_add(&out[ia], a);
        lds_add(&out[ib], ab - a);
        lds_add(&out[ic], c);
        lds_add(&out[id], -(ab + c));
      } else {
        atomic_add(&out[ia], a);
        atomic_add(&out[ib], ab - a);
        atomic_add(&out[ic], c);
        atomic_add(&out[id], -(ab + c));
      }
    }
   }
  }
  if (glds) {  // this workgroup's forces, once
    __syncthreads();
    for (int e = tid; e < 3 * g.n_atoms; e += NT) {
      const double v = gacc[e];
      if (v != 0.0) atomic_add(&g.grad[e], v);
    }
  }
}

// Execution of a gradient class.  Register shape where one bra component has at
// most 54 outputs (the weights W sit in registers): the bra is cut into NCH
// slices of at most 54 outputs, one workgroup each, every slice repeating roots
// and tables (forces are sums, nothing has to be merged).  Even at one
// wavefront per SIMD and several slices that beats the LDS shape, whose lanes
// wait for each other between tables and contraction: (ds|pp) of 32 waters in
// def2-SVP 20.7 ms in the LDS shape, 2.6 ms in this one.
template <int La, int Lb, int Lc, int Ld>
struct GradPolicy {
  static constexpr int na = ncart(La), rest = ncart(Lb) * ncart(Lc) * ncart(Ld);
  static constexpr int NOUT = na * rest;
  static constexpr int NT = NOUT <= 256 ? 64 : 128;  // lanes of the LDS shape
  static constexpr bool regs = rest <= 54;
  static constexpr int CHA1 = regs ? (54 / rest < na ? 54 / rest : na) : na;
  static constexpr int NCH = (na + CHA1 - 1) / CHA1;
  static constexpr int CHA = (na + NCH - 1) / NCH;
  // wavefronts per SIMD that bound the registers: what the compiler reaches
  // with at most 40 bytes of scratch.  (Two for 27 outputs and more cost
  // 500-800 bytes and were slower: (pp|ps) 8.6 -> 11.9 ms, (dp|ps) 4.0 -> 9.8.)
  static constexpr int WPE = CHA * rest <= 3 ? 3 : CHA * rest <= 18 ? 2 : 1;
};

// --------------------------------------------------------------------------
// Register shape: one lane per shell quartet (bra components A0 .. A1 - 1) of a
// bra-anchored chunk, the 2D tables raised by one on A or C held in registers
// (entries raised on both are never used, so the compiler drops them).
// f: the A, AB and C derivatives.  The forces on the bra atoms are summed over
// the lane's quartets and reduced over the wavefront; those on the ket atoms go
// to the workgroup's LDS force array (or to HBM atomics without one).
// --------------------------------------------------------------------------
// LB: the Rys tables of the rule from the workgroup's copy in LDS (lrows)
template <int La, int Lb, int Lc, int Ld, int A0, int A1, bool LB>
__device__ __forceinline__ void grad_quartet_regs(const GradArgs& g, const PairRec& bra, const PairRec& ket,
                                                  bool bk, int ik0, int per, double (&f)[9], lds_cdptr lrows) {
  constexpr int NR = (La + Lb + Lc + Ld + 1) / 2 + 1;
  constexpr int NA = A1 - A0, nb = ncart(Lb), nc = ncart(Lc), nd = ncart(Ld);
  const size_t n = size_t(bra.mn);
  const bool ij = bra.sa == bra.sb, kl = ket.sa == ket.sb;
  const double deg = (ij ? 1.0 : 2.0) * (kl ? 1.0 : 2.0) * (bk ? 1.0 : 2.0);
  const double* __restrict__ D = g.D + bra.moff;
  double W[NA][nb][nc][nd];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < nb; ++b)
#pragma unroll
      for (int c = 0; c < nc; ++c)
#pragma unroll
        for (int d = 0; d < nd; ++d) {
          const size_t mu = bra.fa + A0 + a, nu = bra.fb + b, la = ket.fa + c, si = ket.fb + d;
          const double w = 0.5 * D[mu * n + nu] * D[la * n + si] -
                           0.125 * g.xscale * (D[mu * n + la] * D[nu * n + si] + D[mu * n + si] * D[nu * n + la]);
          W[a][b][c][d] = deg * w * norm_corr(La, A0 + a) * norm_corr(Lb, b) * norm_corr(Lc, c) * norm_corr(Ld, d);
        }
#pragma unroll
  for (int x = 0; x < 9; ++x) f[x] = 0.0;
  const double ABx = bra.ABx, ABy = bra.ABy, ABz = bra.ABz;
  const double CDx = ket.ABx, CDy = ket.ABy, CDz = ket.ABz;
  const int ik1 = min(ket.npp_sig, ik0 + per);
  for (int ik = ik0; ik < ik1; ++ik) {
    const PrimPair Q = g.pp[ket.pp_off + ik];
    const double2 ek = g.ppab[ket.pp_off + ik];
    const double eta = Q.zeta, h_e = g.ppih[ket.pp_off + ik];
    const double tc2 = 2.0 * ek.x;
    for (int ib = 0; ib < bra.npp_sig; ++ib) {
      // the bra is uniform over the workgroup: scalar loads
      const PrimPair P = load_prim(g.pp, bra.pp_off + ib);
      const double ta2 = 2.0 * as_const(reinterpret_cast<const double*>(g.ppab))[2 * (bra.pp_off + ib)];
      const double zeta = P.zeta, h_z = as_const(g.ppih)[bra.pp_off + ib];
      const double x = zeta + eta;
      double y = __builtin_amdgcn_rsq(x);
      y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
      y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
      const double izpe = y * y;
      const double rz = eta * izpe, re = zeta * izpe;
      const double PQx = P.Px - Q.Px, PQy = P.Py - Q.Py, PQz = P.Pz - Q.Pz;
      const double rho = zeta * rz;
      const double T = rho * (PQx * PQx + PQy * PQy + PQz * PQz);
      const double pref = P.Kc * Q.Kc * y;
      if constexpr (La + Lb + Lc + Ld <= 1) {
        // (ss|ss) and (ps|ss): their derivatives are closed forms in F_0..F_2,
        // S_m = pref F_m (two roots and their tables instead took (ps|ss) of 32
        // waters in def2-SVP 9.5 ms).  With V_m = (p.PA) S_m - (rho/zeta)
        // (p.PQ) S_{m+1} the weighted sum over the components p (V_m = W S_m
        // for (ss|ss)):
        //   A:  2 a [PA V_0 - (rho/zeta) PQ V_1 + p (S_0 - (rho/zeta) S_1)/(2 zeta)] - p S_0
        //   AB: -2 rho PQ V_1 - (rho/zeta) S_1 p
        //   C:  2 c [QC V_0 + (rho/eta) PQ V_1 + p S_1 / (2 (zeta + eta))]
        const double pa[3] = {P.PAx, P.PAy, P.PAz}, qc[3] = {Q.PAx, Q.PAy, Q.PAz}, pq[3] = {PQx, PQy, PQz};
        double V0, V1, sA = 0.0, sT = 0.0, sC = 0.0, p[3] = {0, 0, 0};
        if constexpr (La == 0) {
          double F0, F1;
          if constexpr (LB)
            boys01_at(T, lrows, F0, F1);
          else
            boys01_at(T, g.rys + LAI_B8_OFF, F0, F1);
          const double wp = W[0][0][0][0] * pref;
          V0 = wp * F0;
          V1 = wp * F1;
        } else {
          double F0, F1, F2;
          if constexpr (LB)
            boys012_at(T, lrows, F0, F1, F2);
          else
            boys012_at(T, g.rys + LAI_B10_OFF, F0, F1, F2);
          const double S0 = pref * F0, S1 = pref * F1, S2 = pref * F2;
#pragma unroll
          for (int m = 0; m < 3; ++m) p[m] = W[m < NA ? m : 0][0][0][0];
          const double dpa = p[0] * pa[0] + p[1] * pa[1] + p[2] * pa[2];
          const double dpq = -rz * (p[0] * pq[0] + p[1] * pq[1] + p[2] * pq[2]);
          V0 = dpa * S0 + dpq * S1;
          V1 = dpa * S1 + dpq * S2;
          sA = ta2 * h_z * (S0 - rz * S1) - S0;
          sT = -rz * S1;
          sC = tc2 * 0.5 * izpe * S1;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          f[m] += ta2 * (pa[m] * V0 - rz * pq[m] * V1) + p[m] * sA;
          f[3 + m] += -2.0 * rho * pq[m] * V1 + p[m] * sT;
          f[6 + m] += tc2 * (qc[m] * V0 + re * pq[m] * V1) + p[m] * sC;
        }
        continue;
      }
      double u[NR], w[NR];
      if constexpr (!LB)
        rys_roots<NR>(T, g.rys, u, w);
      else if constexpr (NR <= 2)
        rys_roots12<NR>(T, lrows, u, w);
      else
        rys_cheb<NR>(T, lrows, kChebStrideLds<NR>, u, w);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const double ur = u[r];
        const double B00 = 0.5 * ur * izpe, B10 = h_z - h_z * rz * ur, B01 = h_e - h_e * re * ur;
        const double sz = rz * ur, se = re * ur, k0 = -2.0 * rho * ur;
        double Ix[La + 2][Lb + 1][Lc + 2][Ld + 1], Iy[La + 2][Lb + 1][Lc + 2][Ld + 1],
            Iz[La + 2][Lb + 1][Lc + 2][Ld + 1];
        build_2d<La + 1, Lb, Lc + 1, Ld, double>(Ix, P.PAx - sz * PQx, Q.PAx + se * PQx, ABx, CDx, B10, B01, B00,
                                                 1.0);
        build_2d<La + 1, Lb, Lc + 1, Ld, double>(Iy, P.PAy - sz * PQy, Q.PAy + se * PQy, ABy, CDy, B10, B01, B00,
                                                 1.0);
        build_2d<La + 1, Lb, Lc + 1, Ld, double>(Iz, P.PAz - sz * PQz, Q.PAz + se * PQz, ABz, CDz, B10, B01, B00,
                                                 pref * w[r]);
        // the A, AB and C derivatives of one 2D integral (exponents i, j, k, l)
        auto deriv = [&](const double (&I)[La + 2][Lb + 1][Lc + 2][Ld + 1], int i, int j, int k, int l, double kd,
                         double& dA, double& dT, double& dC) {
          const double va = i ? double(i) * I[i ? i - 1 : 0][j][k][l] : 0.0;
          const double vb = j ? double(j) * I[i][j ? j - 1 : 0][k][l] : 0.0;
          const double vc = k ? double(k) * I[i][j][k ? k - 1 : 0][l] : 0.0;
          const double vd = l ? double(l) * I[i][j][k][l ? l - 1 : 0] : 0.0;
          dA = ta2 * I[i + 1][j][k][l] - va;
          dC = tc2 * I[i][j][k + 1][l] - vc;
          dT = kd * I[i][j][k][l];
          if (i || j) dT -= sz * (va + vb);
          if (k || l) dT += se * (vc + vd);
        };
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
          for (int b = 0; b < nb; ++b)
#pragma unroll
            for (int c = 0; c < nc; ++c)
#pragma unroll
              for (int d = 0; d < nd; ++d) {
                const int ax = cart_comp(La, A0 + a, 0), ay = cart_comp(La, A0 + a, 1), az = cart_comp(La, A0 + a, 2);
                const int bx = cart_comp(Lb, b, 0), by = cart_comp(Lb, b, 1), bz = cart_comp(Lb, b, 2);
                const int cx = cart_comp(Lc, c, 0), cy = cart_comp(Lc, c, 1), cz = cart_comp(Lc, c, 2);
                const int dx = cart_comp(Ld, d, 0), dy = cart_comp(Ld, d, 1), dz = cart_comp(Ld, d, 2);
                const double wt = W[a][b][c][d];
                const double x0 = Ix[ax][bx][cx][dx], y0 = Iy[ay][by][cy][dy], z0 = Iz[az][bz][cz][dz];
                double dA[3], dT[3], dC[3];
                deriv(Ix, ax, bx, cx, dx, k0 * PQx, dA[0], dT[0], dC[0]);
                deriv(Iy, ay, by, cy, dy, k0 * PQy, dA[1], dT[1], dC[1]);
                deriv(Iz, az, bz, cz, dz, k0 * PQz, dA[2], dT[2], dC[2]);
                const double rest[3] = {wt * y0 * z0, wt * x0 * z0, wt * x0 * y0};
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                  f[m] += dA[m] * rest[m];
                  f[3 + m] += dT[m] * rest[m];
                  f[6 + m] += dC[m] * rest[m];
                }
              }
      }
    }
  }
}

template <int La, int Lb, int Lc, int Ld, int A0, int A1, bool LB>
__device__ __forceinline__ void grad_chunks_regs(const GradArgs& g, double* gacc, SortLds<false>& srt,
                                                 lds_cdptr lrows) {
  const int tid = threadIdx.x;
  const bool glds = g.glds != 0;
  if (glds) {
    for (int e = tid; e < 3 * g.n_atoms; e += blockDim.x) gacc[e] = 0.0;
    __syncthreads();
  }
  auto add = [&](int i, double v) {
    if (glds)
      lds_add(&gacc[i], v);
    else
      atomic_add(&g.grad[i], v);
  };
  for (int ci = blockIdx.x; ci < g.nchunks; ci += gridDim.x) {
    const JkChunk ch = load_chunk_uniform(g.chunks, ci);
    const PairRec bra = load_pair_uniform(g.pairs, ch.bra);
    const int iA = 3 * g.shell_atom[bra.sa], iB = 3 * g.shell_atom[bra.sb];
    double fab[6] = {0, 0, 0, 0, 0, 0};
    const JkSegs* sg = g.segs + ch.seg;
    const KetSplit sp = ket_split_uniform(g.chain, g.kmax, bra.npp_sig);
    for (int s0 = ch.k0; s0 < ch.k1; s0 += sp.run) {
    const int nsel = sort_run<256>(sg, g.pairs, g.sel, ch.bra, bra, sp, s0, min(ch.k1, s0 + sp.run), srt, 256);
    for (int r = 0; 256 * r < nsel; ++r) {
      const int i = sorted_block(tid, r, 4) + (tid & 63);
      if (i >= nsel) continue;
      const unsigned ent = srt.e[i];
      const int kp = chunk_ket(sg, s0 + entry_pos(ent));
      const PairRec ket = g.pairs[kp];
      double f[9];
      grad_quartet_regs<La, Lb, Lc, Ld, A0, A1, LB>(g, bra, ket, kp == ch.bra, entry_part(ent) * sp.per, sp.per, f,
                                                    lrows);
#pragma unroll
      for (int x = 0; x < 6; ++x) fab[x] += f[x];
      const int iC = 3 * g.shell_atom[ket.sa], iD = 3 * g.shell_atom[ket.sb];
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        add(iC + x, f[6 + x]);
        add(iD + x, -(f[3 + x] + f[6 + x]));  // translational invariance
      }
    }
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double fA = wave_sum(fab[x]), fB = wave_sum(fab[3 + x] - fab[x]);
      if ((tid & 63) == 0) {
        if (fA != 0.0) add(iA + x, fA);
        if (fB != 0.0) add(iB + x, fB);
      }
    }
  }
  if (glds) {  // this workgroup's forces, once
    __syncthreads();
    for (int e = tid; e < 3 * g.n_atoms; e += blockDim.x) {
      const double v = gacc[e];
      if (v != 0.0) atomic_add(&g.grad[e], v);
    }
  }
}

template <int La, int Lb, int Lc, int Ld, int CHA, int C, bool LB>
__device__ __forceinline__ void dispatch_grad(const GradArgs& g, int slice, double* gacc, SortLds<false>& srt,
                                              lds_cdptr lrows) {
  constexpr int na = ncart(La), A0 = C * CHA, A1 = A0 + CHA < na ? A0 + CHA : na;
  if (slice == C) {
    grad_chunks_regs<La, Lb, Lc, Ld, A0, A1, LB>(g, gacc, srt, lrows);
  } else if constexpr (A1 < na) {
    dispatch_grad<La, Lb, Lc, Ld, CHA, C + 1, LB>(g, slice, gacc, srt, lrows);
  }
}

// Dynamic LDS: the Rys tables of the class (kGradTable doubles), then the
// workgroup's forces.  Tables in LDS for one and three roots (23 and 34 KB) and
// for two (63 KB) where the registers leave two workgroups per CU anyway:
// (pp|ps) 8.3 -> 7.5 ms, (ds|ps) 4.6 -> 3.8, (ss|ss) 4.1 -> 3.6; four roots
// (51 KB, one workgroup per CU) did not gain: (dp|pp) 5.2 -> 5.3, (dp|dp) 3.9 ->
// 4.3.
template <int La, int Lb, int Lc, int Ld>
constexpr int grad_table() {
  constexpr int NR = (La + Lb + Lc + Ld + 1) / 2 + 1;
  return NR == 1 || NR == 3 || (NR == 2 && GradPolicy<La, Lb, Lc, Ld>::WPE <= 2) ? lds_rys_doubles(NR) : 0;
}
template <int La, int Lb, int Lc, int Ld>
inline constexpr int kGradTable = grad_table<La, Lb, Lc, Ld>();

template <int La, int Lb, int Lc, int Ld>
__global__ __launch_bounds__(256, (GradPolicy<La, Lb, Lc, Ld>::WPE)) void grad_kernel_regs(GradArgs g) {
  extern __shared__ double dyn[];
  __shared__ SortLds<false> srt;  // lane schedule of the chunk (sort_run)
  constexpr int NB = kGradTable<La, Lb, Lc, Ld>;
  if constexpr (NB > 0) copy_rys_lds<(La + Lb + Lc + Ld + 1) / 2 + 1>(g.rys, dyn);
  dispatch_grad<La, Lb, Lc, Ld, GradPolicy<La, Lb, Lc, Ld>::CHA, 0, (NB > 0)>(g, blockIdx.y, dyn + NB, srt,
                                                                              (lds_cdptr)(dyn));
}

}  // namespace lai
