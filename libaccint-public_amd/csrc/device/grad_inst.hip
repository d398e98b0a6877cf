// grad_inst.hip -- instantiates the gradient kernels for the classes with
// every shell at most d (quartet classes 0..20).  Compiled LAI_NPARTS times
// with -DLAI_PART=k like eri_inst.hip.
#include "grad_kernels.hpp"
#include "launch.hpp"

#ifndef LAI_PART
#error "compile with -DLAI_PART=<k> -DLAI_NPARTS=<n>"
#endif

namespace lai {
namespace {

// per-workgroup force accumulators in LDS up to this many atoms
constexpr int kGradLdsAtoms = 2048;

template <int ID>
void launch_grad(const GradArgs& a0, hipStream_t s, int max_blocks) {
  constexpr int pb = cls_bra(ID), pk = cls_ket(ID);
  constexpr int La = pc_La(pb), Lb = pc_Lb(pb), Lc = pc_La(pk), Ld = pc_Lb(pk);
  using P = GradPolicy<La, Lb, Lc, Ld>;
  if (a0.nchunks <= 0) return;
  GradArgs a = a0;
  a.glds = a.n_atoms <= kGradLdsAtoms ? 1 : 0;
  const size_t dyn = a.glds ? size_t(3) * a.n_atoms * sizeof(double) : 0;
  if constexpr (P::regs) {
    const int blocks = a.nchunks < max_blocks ? a.nchunks : max_blocks;
    auto kern = grad_kernel_regs<La, Lb, Lc, Ld>;
    constexpr size_t tab = size_t(kGradTable<La, Lb, Lc, Ld>) * sizeof(double);
    // up to 63 KB of tables and 48 KB of forces: above the 64 KB default
    static const bool raised =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            int(tab + 3 * kGradLdsAtoms * sizeof(double))) == hipSuccess;
    if (!raised && tab + dyn > 64 * 1024) {  // forces to HBM
      a.glds = 0;
      hipLaunchKernelGGL(kern, dim3(blocks, P::NCH), dim3(256), tab, s, a);
      return;
    }
    hipLaunchKernelGGL(kern, dim3(blocks, P::NCH), dim3(256), tab + dyn, s, a);
  } else {
    // the worklist chunks follow the J/K kernel shape of the class: long ones
    // for its register shape are split over gridDim.y workgroups
    constexpr int split = ClassPolicy<La, Lb, Lc, Ld>::regs ? 64 : 1;
    const int blocks = a.nchunks < max_blocks ? a.nchunks : max_blocks;
    hipLaunchKernelGGL((grad_kernel<La, Lb, Lc, Ld, P::NT>), dim3(blocks, split), dim3(P::NT), dyn, s, a);
  }
}

template <int ID>
void fill(GradLauncher* f) {
  if constexpr (ID % LAI_NPARTS == LAI_PART) f[ID] = &launch_grad<ID>;
  if constexpr (ID + 1 < kNumGradClasses) fill<ID + 1>(f);
}

}  // namespace

#define LAI_CAT2(a, b) a##b
#define LAI_CAT(a, b) LAI_CAT2(a, b)
void LAI_CAT(fill_grad_launchers_part_, LAI_PART)(GradLauncher* f) { fill<0>(f); }

}  // namespace lai
