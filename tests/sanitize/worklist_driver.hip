// worklist_driver.hip -- the worklist code of csrc/device/api.hip on the host
// alone: compiled without device code, with stand-ins for the HIP runtime
// (memory from the heap, allocations that can be made to fail) and for the
// class kernels (each launch looks at what it was given).
//   worklist_driver alloc  every allocation of a rebuild and of a tuning fails
//                          in turn; nothing may run on parts of two lists
//   worklist_driver cut    the chunks of divided kets against their definition
//   worklist_driver flops  the gradient's work model on classes counted by hand
#include "../../libaccint-public_amd/csrc/device/api.hip"

#include <cstdio>
#include <cstdlib>
#include <map>

// ---- HIP runtime ------------------------------------------------------------
static std::map<const char*, size_t> g_live;  // allocations and their sizes
static int g_fail_at = -1;                    // the allocation that fails, counted down
static long g_launches = 0;
static bool g_bad = false;

static void complain(const char* what) {
  std::printf("%s\n", what);
  g_bad = true;
}
template <typename T>
static void want(const T* p, size_t n, const char* what) {
  const char* c = reinterpret_cast<const char*>(p);
  auto it = g_live.upper_bound(c);
  if (it == g_live.begin() || (--it, c + n * sizeof(T) > it->first + it->second)) complain(what);
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (g_fail_at >= 0 && g_fail_at-- == 0) {
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  *p = std::malloc(n);
  g_live[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (p && !g_live.erase(static_cast<char*>(p))) complain("free of what was not allocated");
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  return p->multiProcessorCount = 256, hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 1.f, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(1), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = reinterpret_cast<hipGraph_t>(1), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return *x = reinterpret_cast<hipGraphExec_t>(1), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
static long g_graph_launches = 0;
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return ++g_graph_launches, hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) {
  static void* h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}

// ---- kernels ------------------------------------------------------------------
namespace lai {
__global__ void onee_kernel(OneEArgs) {}
__global__ void fill_zero_kernel(double*, size_t) {}
__global__ void finish_jk_kernel(FinishArgs, int) {}
__global__ void rys_probe_kernel(int, int, const double*, const double*, double*, double*) {}
__global__ void boys_probe_kernel(int, int, const double*, double*) {}
__global__ void gather_pairs_kernel(const PairRec*, const int*, int, PairRec*) {}
__global__ void schwarz_reduce_kernel(const double*, const long long*, const int*, const int*, double*, int) {}
__global__ void worklist_stats_kernel(WlStatsArgs a) {}

static lai_basis* g_basis = nullptr;

// what a class kernel reads is allocated and of the list it was built with
static void look(int nchunks, const JkChunk* ch, const JkSegs* segs, const PairRec* pairs, const QuartetSel& sel) {
  ++g_launches;
  const size_t np = g_basis->pairs_h.size();
  want(ch, size_t(nchunks), "chunks not allocated");
  want(segs, g_basis->segs_h.size(), "segments not allocated");
  want(pairs, np, "pair records not allocated");
  want(sel.Qpair, np, "bounds not allocated");
  if (g_bad) return;
  for (int k = 0; k < nchunks; ++k) {
    if (ch[k].bra < 0 || size_t(ch[k].bra) >= np || ch[k].seg < 0 || size_t(ch[k].seg) >= g_basis->segs_h.size())
      return complain("chunk out of the list");
    const JkSegs& s = segs[ch[k].seg];
    if (ch[k].k0 < 0 || ch[k].k1 > s.cum[s.n] || ch[k].k0 >= ch[k].k1) return complain("chunk out of its run");
  }
}
template <int ID>
static void run_class(const EriArgs& a, hipStream_t, const LaunchTune&) {
  if (a.mode == 0) look(a.nchunks, a.chunks, a.segs, a.pairs, a.sel);
}
static void run_grad(const GradArgs& a, hipStream_t, int) { look(a.nchunks, a.chunks, a.segs, a.pairs, a.sel); }

template <int ID>
static void fill(ClassLauncher* f64, ClassLauncher* f32, ClassInfo* info) {
  constexpr int pb = cls_bra(ID), pk = cls_ket(ID);
  using P = ClassPolicy<pc_La(pb), pc_Lb(pb), pc_La(pk), pc_Lb(pk)>;
  f64[ID] = f32[ID] = &run_class<ID>;
  info[ID].nt = P::regs ? (P::NCH > 1 ? 64 * P::NCH : 256) : (P::waves ? 64 * P::NW : P::NT);
  info[ID].shape = P::shape;
  info[ID].alt = P::alt;
  info[ID].alt2 = P::alt2;
  if constexpr (ID + 1 < kNumClasses) fill<ID + 1>(f64, f32, info);
}
void fill_launchers_part_0(ClassLauncher* f64, ClassLauncher* f32, ClassInfo* info) { fill<0>(f64, f32, info); }
void fill_launchers_part_1(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_2(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_3(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_4(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_5(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_6(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_launchers_part_7(ClassLauncher*, ClassLauncher*, ClassInfo*) {}
void fill_grad_launchers_part_0(GradLauncher* f) {
  for (int c = 0; c < kNumGradClasses; ++c) f[c] = &run_grad;
}
void fill_grad_launchers_part_1(GradLauncher*) {}
void fill_grad_launchers_part_2(GradLauncher*) {}
void fill_grad_launchers_part_3(GradLauncher*) {}
bool persist_covers(int) { return false; }
int launch_persistent(const EriArgs&, const PersistItem*, int, int*, hipStream_t, int) { return 0; }
}  // namespace lai

// ---- a basis -------------------------------------------------------------------
static lai_basis* make_basis(lai_ctx* ctx, int n_atoms, int seed) {
  std::vector<int> L, nprim;
  std::vector<double> xyz, ex, co;
  unsigned s = unsigned(seed) * 2654435761u + 1u;
  auto rnd = [&]() { return double((s = s * 1664525u + 1013904223u) >> 8) / double(1 << 24); };
  for (int a = 0; a < n_atoms; ++a) {
    const double at[3] = {6.0 * rnd(), 6.0 * rnd(), 6.0 * rnd()};
    const int prims[5] = {8, 3, 3, 1, 1}, ls[5] = {0, 0, 1, 1, 2};
    for (int k = 0; k < 5; ++k) {
      L.push_back(ls[k]);
      nprim.push_back(prims[k]);
      xyz.insert(xyz.end(), at, at + 3);
      for (int p = 0; p < prims[k]; ++p) {
        ex.push_back(0.2 * std::pow(3.0, p));
        co.push_back(0.3 + 0.5 * rnd());
      }
    }
  }
  lai_basis* b = nullptr;
  const int ns = int(L.size());
  if (lai_dev_upload_basis(ctx, ns, L.data(), xyz.data(), nprim.data(), ex.data(), co.data(), &b) != LAI_OK)
    std::printf("upload: %s\n", lai_dev_last_error()), std::exit(2);
  std::vector<double> Q(size_t(ns) * (ns + 1) / 2);
  for (auto& q : Q) q = std::pow(10.0, -9.0 * rnd());
  std::vector<int> atom(ns);
  for (int k = 0; k < ns; ++k) atom[k] = k / 5;
  if (lai_dev_set_schwarz(b, Q.data()) != LAI_OK || lai_dev_set_shell_atoms(b, atom.data(), n_atoms) != LAI_OK)
    std::printf("set-up: %s\n", lai_dev_last_error()), std::exit(2);
  g_basis = b;
  return b;
}

static int build(lai_basis* b, double thr) {
  int64_t n, n32;
  uint64_t cs;
  const int rc = lai_dev_build_worklist(b, thr, nullptr, 0, 0.0, &n, &n32, &cs);
  // (the statistics are a kernel's; here every class with chunks has quartets)
  if (rc == LAI_OK)
    for (int c = 0; c < kNumClasses; ++c) b->counts[c] = int64_t(class_quartets(b, c));
  return rc;
}

// Everything that runs the list; returns how many of the calls were refused.
static int run_all(lai_basis* b) {
  double* m = nullptr;
  (void)hipMalloc(reinterpret_cast<void**>(&m), size_t(b->nbf) * b->nbf * 8);
  void* st = reinterpret_cast<void*>(1);
  int refused = 0;
  refused += lai_dev_jk(b, m, m, m, 0, st) == LAI_ERR_INVALID_STATE;
  refused += lai_dev_jk_grad(b, m, 1.0, m, b->n_atoms, st) == LAI_ERR_INVALID_STATE;
  refused += lai_dev_jk_graph_launch(b, st) == LAI_ERR_INVALID_STATE;
  refused += lai_dev_worklist_stats(b, nullptr, nullptr, nullptr, nullptr) == LAI_ERR_INVALID_STATE;
  (void)hipFree(m);
  return refused;
}

static int alloc_test(lai_ctx* ctx) {
  lai_basis* b = make_basis(ctx, 4, 1);
  double* m = nullptr;
  (void)hipMalloc(reinterpret_cast<void**>(&m), size_t(b->nbf) * b->nbf * 8);
  auto whole = [&](double thr) {
    if (build(b, thr) != LAI_OK) complain("a build without failures failed");
    if (lai_dev_jk_graph_capture(b, m, m, m, 0, reinterpret_cast<void*>(1)) != LAI_OK) complain("capture failed");
    if (run_all(b) != 0) complain("a whole list was refused");
  };
  int n = 0;
  for (;; ++n) {  // allocation n of a rebuild fails
    whole(1e-12);
    const long before = g_launches, graphs = g_graph_launches;
    g_fail_at = n;
    const int rc = build(b, 1e-4);
    const bool hit = g_fail_at < 0;
    g_fail_at = -1;
    if (!hit) break;
    if (rc != LAI_ERR_MEMORY) complain("a failed allocation was not reported");
    if (run_all(b) != 4) complain("a list in parts was not refused");
    if (g_launches != before || g_graph_launches != graphs) complain("a list in parts was run");
    if (g_bad) return std::printf("rebuild, allocation %d\n", n), 1;
  }
  std::printf("%d allocations of a rebuild\n", n);
  for (n = 0;; ++n) {  // allocation n of a tuning fails
    whole(1e-12);
    std::vector<lai_class_tune> t(kNumClasses);
    for (int c = 0; c < kNumClasses; ++c) t[c] = lai_class_tune{c, launchers().info[c].shape, 7, 0, 0.0, 0.0};
    g_fail_at = n;
    const int rc = lai_dev_set_tuning(b, t.data(), kNumClasses);
    const bool hit = g_fail_at < 0;
    g_fail_at = -1;
    if (!hit) break;
    if (rc != LAI_ERR_MEMORY) complain("a failed allocation was not reported");
    if (run_all(b) != 4) complain("a list in parts was not refused");
    if (g_bad) return std::printf("tuning, allocation %d\n", n), 1;
    if (lai_dev_set_tuning(b, nullptr, 0) != LAI_OK) complain("the defaults were refused");
  }
  std::printf("%d allocations of a tuning, %ld launches\n", n, g_launches);
  (void)hipFree(m);
  lai_dev_basis_free(b);
  return g_bad;
}

// The chunks of a run by their definition: entry by entry, a chunk ends at the
// first position that has its share of all entries before it.
static std::vector<JkChunk> cut_plainly(const lai_basis* b, const JkChunk& r, int kmax, int cmax, int chain) {
  const JkSegs& sg = b->segs_h[r.seg];
  const KetSplit sp = ket_split(chain, kmax, int(b->lcum[r.bra + 1] - b->lcum[r.bra]));
  std::vector<double> before(1, 0.0);
  double done = 0.0;
  for (int s = 0; s < sg.n; ++s) {
    const long long* l = &b->lcum[sg.start[s]];
    const int len = sg.cum[s + 1] - sg.cum[s];
    for (int m = 1; m <= len; ++m) before.push_back(done + (m + double(l[m] - l[0]) / sp.per));
    done = before.back();
  }
  std::vector<JkChunk> C;
  const int pieces = std::min(r.k1, int(done / cmax) + 1);
  int k0 = 0;
  for (int q = 1; q <= pieces && k0 < r.k1; ++q) {
    int k = k0 + 1;
    while (k < r.k1 && (q == pieces || before[k] < done * q / pieces)) ++k;
    C.push_back(JkChunk{r.bra, r.seg, k0, k});
    k0 = k;
  }
  return C;
}

static int cut_test(lai_ctx* ctx) {
  long divided = 0, several = 0;
  for (int atoms : {1, 2, 5}) {
    lai_basis* b = make_basis(ctx, atoms, atoms);
    if (build(b, 1e-12) != LAI_OK) complain("a build without failures failed");
    for (int c = 0; c < kNumClasses; ++c) {
      const ClassList& C = b->cls[c];
      for (int chain : {C.chain, 1, 16, 100})
        for (int cmax : {1, 3, 64, 256, 2048}) {
          const std::vector<JkChunk> got = cut_runs(b, C, cmax, chain);
          size_t at = 0;
          for (const JkChunk& r : C.runs) {
            const KetSplit sp = ket_split(chain, C.kmax, int(b->lcum[r.bra + 1] - b->lcum[r.bra]));
            int k = 0;
            const size_t first = at;
            for (; at < got.size() && k < r.k1; ++at) {
              const JkChunk& x = got[at];
              if (x.bra != r.bra || x.seg != r.seg || x.k0 != k || x.k1 <= x.k0 || x.k1 > r.k1)
                complain("the chunks of a run are not its parts in order");
              k = x.k1;
            }
            if (k != r.k1) complain("a run is not covered");
            if (sp.per >= C.kmax) continue;
            ++divided;
            const std::vector<JkChunk> want = cut_plainly(b, r, C.kmax, cmax, chain);
            several += want.size() > 1;
            bool same = want.size() == at - first;
            for (size_t i = 0; same && i < want.size(); ++i)
              same = want[i].k0 == got[first + i].k0 && want[i].k1 == got[first + i].k1;
            if (!same) complain("a divided run is cut elsewhere");
            if (g_bad) return std::printf("%d atoms, class %d, chain %d, cap %d\n", atoms, c, chain, cmax), 1;
          }
          if (at != got.size()) complain("chunks beyond the runs");
        }
    }
    lai_dev_basis_free(b);
  }
  std::printf("%ld divided runs, %ld of several chunks\n", divided, several);
  return g_bad || several == 0;
}

// (dp|ps): three roots; tables of x^3 on d, p, p^2 on the ket: 10 recursion
// operations along the bra, 13 + 23 along the ket, 24 of transfer to b, so 70;
// 54 components: 30 + 3 (50 + 3 70 + 12 54).  In every order of the quartet.
static int flops_test() {
  const int q[3][4] = {{2, 1, 1, 0}, {0, 0, 0, 0}, {1, 0, 0, 0}};
  const double want[3] = {2754.0, 104.0, 168.0};
  for (int t = 0; t < 3; ++t)
    for (int o = 0; o < 8; ++o) {
      int l[4] = {q[t][0], q[t][1], q[t][2], q[t][3]};
      if (o & 1) std::swap(l[0], l[1]);
      if (o & 2) std::swap(l[2], l[3]);
      if (o & 4) std::swap(l[0], l[2]), std::swap(l[1], l[3]);
      const double got = fgrad(1, l[0], l[1], l[2], l[3]);
      if (got != want[t])
        std::printf("(%d %d|%d %d): %g instead of %g\n", l[0], l[1], l[2], l[3], got, want[t]), g_bad = true;
    }
  return g_bad;
}

int main(int argc, char** argv) {
  lai_ctx* ctx = nullptr;
  if (lai_dev_init(0, &ctx) != LAI_OK) return std::printf("init: %s\n", lai_dev_last_error()), 2;
  const std::string what = argc > 1 ? argv[1] : "alloc";
  int rc = 2;
  if (what == "alloc") rc = alloc_test(ctx);
  if (what == "cut") rc = cut_test(ctx);
  if (what == "flops") rc = flops_test();
  if (rc == 0) std::printf("worklist driver ok\n");
  return rc;
}
