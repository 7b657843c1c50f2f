// The host side of the solver (cup3d_amd/csrc/solver.cpp, as it is) over a
// stand-in HIP runtime: device memory is host memory full of garbage, every
// allocation is counted and any one of them can be made to fail, and the kernel
// launches that a test looks at check their arguments instead. Calls that no
// test reaches stay unresolved. One scenario a run, named by argv[1]; exit
// status 0 when it holds.
#include "../../cup3d_amd/csrc/solver.cpp"

#include <cstdio>
#include <cstdlib>
#include <set>

namespace {

int g_allocs = 0;        // device and pinned allocations so far
int g_pinned = 0;        // pinned ones
int g_fail_at = -1;      // number of the allocation that fails (-1: none)
std::set<void*> g_live;  // what is allocated
bool g_reject = false;   // the next topology build finds a duplicate block
double g_inv_vol = 0.0;  // of the last mean removal
int g_short_k1 = 0;      // K1 launches that would not read p and nu

hipError_t take(void** p, size_t bytes) {
  *p = nullptr;
  if (g_allocs++ == g_fail_at) return hipErrorOutOfMemory;
  *p = std::malloc(bytes ? bytes : 1);
  std::memset(*p, 0x5a, std::min(bytes, (size_t)1 << 24));
  g_live.insert(*p);
  return hipSuccess;
}
hipError_t give(void* p) {
  if (!p) return hipSuccess;
  if (!g_live.erase(p)) {
    std::printf("free of memory that is not allocated\n");
    std::exit(1);
  }
  std::free(p);
  return hipSuccess;
}

void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("%s\n", what);
  std::exit(1);
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++g_pinned;
  return take(p, n);
}
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
}

namespace cup3d {

int mixed_init_pinv(MixedWorkspace&, const std::vector<double>&, std::string&) { return 0; }
int mixed_set_topology(MixedWorkspace&, int, long long, std::string&) { return 0; }
void mixed_free(MixedWorkspace&) {}
int cnn_init(CnnState&, std::string&) { return 0; }
int cnn_set_topology(CnnState&, int, const int*, const double*, std::string&) { return 0; }
void cnn_free(CnnState&) {}

// A build wants its hash table and info words clear (it clears them when it is
// told to) and leaves them used, the others clear.
void wipe(const TopoTable& t, int* info) {
  for (unsigned long long i = 0; i <= t.mask; ++i) {
    t.keys[i] = ~0ull;
    t.vals[i] = 0x7fffffff;
  }
  for (int i = 0; i < TOPO_INFO_WORDS; ++i) info[i] = TopoInfoInit(i);
}

void launch_topology_insert(hipStream_t, const TopoParams& p, const TopoTable& t, int* info,
                            bool clear, int first, int count, const int* list) {
  if (clear) wipe(t, info);
  bool clean = true;
  for (unsigned long long i = 0; i <= t.mask; ++i)
    clean = clean && t.keys[i] == ~0ull && t.vals[i] == 0x7fffffff;
  for (int i = 0; i < TOPO_INFO_WORDS; ++i) clean = clean && info[i] == TopoInfoInit(i);
  check(clean || first > 0, "a topology build found its hash table or info words used");
  std::memcpy(p.blocks + 4 * (size_t)first, list, (size_t)count * 4 * sizeof(int));
  t.keys[0] = 0;
}

void launch_topology_tables(hipStream_t, const TopoParams& p, const TopoTable& t,
                            const TopoOut& o, int* info, const TopoTable& other, int* other_info,
                            int* host_info) {
  for (unsigned long long i = 0; i <= t.mask; ++i) t.keys[i] = i;
  for (int i = 0; i < TOPO_INFO_WORDS; ++i) info[i] = i;
  std::memset(o.meta, 0, (size_t)p.nb * 32 * sizeof(int));
  for (size_t i = 0; i < topo_waves(p.nb); ++i) o.count[i] = int2{1, 1};
  for (size_t i = 0; i < (size_t)p.nb * 32; ++i) check(o.meta[i] == 0, "overlapping tables");
  if (other.keys) wipe(other, other_info);
  for (int i = 0; i < TOPO_INFO_WORDS; ++i) host_info[i] = TopoInfoInit(i);
  if (g_reject) host_info[TI_DUPLICATE] = 1;
}

void launch_spmv64(hipStream_t, int, const DevGrid<double>&, const double*, double*, const double*,
                   double*, double*, SolverState*, double*, bool, SolverState*) {}
void launch_precond_dst(hipStream_t, int mode, int, const double*, double,
                        const KrylovVectors<double>&, SolverState* st, int, const FinArgs&) {
  if (mode == PREC_P) g_short_k1 += st->p_zero;
}

void launch_remove_mean(hipStream_t, long long, double*, const double*, double inv_vol, double*,
                        double*, double*) {
  g_inv_vol = inv_vol;
}

}  // namespace cup3d

namespace {

cup3d_poisson_t make() {
  cup3d_poisson_config c;
  std::memset(&c, 0, sizeof(c));
  for (int d = 0; d < 3; ++d) {
    c.bpd[d] = 1 << 10;
    c.bc[d] = CUP3D_BC_WALL;
  }
  c.h0 = 1.0 / 24;
  c.max_iter = 10;
  c.max_restarts = 100;
  cup3d_poisson_t H = nullptr;
  check(cup3d_poisson_create(&c, &H) == 0, "create failed");
  return H;
}

std::vector<cup3d_block_desc> row(int n) {
  std::vector<cup3d_block_desc> b(n);
  for (int i = 0; i < n; ++i) b[i] = {i % 3, {i % 1024, i / 1024, n}};
  return b;
}

int topology(cup3d_poisson_t H, int n) {
  const std::vector<cup3d_block_desc> b = row(n);
  return cup3d_poisson_set_topology(H, n, b.data());
}

// Small lists, a larger one whose k-th allocation fails, and small ones again,
// for every k: each build that runs starts from a clear table.
void failed_allocations() {
  for (int k = 0;; ++k) {
    cup3d_poisson_t H = make();
    for (int i = 0; i < 3; ++i) check(topology(H, 100) == 0, "a small list failed");
    g_fail_at = g_allocs + k;
    const bool failed = topology(H, 5000) != 0;
    g_fail_at = -1;
    for (int n : {100, 120, 100, 5000, 100, 6000})
      check(topology(H, n) == 0 && H->nb == n, "a list failed after a failed allocation");
    cup3d_poisson_destroy(H);
    if (!failed) {  // every allocation had its turn
      check(k >= 10, "too few allocations were made to fail");
      return;
    }
  }
}

// The volume is summed by the mesh change, in the order of its blocks, and a
// mean removal divides by it; a rejected list leaves it.
void volume() {
  cup3d_poisson_t H = make();
  alignas(16) double x[2] = {};
  for (int n : {7, 1000, 5}) {
    const std::vector<cup3d_block_desc> b = row(n);
    double want = 0.0;
    for (const cup3d_block_desc& d : b) {
      const double h = 1.0 / 24 / double(1 << d.level);
      want += 512.0 * (h * h * h);
    }
    check(topology(H, n) == 0 && H->volume == want, "volume of a new mesh");
    g_reject = true;
    check(topology(H, 13) != 0, "a duplicate block was accepted");
    g_reject = false;
    check(cup3d_poisson_remove_mean(H, x, nullptr) == 0 && g_inv_vol == 1.0 / want,
          "volume of a mean removal");
  }
  cup3d_poisson_destroy(H);
}

// Meshes each larger than all before: no pinned allocation, and the whole list
// reaches the device, also one longer than the pinned memory it goes through.
void growing_meshes() {
  cup3d_poisson_t H = make();
  const int pinned = g_pinned;
  for (int n : {1, 100, 5000, 65535, 65536, 65537, 140000}) {
    const std::vector<cup3d_block_desc> b = row(n);
    check(topology(H, n) == 0, "a larger mesh failed");
    check(!std::memcmp(H->tp[H->tcur].blocks.p, b.data(), n * sizeof(b[0])),
          "the block list on the device");
  }
  check(g_pinned == pinned, "a mesh change allocated pinned memory");
  cup3d_poisson_destroy(H);
}

// The timed K1 of the implicit diffusion moves the five vectors that its reported
// bytes count: the state it starts from has a p.
void timed_diffusion_kernels() {
  cup3d_poisson_t H = make();
  check(topology(H, 10) == 0, "topology");
  for (int which = 0; which < 3; ++which) {
    double ms = 0, bytes = 0, flops = 0;
    check(cup3d_debug_time_diffusion_kernel(H, which, 1e-3, 1e-2, 3, &ms, &bytes, &flops) == 0,
          "timing failed");
    check(bytes == (which == 1 ? 5.0 : 2.0) * 8 * 512 * 10, "bytes of a timed kernel");
  }
  check(g_short_k1 == 0, "the timed K1 reads three vectors and is reported with five");
  cup3d_poisson_destroy(H);
}

}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "failed_allocations") failed_allocations();
  else if (what == "volume") volume();
  else if (what == "growing_meshes") growing_meshes();
  else if (what == "timed_diffusion_kernels") timed_diffusion_kernels();
  else check(false, "no such scenario");
  check(g_live.empty(), "memory was left allocated");
  std::printf("ok\n");
  return 0;
}
