// Topology build on the device: the per-face tables the SpMV, the caller
// kernels and the learned warm start read (same-level neighbours, face
// kinds, coarse/fine partners, index parities, per-block h, 1/h, h^3), built
// from the block list (level, index[3]) in a few kernels instead of a serial
// host pass. It replaces the face classification of the reference's
// PoissonSolverExp::getMat (source/poisson/PoissonSolverExp.cpp:221-373: the
// per-face same-level / coarser / finer tests of makeFlux, .cpp:157-219, and
// the periodic wrap of .cpp:361), which reruns after every mesh change
// (Simulation.cpp:385).
//
//   k_topo_init    clear the hash table and the info words (a fill kernel, no
//                  memset), where the build before did not
//   k_topo_insert  one thread per block: read it from the copy of the caller's
//                  list in pinned host memory (a launch per 65 536 blocks, which
//                  that memory holds) and keep it, validate level and index, insert
//                  key(level, i, j, k) -> the smallest block id holding it
//                  (open addressing, linear probing, 64-bit CAS)
//   k_topo_tables  eight threads per block: one per face: same-level neighbour
//                  (with the periodic wrap), else the coarser block, else the
//                  four finer blocks by quadrant; a face with none of them
//                  violates the 2:1 balance; one for the duplicate test, h,
//                  1/h, h^3 (FP64 and FP32), index parities, the origin block.
//                  It also clears the other generation's hash table and info
//                  words, which nothing reads any more and the next build uses
//   k_topo_report  the info words, with the face counts added up, to the host
//                  (pinned memory)
// Errors are reported as the smallest offending block (or block face) id, so
// the message names the same block a sequential pass would stop at.
//
// Bound by launches and the round trips of the hash probes, of which a face's
// first six are in flight together. A mesh change of 4440 blocks with one operator
// application takes 63 us on a handle that has had a mesh of that size: 97 us with a
// clearing kernel, separate kernels per block and per face and pageable copies, 70
// us with the list and the info words moved by the copy engine, the probes one
// after the other and a counter update per wavefront (whose 7400 updates of two
// words were most of the 116 us the tables of 59 012 blocks took; now 31 us). A
// larger mesh than all before it is bound by the allocation of the tables and the
// solver's vectors instead: about 1.3 ms at 4000 to 40 000 blocks.

#include <hip/hip_runtime.h>

#include "poisson_internal.h"
#include "topology_gpu.h"

namespace cup3d {
namespace {

constexpr unsigned long long KEY_EMPTY = ~0ull;
constexpr int INDEX_BITS = 20;
constexpr int LEVEL_MAX = 15;

__device__ __forceinline__ unsigned long long tkey(int l, int i, int j, int k) {
  return ((unsigned long long)l << 60) | ((unsigned long long)i << 40) |
         ((unsigned long long)j << 20) | (unsigned long long)k;
}

__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  // splitmix64 finaliser (Steele, Lea, Flood 2014): spreads the packed
  // (level, i, j, k) keys over the table
  x ^= x >> 30;
  x *= 0xbf58476d1ce4e5b9ull;
  x ^= x >> 27;
  x *= 0x94d049bb133111ebull;
  x ^= x >> 31;
  return x;
}

// A lookup in two parts, so that the first probes of several are in flight
// together (key and value of a slot with them): tprobe() starts one, tresolve()
// returns the block, or -1.
struct Probe {
  unsigned long long key, slot, k0;
  int v0;
  bool ok;
};
__device__ __forceinline__ Probe tprobe(const TopoTable& t, int l, int i, int j, int k) {
  Probe q;
  q.ok = l >= 0 && l <= LEVEL_MAX && i >= 0 && j >= 0 && k >= 0 && i < (1 << INDEX_BITS) &&
         j < (1 << INDEX_BITS) && k < (1 << INDEX_BITS);
  q.key = tkey(l, i, j, k);
  q.slot = q.ok ? mix64(q.key) & t.mask : 0;
  q.k0 = t.keys[q.slot];
  q.v0 = t.vals[q.slot];
  return q;
}
__device__ __forceinline__ int tresolve(const TopoTable& t, const Probe& q) {
  if (!q.ok || q.k0 == KEY_EMPTY) return -1;
  if (q.k0 == q.key) return q.v0;
  unsigned long long slot = (q.slot + 1) & t.mask;
  for (unsigned long long probe = 0; probe < t.mask; ++probe) {
    const unsigned long long s = t.keys[slot];
    const int v = t.vals[slot];
    if (s == q.key) return v;
    if (s == KEY_EMPTY) return -1;
    slot = (slot + 1) & t.mask;
  }
  return -1;
}

// level 0..15 and 0 <= index < (bpd << level) <= 2^20 in every direction
__device__ __forceinline__ bool block_ok(const TopoParams& p, int4 B) {
  if (B.x < 0 || B.x > LEVEL_MAX || B.y < 0 || B.z < 0 || B.w < 0) return false;
  const int I[3] = {B.y, B.z, B.w};
  for (int d = 0; d < 3; ++d)
    if (I[d] >= (p.bpd[d] << B.x) || (p.bpd[d] << B.x) > (1 << INDEX_BITS)) return false;
  return true;
}

__global__ __launch_bounds__(WG_THREADS) void k_topo_init(TopoTable t, int* info) {
  const unsigned long long i = (unsigned long long)blockIdx.x * WG_THREADS + threadIdx.x;
  if (i <= t.mask) {
    t.keys[i] = KEY_EMPTY;
    t.vals[i] = 0x7fffffff;
  }
  if (i < TOPO_INFO_WORDS) info[i] = TopoInfoInit(i);
}

__global__ __launch_bounds__(WG_THREADS) void k_topo_insert(TopoParams p, TopoTable t, int* info,
                                                            int first, int count,
                                                            const int* __restrict__ list) {
  const int i = blockIdx.x * WG_THREADS + threadIdx.x, b = first + i;
  if (i >= count) return;
  const int4 B = reinterpret_cast<const int4*>(list)[i];
  reinterpret_cast<int4*>(p.blocks)[b] = B;
  const int l = B.x, I[3] = {B.y, B.z, B.w};
  if (l < 0 || l > LEVEL_MAX || I[0] < 0 || I[1] < 0 || I[2] < 0) {
    atomicMin(&info[TI_INVALID], b);
    return;
  }
  for (int d = 0; d < 3; ++d) {
    // p.bpd[d] << l fits 32 bits (bpd < 2^16, l <= 15)
    if (I[d] >= (p.bpd[d] << l)) {
      atomicMin(&info[TI_OUTSIDE], b);
      return;
    }
    if ((p.bpd[d] << l) > (1 << INDEX_BITS)) {  // the key holds 20-bit indices
      atomicMin(&info[TI_TOO_FINE], b);
      return;
    }
  }
  const unsigned long long key = tkey(l, I[0], I[1], I[2]);
  unsigned long long slot = mix64(key) & t.mask;
  for (unsigned long long probe = 0; probe <= t.mask; ++probe) {
    const unsigned long long prev = atomicCAS(&t.keys[slot], KEY_EMPTY, key);
    if (prev == KEY_EMPTY || prev == key) {
      atomicMin(&t.vals[slot], b);
      return;
    }
    slot = (slot + 1) & t.mask;
  }
  atomicMin(&info[TI_FULL], b);  // unreachable: the table holds >= 2 nb slots
}

// Block b's own entries.
__device__ void topo_block(const TopoParams& p, const TopoTable& t, const TopoOut& o, int* info,
                           int b, int4 B) {
  if (tresolve(t, tprobe(t, B.x, B.y, B.z, B.w)) != b) atomicMin(&info[TI_DUPLICATE], b);
  // h0 / 2^l is exact (a power-of-two scaling), as is its FP32 rounding of
  // the same FP64 value
  const double h = p.h0 / (double)(1 << B.x);
  const double ih = 1.0 / h;
  o.h[b] = h;
  o.invh[b] = ih;
  o.h3[b] = h * h * h;
  o.hf[b] = (float)h;
  o.invhf[b] = (float)ih;
  const int8_t par = (int8_t)((B.y & 1) | ((B.z & 1) << 1) | ((B.w & 1) << 2));
  o.bpar[b] = par;
  o.meta[(size_t)b * 32 + 30] = par;
  o.meta[(size_t)b * 32 + 31] = 0;
  if (B.y == 0 && B.z == 0 && B.w == 0) atomicMax(&info[TI_ORIGIN], b);
}

// Face f of block b; returns its kind.
__device__ int topo_face(const TopoParams& p, const TopoTable& t, const TopoOut& o, int* info,
                         int b, int f, int4 B) {
  const int l = B.x;
  const int d = f >> 1, s = (f & 1) ? 1 : -1;
  const int n = p.bpd[d] << l;
  int I[3] = {B.y, B.z, B.w};
  int kind = FACE_NONE, nbr = -1, part[4] = {-1, -1, -1, -1};
  const bool boundary = (s < 0) ? I[d] == 0 : I[d] == n - 1;
  if (!(boundary && p.bc[d] != 1)) {  // a wall or freespace face has no flux
    I[d] = ((I[d] + s) % n + n) % n;
    // the block of every case at once: the same level, the coarser one, and the
    // four children adjacent to this face
    const int t1 = d == 0 ? 1 : (d == 1 ? 2 : 0), t2 = d == 0 ? 2 : (d == 1 ? 0 : 1);
    const Probe ps = tprobe(t, l, I[0], I[1], I[2]);
    const Probe pc = tprobe(t, l - 1, I[0] >> 1, I[1] >> 1, I[2] >> 1);
    Probe pf[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int C[3] = {2 * I[0], 2 * I[1], 2 * I[2]};
      C[d] += (s < 0) ? 1 : 0;
      C[t1] += q & 1;
      C[t2] += (q >> 1) & 1;
      pf[q] = tprobe(t, l + 1, C[0], C[1], C[2]);
    }
    const int same = tresolve(t, ps);
    if (same >= 0) {
      kind = FACE_SAME;
      nbr = same;
    } else {
      const int c = tresolve(t, pc);
      if (c >= 0) {
        kind = FACE_COARSE;
        part[0] = c;
      } else {
        bool ok = true;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          part[q] = tresolve(t, pf[q]);
          ok = ok && part[q] >= 0;
        }
        if (ok) {
          kind = FACE_FINE;
        } else {
          atomicMin(&info[TI_BALANCE], b * 6 + f);
#pragma unroll
          for (int q = 0; q < 4; ++q) part[q] = -1;
        }
      }
    }
  }
  const size_t gid = (size_t)b * 6 + f;
  o.kind[gid] = (int8_t)kind;
  o.nbr[gid] = nbr;
  reinterpret_cast<int4*>(o.fnb)[gid] = make_int4(part[0], part[1], part[2], part[3]);
  reinterpret_cast<int4*>(o.meta + (size_t)b * 32)[f] = make_int4(part[0], part[1], part[2], part[3]);
  o.meta[(size_t)b * 32 + 24 + f] = kind;
  return kind;
}

__global__ __launch_bounds__(WG_THREADS) void k_topo_tables(TopoParams p, TopoTable t, TopoOut o,
                                                            int* info, TopoTable other,
                                                            int* other_info) {
  const long long gid = (long long)blockIdx.x * WG_THREADS + threadIdx.x;
  const int b = (int)(gid >> 3), f = (int)(gid & 7);
  int kind = FACE_NONE;
  if (b < p.nb) {
    const int4 B = reinterpret_cast<const int4*>(p.blocks)[b];
    if (block_ok(p, B)) {  // else reported by k_topo_insert
      if (f < 6) kind = topo_face(p, t, o, info, b, f, B);
      else if (f == 6) topo_block(p, t, o, info, b, B);
    }
  }
  // a count per wavefront, added by k_topo_report
  const unsigned long long nc = __ballot(kind == FACE_COARSE), nf = __ballot(kind == FACE_FINE);
  if ((threadIdx.x & 63) == 0) o.count[gid >> 6] = make_int2(__popcll(nc), __popcll(nf));
  if (other.keys) {
    for (unsigned long long i = gid; i <= other.mask; i += (unsigned long long)gridDim.x * WG_THREADS) {
      other.keys[i] = KEY_EMPTY;
      other.vals[i] = 0x7fffffff;
    }
    if (gid < TOPO_INFO_WORDS) other_info[gid] = TopoInfoInit(gid);
  }
}

__global__ __launch_bounds__(WG_THREADS) void k_topo_report(const int* info, const int2* count,
                                                            int waves, int* host) {
  __shared__ int sum[2];
  if (threadIdx.x < 2) sum[threadIdx.x] = 0;
  __syncthreads();
  int nc = 0, nf = 0;
  for (int i = threadIdx.x; i < waves; i += WG_THREADS) {
    nc += count[i].x;
    nf += count[i].y;
  }
  atomicAdd(&sum[0], nc);
  atomicAdd(&sum[1], nf);
  __syncthreads();
  const int i = threadIdx.x;
  if (i < TOPO_INFO_WORDS)
    host[i] = i == TI_N_COARSE ? sum[0] : (i == TI_N_FINE ? sum[1] : info[i]);
}

}  // namespace

void launch_topology_insert(hipStream_t s, const TopoParams& p, const TopoTable& t, int* info,
                            bool clear, int first, int count, const int* list) {
  if (clear) {
    const unsigned long long cap = t.mask + 1;
    const int ninit = (int)((cap + WG_THREADS - 1) / WG_THREADS);
    k_topo_init<<<ninit, WG_THREADS, 0, s>>>(t, info);
  }
  const int nwb = (count + WG_THREADS - 1) / WG_THREADS;
  k_topo_insert<<<nwb, WG_THREADS, 0, s>>>(p, t, info, first, count, list);
}

void launch_topology_tables(hipStream_t s, const TopoParams& p, const TopoTable& t,
                            const TopoOut& o, int* info, const TopoTable& other, int* other_info,
                            int* host_info) {
  const int nwt = (int)(((long long)p.nb * 8 + WG_THREADS - 1) / WG_THREADS);
  k_topo_tables<<<nwt, WG_THREADS, 0, s>>>(p, t, o, info, other, other_info);
  k_topo_report<<<1, WG_THREADS, 0, s>>>(info, o.count, nwt * (WG_THREADS / 64), host_info);
}

}  // namespace cup3d
