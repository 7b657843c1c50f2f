// HIP kernels of the pressure-Poisson solve for gfx950 (MI355X).
//
// Vectors live in HBM as contiguous [nblocks][8][8][8] arrays, blockID-major,
// [iz][iy][ix] inside a block (Cubism's ScalarBlock order, the flat index
// j = blockID*512 + iz*64 + iy*8 + ix of PoissonSolverAMR.cpp:76).
//
// One classical BiCGSTAB iteration (BiCGSTAB.cu:474-608) runs as five fused
// kernels. Every reduction is a deterministic two-pass sum: per-workgroup
// partials, then these in workgroup order, by every workgroup of the kernel that
// uses the sum on grids of up to FIN_MAX_BLOCKS blocks, by a finalize kernel of
// one workgroup beyond (and at the ends of batches). The scalar recurrences run
// with them, on the device. The host of an FP64 solve follows a progress word
// that each iteration writes, two iterations ahead of it; that of a mixed solve
// waits every few iterations:
//   K1 k_precond_dst<P> p = r + beta (p - omega nu)  [p = r after a restart,
//                     rhat = r]; z1 = M^-1 p
//   K2 k_spmv<DOT1>   nu = A z1; alpha = rho / ((rhat, nu) + eps)
//   K3 k_precond_dst<S> s = r - alpha nu (in r); z2 = M^-1 s
//   K4 k_spmv<DOT2>   t = A z2; omega = (t, s) / ((t, t) + eps)
//   K5 k_update       x' = x + alpha z1 + omega z2; r = s - omega t;
//                     rho' = (rhat, r), |r|; x_opt / convergence / restart
// M^-1 = blockdiag(h_b^-1 P_inv), applied by sine transforms (diffusion.hip). On
// small single-level grids K1 and K2, and K3 and K4, are one kernel each.

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels.h"
#include "krylov.h"

namespace cup3d {

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
void launch_getvec64(hipStream_t s, long long n, long long zero_row, const double* rhs,
                     const double* x0, double* b, double* x, const SolverState& init,
                     SolverState* st, double* part, double tol_b) {
  const int nwg = (int)((n + 4 * BLEN - 1) / (4 * BLEN));
  // in place, and the rhs shares a part of x: the zeroed cell is another cell of the
  // rhs, which another workgroup reads, so it is zeroed behind the copy
  const uintptr_t r0 = (uintptr_t)rhs, xa = (uintptr_t)x, len = (uintptr_t)n * sizeof(double);
  const bool later = x == x0 && rhs != x && r0 < xa + len && xa < r0 + len;
  k_getvec<<<nwg, WG_THREADS, 0, s>>>(n, zero_row, rhs, x0, b, later ? nullptr : x, part);
  if (later) launch_zero_cell(s, x, zero_row);
  k_getvec_fin<<<1, WG_THREADS, 0, s>>>(init, st, part, nwg, tol_b);
}

const double* launch_start_zero64(hipStream_t s, int nb, long long zero_row, const double* rhs,
                                  const double* x, double* b, const SolverState& init,
                                  SolverState* st, SolverState* hst, double* part, double tol_b) {
  const uintptr_t n = (uintptr_t)nb * BLEN * sizeof(double), r0 = (uintptr_t)rhs, x0 = (uintptr_t)x;
  const bool copy = zero_row >= 0 || (r0 < x0 + n && x0 < r0 + n);
  k_start_zero<<<(nb + 3) / 4, WG_THREADS, 0, s>>>(nb, zero_row, rhs, copy ? b : nullptr, part);
  launch_start_fin(s, nb, init, st, hst, part, tol_b);
  return copy ? b : rhs;
}

void launch_start_fin(hipStream_t s, int nb, const SolverState& init, SolverState* st,
                      SolverState* hst, const double* part, double tol_b) {
  k_start_fin<<<1, WG_THREADS, 0, s>>>(init, st, hst, part, (nb + 3) / 4, tol_b);
}

void launch_spmv64(hipStream_t s, int mode, const DevGrid<double>& g, const double* x, double* y,
                   const double* a, double* c, double* c2, SolverState* st, double* part,
                   bool fin, SolverState* hst) {
  switch (mode) {
    case SPMV_PLAIN: spmv_launch<double, SPMV_PLAIN>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
    case SPMV_INIT: spmv_launch<double, SPMV_INIT>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
    case SPMV_DOT1: spmv_launch<double, SPMV_DOT1>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
    case SPMV_DOT2: spmv_launch<double, SPMV_DOT2>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
    case SPMV_RESID: spmv_launch<double, SPMV_RESID>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
    case SPMV_START: spmv_launch<double, SPMV_START>(s, g, x, y, a, c, c2, st, part, false); break;
    case SPMV_NET: spmv_launch<double, SPMV_NET>(s, g, x, y, a, c, c2, st, part, false); break;
    case SPMV_FINAL: spmv_launch<double, SPMV_FINAL>(s, g, x, y, a, c, c2, st, part, fin, hst); break;
  }
}

int launch_update64(hipStream_t s, const DevGrid<double>& g, const KrylovVectors<double>& v,
                    SolverState* st, double* part, int fin, bool last, SolverState* hst,
                    unsigned long long* prog, const FinArgs* sums) {
  return launch_k5<double>(s, g, v, st, part, fin, last, hst, nullptr, prog, sums);
}

// ---------------------------------------------------------------------------
// Warm start from the previous steps: directions and their least-squares
// weights (the weights themselves are solved on the host from the Gram
// matrix of the initial residual and the directions' images under A).
// ---------------------------------------------------------------------------
// d = a - b, zero in the bMean cell
__global__ __launch_bounds__(WG_THREADS) void k_guess_direction(long long n,
                                                                const double* __restrict__ a,
                                                                const double* __restrict__ b,
                                                                long long row,
                                                                double* __restrict__ d) {
  for (long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x; i < n;
       i += (long long)gridDim.x * WG_THREADS)
    d[i] = i == row ? 0.0 : a[i] - b[i];
}

// Gram matrix of up to GUESS_MAXV vectors (upper triangle, row by row:
// (0,0), (0,1), ..., (1,1), ...), fixed-order partial sums; NV vectors.
template <int NV>
__global__ __launch_bounds__(WG_THREADS) void k_guess_gram(long long n, GuessVecs r,
                                                           double* part) {
  constexpr int ND = NV * (NV + 1) / 2;
  double v[ND];
#pragma unroll
  for (int k = 0; k < ND; ++k) v[k] = 0.0;
  const long long base = (long long)blockIdx.x * (4 * BLEN);
  for (int e = threadIdx.x; e < 4 * BLEN; e += WG_THREADS) {
    const long long i = base + e;
    if (i < n) {
      double q[NV];
#pragma unroll
      for (int a = 0; a < NV; ++a) q[a] = r.v[a][i];
      int k = 0;
#pragma unroll
      for (int a = 0; a < NV; ++a)
#pragma unroll
        for (int b = a; b < NV; ++b) v[k++] += q[a] * q[b];
    }
  }
  grid_store_partial<ND>(v, part);
}

// Sums the partials and scatters them into the GUESS_MAXV-wide triangle
// (the entries of absent vectors 0).
template <int NV>
__global__ __launch_bounds__(WG_THREADS) void k_guess_gram_fin(const double* part, int nparts,
                                                               double* dots) {
  constexpr int ND = NV * (NV + 1) / 2;
  double tot[ND];
  grid_sum_partials<ND>(part, nparts, tot);
  if (threadIdx.x == 0) {
    int k = 0, o = 0;
    for (int a = 0; a < GUESS_MAXV; ++a)
      for (int b = a; b < GUESS_MAXV; ++b, ++o) dots[o] = a < NV && b < NV ? tot[k++] : 0.0;
  }
}

struct GuessWeights {
  double w[HIST_MAX];
};

// x = x0 + sum_{k < m} g_k (h_{k-1} - h_k) + gnet (pred - x0), h_{-1} = x0;
// the bMean cell keeps x0's value (every direction is zero there)
__global__ __launch_bounds__(WG_THREADS) void k_guess_blend(long long n,
                                                            const double* __restrict__ x0,
                                                            GuessVecs h, GuessWeights g, int m,
                                                            const double* __restrict__ pred,
                                                            double gnet, long long row,
                                                            double* __restrict__ x) {
  for (long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x; i < n;
       i += (long long)gridDim.x * WG_THREADS) {
    const double b = x0[i];
    double v = b, prev = b;
    for (int k = 0; k < m; ++k) {
      const double hk = h.v[k][i];
      v = fma(g.w[k], prev - hk, v);
      prev = hk;
    }
    if (gnet != 0.0) v = fma(gnet, pred[i] - b, v);
    x[i] = i == row ? b : v;
  }
}

// Streaming copy for the bandwidth ceiling report (nontemporal float4 loads
// and stores, grid-stride over a fixed grid).
typedef float f32x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(WG_THREADS) void k_stream_copy(long long n4,
                                                            const f32x4* __restrict__ a,
                                                            f32x4* __restrict__ b) {
  for (long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x; i < n4;
       i += (long long)gridDim.x * WG_THREADS)
    __builtin_nontemporal_store(__builtin_nontemporal_load(&a[i]), &b[i]);
}

void launch_stream_copy(hipStream_t s, long long n4, const void* a, void* b) {
  k_stream_copy<<<1024, WG_THREADS, 0, s>>>(n4, static_cast<const f32x4*>(a),
                                            static_cast<f32x4*>(b));
}

// Between pinned host memory and a device vector. PCIe bounds it: 64 workgroups
// keep 256 KiB in flight, which reaches the link's 55 GB/s from 1 MiB on.
__global__ __launch_bounds__(WG_THREADS) void k_host_copy(long long n4,
                                                          const f32x4* __restrict__ a,
                                                          f32x4* __restrict__ b) {
  for (long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x; i < n4;
       i += (long long)gridDim.x * WG_THREADS)
    b[i] = a[i];
}

void launch_host_copy(hipStream_t s, long long n4, const void* a, void* b) {
  const int nwg = (int)std::min<long long>((n4 + WG_THREADS - 1) / WG_THREADS, 64);
  k_host_copy<<<nwg, WG_THREADS, 0, s>>>(n4, static_cast<const f32x4*>(a), static_cast<f32x4*>(b));
}

// Caller-side projection after a solve (PressureProjection.cpp:404-431):
// x -= sum_b h_b^3 sum x / sum_b 512 h_b^3, the volume-weighted mean, with the
// sum in a fixed order.
__global__ __launch_bounds__(WG_THREADS) void k_wsum(long long n, const double* __restrict__ x,
                                                     const double* __restrict__ h3,
                                                     double* part) {
  double v[1] = {0.0};
  const long long i0 = (long long)blockIdx.x * (4 * BLEN) + 8 * threadIdx.x;
  if (i0 < n) {
    double xv[8];
    load8(x + i0, xv);
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += xv[e];
    v[0] = h3[i0 / BLEN] * s;
  }
  grid_store_partial<1>(v, part);
}

__global__ __launch_bounds__(WG_THREADS) void k_wsum_fin(const double* part, int nparts,
                                                         double* out, double* host) {
  double tot[1];
  grid_sum_partials<1>(part, nparts, tot);
  if (threadIdx.x == 0) out[0] = host[0] = tot[0];
}

// x -= mean. SUMS: every workgroup adds the partials itself, in the finalize
// kernel's order, and the first one gives the sum to the host.
template <bool SUMS>
__global__ __launch_bounds__(WG_THREADS) void k_sub_mean(long long n, double* __restrict__ x,
                                                         const double* __restrict__ part,
                                                         int nparts, double inv_vol,
                                                         double* __restrict__ host) {
  typedef double double2_t __attribute__((ext_vector_type(2)));
  double tot[1];
  if (SUMS) {
    grid_sum_partials<1>(part, nparts, tot);
    if (blockIdx.x == 0 && threadIdx.x == 0) host[0] = tot[0];
  } else {
    tot[0] = part[0];
  }
  const double m = tot[0] * inv_vol;
  double2_t* __restrict__ x2 = reinterpret_cast<double2_t*>(x);
  for (long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x; i < n / 2;
       i += (long long)gridDim.x * WG_THREADS)
    x2[i] -= (double2_t){m, m};
}

// On grids of up to FIN_MAX_BLOCKS blocks (2048 partials) the sum's finalize
// kernel, 3 us and a launch, is left out; adding all partials in every workgroup
// costs as much at 16 384 blocks (45 us either way) and 118 against 107 us at
// 51 200. A call on 64 blocks 21.4 -> 17.7 us, on 8192 35.5 -> 33.7 us (with the
// sum written to the host by a kernel, not copied).
void launch_remove_mean(hipStream_t s, long long n, double* x, const double* h3, double inv_vol,
                        double* part, double* wsum, double* host) {
  const int nwg = (int)((n + 4 * BLEN - 1) / (4 * BLEN));
  const int nsub = (int)std::min<long long>((n / 2 + WG_THREADS - 1) / WG_THREADS, 8192);
  k_wsum<<<nwg, WG_THREADS, 0, s>>>(n, x, h3, part);
  if (n <= (long long)FIN_MAX_BLOCKS * BLEN) {
    k_sub_mean<true><<<std::min(nsub, 1024), WG_THREADS, 0, s>>>(n, x, part, nwg, inv_vol, host);
  } else {
    k_wsum_fin<<<1, WG_THREADS, 0, s>>>(part, nwg, wsum, host);
    k_sub_mean<false><<<nsub, WG_THREADS, 0, s>>>(n, x, wsum, 1, inv_vol, host);
  }
}


__global__ void k_zero_cell(double* __restrict__ x, long long row) { x[row] = 0.0; }

void launch_zero_cell(hipStream_t s, double* x, long long row) {
  if (row >= 0) k_zero_cell<<<1, 1, 0, s>>>(x, row);
}

void launch_guess_direction(hipStream_t s, long long n, const double* a, const double* b,
                            long long row, double* d) {
  const int nwg = (int)std::min<long long>((n + WG_THREADS - 1) / WG_THREADS, 8192);
  k_guess_direction<<<nwg, WG_THREADS, 0, s>>>(n, a, b, row, d);
}

template <int NV>
static void guess_gram_nv(hipStream_t s, long long n, const GuessVecs& r, double* part,
                          double* dots) {
  const int nwg = (int)((n + 4 * BLEN - 1) / (4 * BLEN));
  k_guess_gram<NV><<<nwg, WG_THREADS, 0, s>>>(n, r, part);
  k_guess_gram_fin<NV><<<1, WG_THREADS, 0, s>>>(part, nwg, dots);
}

void launch_guess_gram(hipStream_t s, long long n, const GuessVecs& r, int nv, double* part,
                       double* dots) {
  static_assert(GUESS_MAXV == 10, "one instance per vector count");
  switch (nv) {
    case 1: guess_gram_nv<1>(s, n, r, part, dots); break;
    case 2: guess_gram_nv<2>(s, n, r, part, dots); break;
    case 3: guess_gram_nv<3>(s, n, r, part, dots); break;
    case 4: guess_gram_nv<4>(s, n, r, part, dots); break;
    case 5: guess_gram_nv<5>(s, n, r, part, dots); break;
    case 6: guess_gram_nv<6>(s, n, r, part, dots); break;
    case 7: guess_gram_nv<7>(s, n, r, part, dots); break;
    case 8: guess_gram_nv<8>(s, n, r, part, dots); break;
    case 9: guess_gram_nv<9>(s, n, r, part, dots); break;
    default: guess_gram_nv<10>(s, n, r, part, dots); break;
  }
}

void launch_guess_blend(hipStream_t s, long long n, const double* x0, const GuessVecs& h,
                        const double* gt, int m, const double* pred, double gnet, long long row,
                        double* x) {
  GuessWeights g{};
  for (int k = 0; k < m && k < HIST_MAX; ++k) g.w[k] = gt[k];
  const int nwg = (int)std::min<long long>((n + WG_THREADS - 1) / WG_THREADS, 8192);
  k_guess_blend<<<nwg, WG_THREADS, 0, s>>>(n, x0, h, g, m < HIST_MAX ? m : HIST_MAX, pred, gnet,
                                           row, x);
}

}  // namespace cup3d
