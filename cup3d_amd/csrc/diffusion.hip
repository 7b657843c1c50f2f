// Implicit diffusion on the device: the block preconditioner and the
// velocity gather/scatter around the three solves of one step
// (AdvectionDiffusionImplicit.h:21-525, AdvectionDiffusionImplicit.cpp:
// 354-419). The operator itself is k_spmv with HELM (krylov.h).
//
// Preconditioner. The reference runs, per block, CG on the local matrix
// A_loc(sigma) = 6-neighbour adjacency + (-6 - h^2 sigma) I with zero
// padding, sigma = 1 / (nu dt), to 1e-7 of its initial residual
// (DiffusionSolverAMRKernels.cpp:149-213), i.e. it approximates
// z_b = h_b^-1 A_loc(sigma_b)^-1 p_b, a matrix that differs per level. That
// matrix is diagonalised by the 3-D discrete sine transform for every sigma:
//   A_loc(sigma)^-1 = S diag(1 / (l_a + l_b + l_c - h^2 sigma)) S,
//   S = S1 (x) S1 (x) S1,  S1[k][i] = sqrt(2/9) sin(pi (k+1)(i+1) / 9),
//   l_k = 2 cos(pi (k+1) / 9) - 2,
// S1 symmetric and orthogonal. So the exact block inverse of any level is
// three separable 8-point transforms, a per-mode scaling and three more
// transforms: 96 flops per cell instead of a 512 x 512 product, no per-level
// matrices, and the kernel is bound by HBM like the vector updates it is
// fused with.
//
// One wavefront per block. Every 1-D transform runs on eight values in one
// lane's registers: the z transforms on the column of lane (ix, iy), the y and
// x transforms after a transposition through the wavefront's own LDS slice
// (eight writes and eight reads a lane; rows padded to 9 values and planes to
// 72, so that the reads along x and along y fall in distinct banks), and the
// wavefront synchronises only with itself. S1 has four distinct magnitudes and
// S1[k][7-i] = (-1)^k S1[k][i], so a transform is 8 additions and 32
// multiplications by literals, and no table is read.
// Transforming y and x with one LDS read per product, S1 in scalar registers
// (64 of them spilled) and eight divisions a lane instead, K1 on 64 blocks, one
// wavefront's latency, took 9.2 us; now 6.4 us (8192 blocks: 34.2 -> 31.7 us).

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "diffusion.h"
#include "krylov.h"

namespace cup3d {
namespace {

constexpr int DL_ROW = 9;               // padded row (ix) stride, values
constexpr int DL_PLANE = BS * DL_ROW;   // one z plane (or z mode)
constexpr int DL_WAVE = BS * DL_PLANE;  // one wavefront's slice

// sqrt(2/9) sin(pi m / 9), m = 1..4, and the eigenvalues 2 cos(pi (k+1) / 9) - 2
constexpr double DST_C[4] = {0.1612298417653168423518581, 0.3030129851146957862456487,
                             0.4082482904638630163662140, 0.4642428268800126285975068};
__device__ constexpr double DST_L[BS] = {
    -0.1206147584281832318917814, -0.4679111137620439295952147, -1.0,
    -1.652703644666139302296567,  -2.347296355333860697703433,  -3.0,
    -3.532088886237956070404785,  -3.879385241571816768108219};

__device__ constexpr double dst_entry(int k, int i) {  // S1[k][i]
  int m = (k + 1) * (i + 1) % 18;
  double sign = 1.0;
  if (m > 9) {
    m = 18 - m;
    sign = -1.0;
  }
  if (m > 4) m = 9 - m;
  return m == 0 ? 0.0 : sign * DST_C[m - 1];
}

// v = S1 v (S1 symmetric and orthogonal: also the inverse transform)
template <typename T>
__device__ __forceinline__ void dst8(T (&v)[BS]) {
  T e[2][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    e[0][i] = v[i] + v[7 - i];
    e[1][i] = v[i] - v[7 - i];
  }
#pragma unroll
  for (int k = 0; k < BS; ++k) {
    T acc = (T)dst_entry(k, 0) * e[k & 1][0];
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (dst_entry(k, i) != 0.0) acc = fma((T)dst_entry(k, i), e[k & 1][i], acc);
    v[k] = acc;
  }
}

// The lane's values to and from the slice, strides in values: index j of the
// lane's axis at base + j * stride.
template <int STRIDE, typename T>
__device__ __forceinline__ void put8(T* L, int base, const T (&v)[BS]) {
#pragma unroll
  for (int j = 0; j < BS; ++j) L[base + j * STRIDE] = v[j];
  wave_sync();
}
template <int STRIDE, typename T>
__device__ __forceinline__ void get8(const T* L, int base, T (&v)[BS]) {
#pragma unroll
  for (int j = 0; j < BS; ++j) v[j] = L[base + j * STRIDE];
  wave_sync();
}

// 1 / x to the last bit or two: the hardware's estimate and two Newton steps
// (one in FP32). The block inverse it scales stays as accurate as with divisions,
// whose error is that of the six transforms: rms per block against 80-bit
// arithmetic on 1728 blocks of white noise 1.76e-7 in FP32 and 2.6e-16 in FP64
// (Helmholtz 2.5e-16), by divisions 1.73e-7, 2.5e-16 and 2.5e-16; with one LDS read
// per product and table values (see above) it was 1.90e-7, 9.1e-16 and 1.4e-15.
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}

// z = h^-1 A_loc(sigma_b)^-1 v for the column v of this lane (in place).
template <typename T>
__device__ __forceinline__ void dst_apply(T* L, int lane, T h, T sigma, T (&v)[BS]) {
  const int a = lane & 7, c = lane >> 3;
  const int zcol = c * DL_ROW + a, ycol = c * DL_PLANE + a, xrow = c * DL_PLANE + a * DL_ROW;
  const T shift = h * h * sigma;
  const T base = (T)DST_L[a] + (T)DST_L[c] - shift;  // of (ky, kz) = (a, c)
  dst8(v);  // z, lane (ix, iy)
  put8<DL_PLANE>(L, zcol, v);
  get8<DL_ROW>(L, ycol, v);
  dst8(v);  // y, lane (ix, kz)
  put8<DL_ROW>(L, ycol, v);
  get8<1>(L, xrow, v);
  dst8(v);  // x, lane (ky, kz)
  const T ih = (T)1 / h;
  if (shift < (T)1e18) {  // the estimate's range; a shift beyond it divides
#pragma unroll
    for (int k = 0; k < BS; ++k) v[k] *= recip(base + (T)DST_L[k]) * ih;
  } else {
#pragma unroll
    for (int k = 0; k < BS; ++k) v[k] = v[k] / (h * (base + (T)DST_L[k]));
  }
  dst8(v);  // inverse x
  put8<1>(L, xrow, v);
  get8<DL_ROW>(L, ycol, v);
  dst8(v);  // inverse y
  put8<DL_ROW>(L, ycol, v);
  get8<DL_PLANE>(L, zcol, v);
  dst8(v);  // inverse z
}

// K1 / K3 of the classical iteration (kernels.hip) with this preconditioner,
// in FP64 (the FP64 forms) or FP32 (the inner solve of the mixed forms):
//   PREC_P  p = r + beta (p - omega nu) [p = r after a restart, rhat = r];
//           z1 = M^-1 p
//   PREC_S  s = r - alpha nu (into r); z2 = M^-1 s
//   PREC_PLAIN  z1 = M^-1 p
template <typename T, int MODE, int FIN>
__global__ __launch_bounds__(WG_THREADS) void k_precond_dst(int nb, const T* __restrict__ hb,
                                                            T sigma, KrylovVectors<T> v,
                                                            SolverState* st, FinArgs f) {
  __shared__ T Ls[WG_THREADS / 64][DL_WAVE];
  __shared__ SolverState S;
  if (!FIN && MODE != PREC_PLAIN && st->status != ST_RUNNING) return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.x * (WG_THREADS / 64) + w;
  const size_t off = (size_t)b * BLEN + lane;
  T c[BS], ra[BS], rb[BS];
  // after a restart (and in the first iteration) p = r: nu and p are not read
  const bool fresh = !FIN && MODE == PREC_P && st->p_zero;
  if (b < nb) {
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) {
      const size_t i = off + iz * 64;
      if (MODE == PREC_P) {
        ra[iz] = v.r[i];
        if (!fresh) {
          rb[iz] = v.nu[i];
          c[iz] = v.p[i];
        }
      } else if (MODE == PREC_S) {
        ra[iz] = v.r[i];
        rb[iz] = v.nu[i];
      } else {
        c[iz] = v.p[i];
      }
    }
  }
  const SolverState* sp = st;
  if constexpr (FIN != FIN_KERNEL) {
    T yr = 0;
    consumer_state<MODE == PREC_P ? USE_P : USE_S, FIN, T>(st, f, S, yr);
    if (S.status != ST_RUNNING) return;
    sp = &S;
    if (FIN == FIN_ROW && MODE == PREC_S && b < nb && (long long)off == f.row) {
      rb[0] = yr;  // the mean-constraint row of nu, which the SpMV left out
      v.nu[off] = yr;
    }
  }
  if (b >= nb) return;  // no workgroup barrier below: only this wavefront's slice
  const T beta = MODE == PREC_P ? (T)sp->beta : (T)0;
  const T omega = MODE == PREC_P ? (T)sp->omega : (T)0;
  const T alpha = MODE == PREC_S ? (T)sp->alpha : (T)0;
  const int pzero = MODE == PREC_P ? sp->p_zero : 0;
  const int restart = MODE == PREC_P ? sp->restart_pending : 0;
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) {
    const size_t i = off + iz * 64;
    if (MODE == PREC_P) {
      // BiCGSTAB.cu:518-522
      c[iz] = pzero ? ra[iz] : fma(beta, fma(-omega, rb[iz], c[iz]), ra[iz]);
      v.pw[i] = c[iz];
      if (restart) v.rhat[i] = ra[iz];
    } else if (MODE == PREC_S) {
      c[iz] = fma(-alpha, rb[iz], ra[iz]);  // :546-549
      v.s[i] = c[iz];
    }
  }
  dst_apply<T>(Ls[w], lane, hb[b], sigma, c);
  T* __restrict__ out = MODE == PREC_S ? v.z2 : v.z1;
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) out[off + iz * 64] = c[iz];
}

// K1 and K2, or K3 and K4, in one kernel: the block inverse and the operator on
// its result, for single-level grids of up to FUSE_MAX_BLOCKS blocks. Such
// kernels are bound by their launches and by chains of memory latencies, not by
// the work, so a workgroup of seven wavefronts makes the vectors of its block and
// of the six neighbours for itself (each wavefront one block, seven times the
// arithmetic) and needs no other workgroup's result: three launches an iteration
// instead of five. On 64 blocks K1 and K2 took 6.7 + 4.7 us and take 8.1, K3 and K4
// 5.5 + 4.3 us and take 7.1; a solve of ten iterations 320 -> 275 us.
// Wavefront 0 has the workgroup's own block and writes it; the neighbours'
// wavefronts leave the layer of cells that touches it in LDS. The product is
// split over four wavefronts, two z planes each. What a neighbour's workgroup
// reads is not written in the same kernel: p, nu and s leave for vectors other
// than those they are made from (v.pw, y of PREC_P, v.s), and so do the sums.
//   PREC_P  p, z1, y = nu = A z1; sums (rhat, nu)
//   PREC_S  s, z2, y = t = A z2;  sums (t, s), (t, t)
// BM1: the mean-constraint row as k_spmv leaves it (its sum first, its other
// factor behind the sums). HELM: as in k_spmv.
constexpr int FUSE_T = 7 * 64;

template <int MODE, int FIN, bool BM1, bool HELM>
__global__ __launch_bounds__(FUSE_T) void k_precond_spmv(DevGrid<double> g,
                                                         KrylovVectors<double> v,
                                                         double* __restrict__ y, SolverState* st,
                                                         FinArgs f, double* __restrict__ part) {
  constexpr int N = (BM1 ? 1 : 0) + (MODE == PREC_P ? 1 : 2);
  __shared__ double Ls[7][DL_WAVE];
  __shared__ double xs[BLEN], fc[6][64], sv[MODE == PREC_S ? BLEN : 1], red[N][4];
  __shared__ SolverState S;
  if (!FIN && st->status != ST_RUNNING) return;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ix = lane & 7, iy = lane >> 3;
  const int bw = w == 0 ? b : g.nbr[b * 6 + w - 1];  // -1: no block there
  const size_t off = (size_t)(bw < 0 ? 0 : bw) * BLEN + lane, own = (size_t)b * BLEN + lane;
  double c[BS], ra[BS], rb[BS];
  const bool fresh = !FIN && MODE == PREC_P && st->p_zero;
  if (bw >= 0) {
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) {
      const size_t i = off + iz * 64;
      ra[iz] = v.r[i];
      if (!fresh) rb[iz] = v.nu[i];
      if (MODE == PREC_P && !fresh) c[iz] = v.p[i];
    }
  }
  const SolverState* sp = st;
  if constexpr (FIN != FIN_KERNEL) {
    double yr = 0;
    consumer_state<MODE == PREC_P ? USE_P : USE_S, FIN, double>(st, f, S, yr);
    if (S.status != ST_RUNNING) return;
    sp = &S;
    if (FIN == FIN_ROW && MODE == PREC_S && bw >= 0 && (long long)off == f.row) {
      rb[0] = yr;  // the mean-constraint row of nu, which the product left out
      if (w == 0) v.nu[off] = yr;
    }
  }
  const int pzero = MODE == PREC_P ? sp->p_zero : 0;
  const int restart = MODE == PREC_P ? sp->restart_pending : 0;
  // rhat in the cells of this wavefront's two planes (r itself after a restart)
  double a[2] = {};
  if (MODE == PREC_P && w < 4) {
    const double* rhat = restart ? v.r : (sp->rhat_own ? v.rhat : v.rhat0);
#pragma unroll
    for (int k = 0; k < 2; ++k) a[k] = rhat[own + (2 * w + k) * 64];
  }
  if (bw >= 0) {
    const double beta = MODE == PREC_P ? sp->beta : 0.0, omega = MODE == PREC_P ? sp->omega : 0.0;
    const double alpha = MODE == PREC_S ? sp->alpha : 0.0;
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) {
      const size_t i = off + iz * 64;
      if (MODE == PREC_P) {
        c[iz] = pzero ? ra[iz] : fma(beta, fma(-omega, rb[iz], c[iz]), ra[iz]);
        if (w == 0) v.pw[i] = c[iz];
        if (w == 0 && restart) v.rhat[i] = ra[iz];
      } else {
        c[iz] = fma(-alpha, rb[iz], ra[iz]);
        if (w == 0) {
          v.s[i] = c[iz];
          sv[iz * 64 + lane] = c[iz];
        }
      }
    }
    dst_apply<double>(Ls[w], lane, g.h[bw], HELM ? g.helm_sigma : 0.0, c);
    if (w == 0) {
      double* __restrict__ out = MODE == PREC_S ? v.z2 : v.z1;
#pragma unroll
      for (int iz = 0; iz < BS; ++iz) {
        out[off + iz * 64] = c[iz];
        xs[iz * 64 + lane] = c[iz];
      }
    } else if (w < 3) {  // the neighbour's last (first) layer in x
      if (ix == (w == 1 ? 7 : 0)) {
#pragma unroll
        for (int iz = 0; iz < BS; ++iz) fc[w - 1][iz * 8 + iy] = c[iz];
      }
    } else if (w < 5) {
      if (iy == (w == 3 ? 7 : 0)) {
#pragma unroll
        for (int iz = 0; iz < BS; ++iz) fc[w - 1][iz * 8 + ix] = c[iz];
      }
    } else {
      fc[w - 1][lane] = w == 5 ? c[7] : c[0];
    }
  }
  __syncthreads();
  if (w < 4) {
    const double h = g.h[b];
    int none = 0;  // faces without a neighbour: the ghost is the cell itself
#pragma unroll
    for (int q = 0; q < 6; ++q) none |= (g.nbr[b * 6 + q] < 0 ? 1 : 0) << q;
    const bool origin = g.bmean_row == (long long)b * BLEN;
    double sum[3] = {0.0, 0.0, 0.0};  // sum of x, then the dots
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int iz = 2 * w + k, li = iz * 64 + lane;
      const double c0 = xs[li];
      auto side = [&](bool inside, int step, int face, int cell) {
        if (inside) return xs[li + step];
        return (none >> face) & 1 ? c0 : fc[face][cell];
      };
      const double xm = side(ix > 0, -1, 0, iz * 8 + iy), xp = side(ix < 7, 1, 1, iz * 8 + iy);
      const double ym = side(iy > 0, -8, 2, iz * 8 + ix), yp = side(iy < 7, 8, 3, iz * 8 + ix);
      const double zm = side(iz > 0, -64, 4, lane), zp = side(iz < 7, 64, 5, lane);
      double yy = h * ((((xm + xp) + (ym + yp)) + (zm + zp)) - 6.0 * c0);
      if (HELM) {
        const int dm = none & g.dmask;
        const int nd = (ix == 0 ? (dm & 1) : 0) + (ix == 7 ? ((dm >> 1) & 1) : 0) +
                       (iy == 0 ? ((dm >> 2) & 1) : 0) + (iy == 7 ? ((dm >> 3) & 1) : 0) +
                       (iz == 0 ? ((dm >> 4) & 1) : 0) + (iz == 7 ? ((dm >> 5) & 1) : 0);
        yy += (-(h * h * h) * g.helm_sigma - (double)(2 * nd) * h) * c0;
      }
      if (MODE == PREC_S) a[k] = sv[li];
      sum[0] += c0;
      if (origin && li == 0) {
        if (BM1) {  // the row is the sum over the grid, which the consumer adds
          part[(size_t)N * gridDim.x] = a[k];
          continue;
        }
        if (g.bmean == 3) yy = h * c0;  // row h I
      }
      y[own + iz * 64] = yy;
      sum[1] += a[k] * yy;
      sum[2] += yy * yy;
    }
    sum[0] *= h * h * h;
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const double t = wave_sum(sum[q + (BM1 ? 0 : 1)]);
      if (lane == 0) red[q][w] = t;
    }
  }
  __syncthreads();
  if (threadIdx.x < N) {
    const double* r = red[threadIdx.x];
    part[(size_t)b * N + threadIdx.x] = ((r[0] + r[1]) + r[2]) + r[3];
  }
}

template <typename T, int MODE, int FIN>
void launch_precond_dst_m(hipStream_t s, int nb, const T* h, T sigma,
                          const KrylovVectors<T>& v, SolverState* st, const FinArgs& f) {
  const int nwg = (nb + WG_THREADS / 64 - 1) / (WG_THREADS / 64);
  k_precond_dst<T, MODE, FIN><<<nwg, WG_THREADS, 0, s>>>(nb, h, sigma, v, st, f);
}

template <typename T>
void launch_precond_dst_t(hipStream_t s, int mode, int nb, const T* h, T sigma,
                          const KrylovVectors<T>& v, SolverState* st, int fin, const FinArgs& f) {
  if (mode == PREC_P && fin)
    launch_precond_dst_m<T, PREC_P, FIN_SUMS>(s, nb, h, sigma, v, st, f);
  else if (mode == PREC_P)
    launch_precond_dst_m<T, PREC_P, FIN_KERNEL>(s, nb, h, sigma, v, st, f);
  else if (mode == PREC_S && fin == FIN_ROW)
    launch_precond_dst_m<T, PREC_S, FIN_ROW>(s, nb, h, sigma, v, st, f);
  else if (mode == PREC_S && fin)
    launch_precond_dst_m<T, PREC_S, FIN_SUMS>(s, nb, h, sigma, v, st, f);
  else if (mode == PREC_S)
    launch_precond_dst_m<T, PREC_S, FIN_KERNEL>(s, nb, h, sigma, v, st, f);
  else
    launch_precond_dst_m<T, PREC_PLAIN, FIN_KERNEL>(s, nb, h, sigma, v, st, f);
}

// u* += the three solutions (AdvectionDiffusionImplicit.cpp:407-418), two
// cells (three 16-byte accesses) per thread; a null solution is 0.
__global__ __launch_bounds__(WG_THREADS) void k_diff_add(long long n, const double* __restrict__ x,
                                                         const double* __restrict__ y,
                                                         const double* __restrict__ z,
                                                         double* __restrict__ vel) {
  typedef double double2_t __attribute__((ext_vector_type(2)));
  const long long i = (long long)blockIdx.x * WG_THREADS + threadIdx.x;
  if (2 * i >= n) return;
  const double2_t zero = {0.0, 0.0};
  const double2_t a = x ? reinterpret_cast<const double2_t*>(x)[i] : zero;
  const double2_t b = y ? reinterpret_cast<const double2_t*>(y)[i] : zero;
  const double2_t c = z ? reinterpret_cast<const double2_t*>(z)[i] : zero;
  double2_t* __restrict__ v = reinterpret_cast<double2_t*>(vel) + 3 * i;
  v[0] += (double2_t){a.x, b.x};
  v[1] += (double2_t){c.x, a.y};
  v[2] += (double2_t){b.y, c.y};
}

}  // namespace

void launch_precond_dst(hipStream_t s, int mode, int nb, const double* h,
                        double sigma, const KrylovVectors<double>& v, SolverState* st, int fin,
                        const FinArgs& f) {
  launch_precond_dst_t<double>(s, mode, nb, h, sigma, v, st, fin, f);
}

void launch_precond_dst32(hipStream_t s, int mode, int nb, const float* h,
                          const KrylovVectors<float>& v, SolverState* st, int fin,
                          const FinArgs& f) {
  launch_precond_dst_t<float>(s, mode, nb, h, 0.0f, v, st, fin, f);
}

template <int MODE, int FIN>
static void launch_fused_m(hipStream_t s, const DevGrid<double>& g, const KrylovVectors<double>& v,
                           double* y, SolverState* st, const FinArgs& f, double* part) {
  if (g.helm)
    k_precond_spmv<MODE, FIN, false, true><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
  else if (g.bmean == 1 && g.bmean_row >= 0)
    k_precond_spmv<MODE, FIN, true, false><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
  else
    k_precond_spmv<MODE, FIN, false, false><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
}

void launch_precond_spmv64(hipStream_t s, int mode, const DevGrid<double>& g,
                           const KrylovVectors<double>& v, double* y, SolverState* st, int fin,
                           const FinArgs& f, double* part) {
  if (mode == PREC_P && fin) launch_fused_m<PREC_P, FIN_SUMS>(s, g, v, y, st, f, part);
  else if (mode == PREC_P) launch_fused_m<PREC_P, FIN_KERNEL>(s, g, v, y, st, f, part);
  else if (fin == FIN_ROW)
    k_precond_spmv<PREC_S, FIN_ROW, true, false><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
  else if (g.helm)
    k_precond_spmv<PREC_S, FIN_SUMS, false, true><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
  else
    k_precond_spmv<PREC_S, FIN_SUMS, false, false><<<g.nb, FUSE_T, 0, s>>>(g, v, y, st, f, part);
}

void launch_diffusion_add(hipStream_t s, long long n, const double* const x[3], double* vel) {
  const int nwg = (int)((n / 2 + WG_THREADS - 1) / WG_THREADS);
  k_diff_add<<<nwg, WG_THREADS, 0, s>>>(n, x[0], x[1], x[2], vel);
}

}  // namespace cup3d
