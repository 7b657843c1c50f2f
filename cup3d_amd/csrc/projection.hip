// The caller around the solve, on the device: the rhs of the pressure
// equation (KernelPressureRHS, source/operators/PressureProjection.cpp:96-199)
// and the pressure-gradient velocity update (KernelGradP :244-323 and
// :449-466), with the flux correction at coarse-fine faces, over Cubism's
// block layout (velocities [nb][8][8][8][3], scalars [nb][8][8][8]).
//
// Lab (ghost) values one cell outside a block, per face kind:
//   same level      the neighbour's cell (periodic wrap through the tables);
//   coarser         2/3 f_close - 1/5 f_far + 8/15 T(f_coarse), the fine ghost
//                   of the operator's interface interpolation (exact for
//                   quadratics; the Taylor value T as the SpMV evaluates it);
//   domain boundary velocity (BlockLabBC, Definitions.h:284-435): the normal
//                   component mirrored, ghost = -u, for walls and freespace;
//                   pressure (BlockLabNeumann3D): ghost = p;
//   finer           the coarse cell carries no face term of its own and gets
//                   the sum of the four fine cells' face terms instead, each
//                   with its own fine ghost (Cubism's flux correction).
// A face term is s fac (f_nb + f_c) for side s = -1 / +1, so the interior
// formula fac (f(x+h) - f(x-h)) is the sum of a cell's two face terms.
//
// One wavefront per block, as the SpMV: lane (ix, iy) walks its z column. A
// block of a vector field is 12 KiB of consecutive doubles: it is loaded as
// twelve 16-byte loads per lane and staged in the wavefront's LDS slice, from
// which every lane picks the components of its cell and its x/y neighbours;
// only the face cells of the neighbours are read with a stride. The gradient
// goes through the same slice the other way, so the velocity is updated with
// 16-byte accesses too. Bound by HBM (rhs: 3 vectors in, 1 out; update: 1 + 3
// in, 3 out). With one thread per cell (strided 8-byte loads, the interface
// code in every thread, its index arrays in scratch memory) the rhs took
// 1036 us and the update 827 us on the 30.2 M-cell grid (966 MB and 1.69 GB
// of vectors); now they take 231 us (4.2 TB/s) and 318 us (5.3 TB/s).

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels.h"
#include "krylov.h"

namespace cup3d {

namespace {

typedef double double2_t __attribute__((ext_vector_type(2)));

constexpr int VLEN = 3 * BLEN;       // doubles of one block of a vector field
constexpr int V2 = VLEN / (2 * 64);  // double2 per lane

// T of the four fine cells of a coarse cell: base + s1 a + s2 b + s1 s2 m, the
// terms of taylor_sum; get(o1, o2) reads the coarse face layer at tangential
// offsets from the cell.
struct TaylorTerms {
  double base, a, b, m;
};
template <typename F>
__device__ __forceinline__ TaylorTerms taylor_terms(F&& get, int k1, int k2) {
  const int o1 = k1 == TK_CEN ? -1 : (k1 == TK_BWD ? -2 : 0);
  const int o2 = k2 == TK_CEN ? -1 : (k2 == TK_BWD ? -2 : 0);
  const double p0 = get(o1, 0), p1 = get(o1 + 1, 0), p2 = get(o1 + 2, 0);
  const double q0 = get(0, o2), q1 = get(0, o2 + 1), q2 = get(0, o2 + 2);
  TaylorTerms t;
  t.base = get(0, 0) + 0.03125 * ((p0 + p2) + (q0 + q2)) - 0.0625 * (p1 + q1);
  const auto d1 = [](int k, double x0, double x1, double x2) {
    return k == TK_CEN ? 0.125 * (x2 - x0)
                       : (k == TK_BWD ? 0.125 * x0 - 0.5 * x1 + 0.375 * x2
                                      : 0.5 * x1 - 0.375 * x0 - 0.125 * x2);
  };
  t.a = d1(k1, p0, p1, p2);
  t.b = d1(k2, q0, q1, q2);
  const int m1a = k1 == TK_FWD ? 0 : -1, m1b = k1 == TK_BWD ? 0 : 1;
  const int m2a = k2 == TK_FWD ? 0 : -1, m2b = k2 == TK_BWD ? 0 : 1;
  const double w1 = k1 == TK_CEN ? 0.125 : 0.25, w2 = k2 == TK_CEN ? 0.125 : 0.25;
  t.m = w1 * w2 * ((get(m1b, m2b) - get(m1a, m2b)) - (get(m1b, m2a) - get(m1a, m2a)));
  return t;
}

// One coarse-fine face f of block b, evaluated by lane (t1, t2) = (lane & 7,
// lane >> 3) for its face cell, for component comp of an NC-component field F:
//   coarser neighbour  s c_own (G + f)          (this cell's own face term)
//   finer neighbours   s c_fine sum_q chi_q (G_q + f_q)   (the flux correction)
// s = -1 / +1 on the low / high side; own(cell) reads the staged block, pl is a
// 64-value plane of this wavefront, chi (may be null) the obstacle indicator.
template <int NC, typename Own>
__device__ __forceinline__ double iface_term(const double* __restrict__ F,
                                             const double* __restrict__ chi, Own&& own,
                                             double* pl, int f, int fk, int comp, int par,
                                             int lane, int nb0, int nbq, double c_own,
                                             double c_fine) {
  const int d = f >> 1;
  const bool minus = (f & 1) == 0;
  const int t1 = d == 0 ? 1 : (d == 1 ? 2 : 0), t2 = d == 0 ? 2 : (d == 1 ? 0 : 1);
  const int st1 = t1 == 0 ? 1 : (t1 == 1 ? 8 : 64), st2 = t2 == 0 ? 1 : (t2 == 1 ? 8 : 64);
  const int sd = d == 0 ? 1 : (d == 1 ? 8 : 64);
  const int u = lane & 7, v = lane >> 3;
  const int cl = (minus ? 0 : 7) * sd + u * st1 + v * st2;  // this lane's face cell
  const double sgn = minus ? -1.0 : 1.0;
  if (fk == FACE_COARSE) {
    pl[lane] = F[coarse_plane_index(f, nb0, lane) * NC + comp];
    wave_sync();
    const int c1 = (u >> 1) + (((par >> t1) & 1) ? BS / 2 : 0);
    const int c2 = (v >> 1) + (((par >> t2) & 1) ? BS / 2 : 0);
    const TaylorTerms t = taylor_terms([&](int o1, int o2) { return pl[(c2 + o2) * 8 + c1 + o1]; },
                                       taylor_kind(c1), taylor_kind(c2));
    const double s1 = (u & 1) ? 1.0 : -1.0, s2 = (v & 1) ? 1.0 : -1.0;
    const double T = t.base + s1 * t.a + s2 * t.b + s1 * s2 * t.m;
    const double close = own(cl), far = own(cl + (minus ? sd : -sd));
    return sgn * c_own * ((5.0 / 3.0) * close - 0.2 * far + (8.0 / 15.0) * T);
  }
  // the four fine cells behind this coarse cell, in the finer block of its
  // quadrant; their ghosts share this cell's Taylor expansion
  const size_t fo = (size_t)nbq * BLEN;
  const int lc = minus ? BS - 1 : 0, lf = minus ? BS - 2 : 1;
  double fc[4], ff[4], x4[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int f1 = (u & 3) * 2 + (q & 1), f2 = (v & 3) * 2 + (q >> 1);
    const size_t kc = fo + lc * sd + f1 * st1 + f2 * st2;
    fc[q] = F[kc * NC + comp];
    ff[q] = F[(fo + lf * sd + f1 * st1 + f2 * st2) * NC + comp];
    x4[q] = chi ? chi[kc] : 1.0;
  }
  const TaylorTerms t =
      taylor_terms([&](int o1, int o2) { return own(cl + o1 * st1 + o2 * st2); }, taylor_kind(u),
                   taylor_kind(v));
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double s1 = (q & 1) ? 1.0 : -1.0, s2 = (q >> 1) ? 1.0 : -1.0;
    const double T = t.base + s1 * t.a + s2 * t.b + s1 * s2 * t.m;
    acc += x4[q] * ((5.0 / 3.0) * fc[q] - 0.2 * ff[q] + (8.0 / 15.0) * T);
  }
  return sgn * c_fine * acc;
}

// The face term of lane (t1, t2) goes through the plane to the lane that owns
// the cell: acc[iz] += the term of face f at this lane's cells.
__device__ __forceinline__ void scatter_face(double* pl, int f, int lane, double term,
                                             double (&acc)[BS]) {
  const int d = f >> 1, ix = lane & 7, iy = lane >> 3;
  const bool minus = (f & 1) == 0;
  const int at = minus ? 0 : BS - 1;
  wave_sync();  // the plane's readers are done
  pl[lane] = term;
  wave_sync();
  if (d == 2) {  // (t1, t2) = (x, y): this lane's own cell
    if (minus) acc[0] += term;
    else acc[BS - 1] += term;
  } else if (d == 0 ? ix == at : iy == at) {
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) acc[iz] += d == 0 ? pl[iy + 8 * iz] : pl[iz + 8 * ix];
  }
  wave_sync();
}

// This wavefront's block b of a vector field, as consecutive 16-byte loads.
__device__ __forceinline__ void load_block(const double* __restrict__ F, size_t b, int lane,
                                           double2_t (&r)[V2]) {
  const double2_t* __restrict__ p = reinterpret_cast<const double2_t*>(F + b * VLEN);
#pragma unroll
  for (int k = 0; k < V2; ++k) r[k] = p[k * 64 + lane];
}

// A block is a workgroup of its own: its 12.5 KiB of LDS come free with it, not
// with the slowest of four (3-level AMR grid of 4440 blocks, with an obstacle: a
// call 50 -> 47 us). On the school grid's 59 012 blocks the reads bound it, 0.98 GB
// for 0.73 GB of velocity, the rest neighbours' faces no longer in the L2: 231 us
// (5.3 TB/s) either way. Storing the result past the caches takes 7 us less there,
// but the increment form, which reads it next, as much more.
// KernelPressureRHS: out = fac (uE - uW + vN - vS + wB - wF) - chi fac (the
// same of udef) + the finer faces' flux corrections, fac = h^2 / (2 dt).
template <bool IFACE, bool OBST>
__global__ __launch_bounds__(64) void k_pressure_rhs(DevGrid<double> g,
                                                     const double* __restrict__ vel,
                                                     const double* __restrict__ udef,
                                                     const double* __restrict__ chi, double dt,
                                                     double* __restrict__ out) {
  __shared__ double L[VLEN], pl[IFACE ? 64 : 1];
  const int lane = threadIdx.x, b = xcd_remap(blockIdx.x, gridDim.x);
  const int ix = lane & 7, iy = lane >> 3;
  const size_t off = (size_t)b * BLEN;
  int meta = 0;
  if (IFACE) meta = g.bmeta[(size_t)b * 32 + (lane & 31)];
  const int* nb6 = g.nbr + b * 6;
  const int nx = ix == 0 ? nb6[0] : (ix == BS - 1 ? nb6[1] : -1);
  const int ny = iy == 0 ? nb6[2] : (iy == BS - 1 ? nb6[3] : -1);
  const int nzm = nb6[4], nzp = nb6[5];
  const double h = g.h[b], fac = 0.5 * h * h / dt;
  const double hf = 0.5 * h, fac_f = 0.5 * hf * hf / dt;
  double acc[BS], cv[BS];
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) {
    acc[iz] = 0.0;
    cv[iz] = OBST ? chi[off + iz * 64 + lane] : 0.0;
  }
#pragma unroll 1
  for (int field = 0; field < (OBST ? 2 : 1); ++field) {
    const double* __restrict__ F = OBST && field ? udef : vel;
    double2_t r[V2];
    load_block(F, b, lane, r);
    // face cells of the same-level neighbours (each component along its axis)
    double hx[BS], hy[BS], zlo = 0.0, zhi = 0.0;
    if (nx >= 0) {
      const double* p = F + 3 * ((size_t)nx * BLEN + iy * 8 + (ix == 0 ? BS - 1 : 0));
#pragma unroll
      for (int iz = 0; iz < BS; ++iz) hx[iz] = p[3 * 64 * iz];
    }
    if (ny >= 0) {
      const double* p = F + 3 * ((size_t)ny * BLEN + (iy == 0 ? BS - 1 : 0) * 8 + ix) + 1;
#pragma unroll
      for (int iz = 0; iz < BS; ++iz) hy[iz] = p[3 * 64 * iz];
    }
    if (nzm >= 0) zlo = F[3 * ((size_t)nzm * BLEN + 7 * 64 + lane) + 2];
    if (nzp >= 0) zhi = F[3 * ((size_t)nzp * BLEN + lane) + 2];
    wave_sync();  // the slice's readers of the previous field are done
#pragma unroll
    for (int k = 0; k < V2; ++k) *reinterpret_cast<double2_t*>(&L[2 * (k * 64 + lane)]) = r[k];
    wave_sync();
    double wc[BS];
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) wc[iz] = L[3 * (iz * 64 + lane) + 2];
#pragma unroll
    for (int iz = 0; iz < BS; ++iz) {
      const int c = 3 * (iz * 64 + lane);
      // the ghost of a face without a same-level neighbour is -own: no face
      // term (domain boundary), or the one iface_term adds
      const double u = L[c], v = L[c + 1];
      const double xo = nx >= 0 ? hx[iz] : -u, yo = ny >= 0 ? hy[iz] : -v;
      const double xm = ix > 0 ? L[c - (ix > 0 ? 3 : 0)] : xo;
      const double xp = ix < 7 ? L[c + (ix < 7 ? 3 : 0)] : xo;
      const double ym = iy > 0 ? L[c + 1 - (iy > 0 ? 24 : 0)] : yo;
      const double yp = iy < 7 ? L[c + 1 + (iy < 7 ? 24 : 0)] : yo;
      const double zm = iz > 0 ? wc[iz > 0 ? iz - 1 : 0] : (nzm >= 0 ? zlo : -wc[0]);
      const double zp = iz < 7 ? wc[iz < 7 ? iz + 1 : 7] : (nzp >= 0 ? zhi : -wc[7]);
      const double s = xp - xm + yp - ym + zp - zm;
      acc[iz] += (OBST && field ? -cv[iz] * fac : fac) * s;
    }
    if (IFACE) {
      const int par = __builtin_amdgcn_readlane(meta, 30);
      const int fq = (ix >= BS / 2 ? 1 : 0) + (iy >= BS / 2 ? 2 : 0);
#pragma unroll 1
      for (int f = 0; f < 6; ++f) {
        const int fk = __builtin_amdgcn_readlane(meta, 24 + f);
        if (fk < FACE_COARSE) continue;
        const int d = f >> 1;
        double c_own = fac, c_fine = fac_f;
        if (OBST && field) {  // -chi of this lane's face cell, and of its fine cells
          const int fc = (f & 1) ? BS - 1 : 0;
          const int cl = d == 0 ? fc + 8 * ix + 64 * iy
                                : (d == 1 ? 8 * fc + 64 * ix + iy : 64 * fc + ix + 8 * iy);
          c_own = -fac * chi[off + cl];
          c_fine = -fac_f;
        }
        const double term = iface_term<3>(
            F, OBST && field ? chi : nullptr, [&](int cell) { return L[3 * cell + d]; }, pl, f,
            fk, d, par, lane, __builtin_amdgcn_readlane(meta, 4 * f), __shfl(meta, 4 * f + fq, 64),
            c_own, c_fine);
        scatter_face(pl, f, lane, term, acc);
      }
    }
  }
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) out[off + iz * 64 + lane] = acc[iz];
}

// KernelGradP and the velocity update: o = -dt h^2 / 2 (p(x+h) - p(x-h)) per
// component plus the finer faces' flux corrections; vel += o / h^3.
template <bool IFACE>
__global__ __launch_bounds__(WG_THREADS) void k_grad_p_update(DevGrid<double> g,
                                                              const double* __restrict__ p,
                                                              double dt,
                                                              double* __restrict__ vel) {
  __shared__ double Ls[WG_THREADS / 64][VLEN];  // the block of p, then its gradient
  __shared__ double pls[IFACE ? WG_THREADS / 64 : 1][IFACE ? 64 : 1];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = xcd_remap(blockIdx.x, gridDim.x) * (WG_THREADS / 64) + w;
  if (b >= g.nb) return;  // no workgroup barrier below: only this wavefront's slice
  const int ix = lane & 7, iy = lane >> 3;
  const size_t off = (size_t)b * BLEN;
  double* L = Ls[w];
  int meta = 0;
  if (IFACE) meta = g.bmeta[(size_t)b * 32 + (lane & 31)];
  const int* nb6 = g.nbr + b * 6;
  const int nx = ix == 0 ? nb6[0] : (ix == BS - 1 ? nb6[1] : -1);
  const int ny = iy == 0 ? nb6[2] : (iy == BS - 1 ? nb6[3] : -1);
  const int nzm = nb6[4], nzp = nb6[5];
  const double h = g.h[b], fac = -0.5 * dt * h * h;
  const double hf = 0.5 * h, fac_f = -0.5 * dt * hf * hf;
  const double inv = 1.0 / (h * h * h);
  double col[BS], hx[BS], hy[BS], zlo = 0.0, zhi = 0.0;
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) col[iz] = p[off + iz * 64 + lane];
  const double* px = p + (nx >= 0 ? (size_t)nx * BLEN + iy * 8 + (ix == 0 ? BS - 1 : 0) : off + lane);
  const double* py = p + (ny >= 0 ? (size_t)ny * BLEN + (iy == 0 ? BS - 1 : 0) * 8 + ix : off + lane);
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) {
    hx[iz] = px[iz * 64];
    hy[iz] = py[iz * 64];
  }
  zlo = p[nzm >= 0 ? (size_t)nzm * BLEN + 7 * 64 + lane : off + lane];
  zhi = p[nzp >= 0 ? (size_t)nzp * BLEN + lane : off + 7 * 64 + lane];
  double2_t r[V2];
  load_block(vel, b, lane, r);
  // the ghost of a face without a same-level neighbour is the cell itself
  // (domain boundary: zero gradient) or, at coarse-fine faces, minus the
  // cell: no face term but the one iface_term adds
  double sx = 1.0, sy = 1.0, szm = 1.0, szp = 1.0;
  if (IFACE) {
    int cf = 0;
#pragma unroll
    for (int f = 0; f < 6; ++f)
      cf |= (__builtin_amdgcn_readlane(meta, 24 + f) >= FACE_COARSE ? 1 : 0) << f;
    sx = (ix == 0 && (cf & 1)) || (ix == BS - 1 && (cf & 2)) ? -1.0 : 1.0;
    sy = (iy == 0 && (cf & 4)) || (iy == BS - 1 && (cf & 8)) ? -1.0 : 1.0;
    szm = (cf & 16) ? -1.0 : 1.0;
    szp = (cf & 32) ? -1.0 : 1.0;
  }
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) L[iz * 64 + lane] = col[iz];
  wave_sync();
  double gx[BS], gy[BS], gz[BS];
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) {
    const int c = iz * 64 + lane;
    const double xm = ix > 0 ? L[c - (ix > 0 ? 1 : 0)] : sx * hx[iz];
    const double xp = ix < 7 ? L[c + (ix < 7 ? 1 : 0)] : sx * hx[iz];
    const double ym = iy > 0 ? L[c - (iy > 0 ? 8 : 0)] : sy * hy[iz];
    const double yp = iy < 7 ? L[c + (iy < 7 ? 8 : 0)] : sy * hy[iz];
    const double zm = iz > 0 ? col[iz > 0 ? iz - 1 : 0] : szm * zlo;
    const double zp = iz < 7 ? col[iz < 7 ? iz + 1 : 7] : szp * zhi;
    gx[iz] = fac * (xp - xm);
    gy[iz] = fac * (yp - ym);
    gz[iz] = fac * (zp - zm);
  }
  if (IFACE) {
    const int par = __builtin_amdgcn_readlane(meta, 30);
    const int fq = (ix >= BS / 2 ? 1 : 0) + (iy >= BS / 2 ? 2 : 0);
#pragma unroll 1
    for (int f = 0; f < 6; ++f) {
      const int fk = __builtin_amdgcn_readlane(meta, 24 + f);
      if (fk < FACE_COARSE) continue;
      const double term = iface_term<1>(
          p, nullptr, [&](int cell) { return L[cell]; }, pls[w], f, fk, 0, par, lane,
          __builtin_amdgcn_readlane(meta, 4 * f), __shfl(meta, 4 * f + fq, 64), fac, fac_f);
      if (f < 2) scatter_face(pls[w], f, lane, term, gx);
      else if (f < 4) scatter_face(pls[w], f, lane, term, gy);
      else scatter_face(pls[w], f, lane, term, gz);
    }
  }
  wave_sync();  // the readers of p's block are done
#pragma unroll
  for (int iz = 0; iz < BS; ++iz) {
    const int c = 3 * (iz * 64 + lane);
    L[c] = inv * gx[iz];
    L[c + 1] = inv * gy[iz];
    L[c + 2] = inv * gz[iz];
  }
  wave_sync();
  double2_t* __restrict__ o = reinterpret_cast<double2_t*>(vel + (size_t)b * VLEN);
#pragma unroll
  for (int k = 0; k < V2; ++k)
    o[k * 64 + lane] = r[k] + *reinterpret_cast<const double2_t*>(&L[2 * (k * 64 + lane)]);
}

}  // namespace

void launch_pressure_rhs(hipStream_t s, const DevGrid<double>& g, const double* vel,
                         const double* udef, const double* chi, double dt, double* out) {
  if (g.has_iface && udef)
    k_pressure_rhs<true, true><<<g.nb, 64, 0, s>>>(g, vel, udef, chi, dt, out);
  else if (g.has_iface)
    k_pressure_rhs<true, false><<<g.nb, 64, 0, s>>>(g, vel, udef, chi, dt, out);
  else if (udef)
    k_pressure_rhs<false, true><<<g.nb, 64, 0, s>>>(g, vel, udef, chi, dt, out);
  else
    k_pressure_rhs<false, false><<<g.nb, 64, 0, s>>>(g, vel, udef, chi, dt, out);
}

void launch_grad_p_update(hipStream_t s, const DevGrid<double>& g, const double* p, double dt,
                          double* vel) {
  const int nwg = (g.nb + WG_THREADS / 64 - 1) / (WG_THREADS / 64);
  if (g.has_iface) k_grad_p_update<true><<<nwg, WG_THREADS, 0, s>>>(g, p, dt, vel);
  else k_grad_p_update<false><<<nwg, WG_THREADS, 0, s>>>(g, p, dt, vel);
}

}  // namespace cup3d
