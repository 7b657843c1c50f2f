// Kernel launch interface of libcup3d_poisson (host side).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "poisson_internal.h"

namespace cup3d {

// PLAIN  y = A x                       INIT   c = c2 = a - A x, |A x|^2, |c|^2
//                                             (y: room for bMean 2)
// DOT1   y = A x, (a, y), a from c     DOT2   y = A x, (a, y), (y, y)
//        after a restart (c may be null)
// RESID  c = a - A x, |c|^2
// START  -h^3 sigma a - A x into g.xo[0 .. 2] and its norms, for the three
//        components of the [n][3] fields x and a (Helmholtz grids)
// NET    c = a - A x, |c / h|^2, |x|^2 (bMean 0)
// FINAL  |a - A x|^2 of the best iterate x (g.xo, the state), copied to y (may be null)
enum SpmvMode {
  SPMV_PLAIN = 0, SPMV_INIT = 1, SPMV_DOT1 = 2, SPMV_DOT2 = 3, SPMV_RESID = 4, SPMV_START = 5,
  SPMV_FINAL = 6, SPMV_NET = 7
};
enum PrecMode { PREC_PLAIN = 0, PREC_P = 1, PREC_S = 2 };

// Where the scalars of an iteration are computed: by finalize kernels, or by
// the kernels that use them (krylov.h), with the bMean = 1 row or without.
enum Fin { FIN_KERNEL = 0, FIN_SUMS = 1, FIN_ROW = 2 };
struct FinArgs {
  const double* part = nullptr;
  int nparts = 0;
  long long row = -1;
  // K1: where the host follows the iterations (both pinned, null: nowhere). The
  // word takes 2 * iterations done, + 1 when that ended the solve; the state is
  // there before such a word.
  unsigned long long* prog = nullptr;
  SolverState* hst = nullptr;
};
constexpr int FIN_MAX_BLOCKS = 8192;

// The way a grid's iterations take (bMean = 2 needs its sum before the
// epilogue of the SpMV, so it keeps the kernels).
inline int fin_mode(int nb, int bmean, long long row) {
  if (nb > FIN_MAX_BLOCKS || bmean == 2) return FIN_KERNEL;
  return bmean == 1 && row >= 0 ? FIN_ROW : FIN_SUMS;
}
// The sums of K5 lie behind those of the SpMVs, which K5 still reads.
inline double* k5_part(double* part, int nb) { return part + 4 * (size_t)((nb + 3) / 4 + 8); }
// Grids whose FP64 iterations take three kernels instead of five
// (launch_precond_spmv64): one level, and a workgroup a CU at most. Ten iterations
// with five kernels and with three: 64 blocks 320 -> 275 us, 128 327 -> 285, 256
// 331 -> 304; past one workgroup a CU the seven-fold work tells, 384 blocks 343 ->
// 365 us, 1024 397 -> 510.
constexpr int FUSE_MAX_BLOCKS = 256;
constexpr int FUSE_VECTORS = 3;  // second vectors of p and nu, one for s
inline bool fused_blocks(int nb, bool has_iface, int fin) {
  return nb <= FUSE_MAX_BLOCKS && !has_iface && fin != FIN_KERNEL;
}
// Their sums, of the first product (which 0) and the second: up to three values
// a block and one word, behind all others.
inline double* fused_part(double* part, int nb, int which) {
  return part + 16 * (size_t)((nb + 3) / 4 + 8) + which * (size_t)(3 * nb + 8);
}
// Behind both, those of SPMV_START: (nb + 3) / 4 per component, kept until each
// component's solve.
inline double* start_part(double* part, int nb) { return part + 8 * (size_t)((nb + 3) / 4 + 8); }
// Copies of the solver state (krylov.h): st[0] is the one that counts between
// batches of iterations. hst, where a launch takes it: the host's pinned copy,
// written by the finalize kernel.
constexpr int STATE_COPIES = 3;

// The state starts as `init`, with ||b|| and the absolute tolerance. x may be x0, and
// the rhs may overlap either.
void launch_getvec64(hipStream_t s, long long n, long long zero_row, const double* rhs,
                     const double* x0, double* b, double* x, const SolverState& init,
                     SolverState* st, double* part, double tol_b);
// The same and the first iteration's scalars for x0 = 0, where b is the initial
// residual. Returns b: rhs itself, or its copy in `b` where the bMean row is zeroed
// or the rhs overlaps x, which takes the solution (30.2 M cells: 48 us to sum it
// against 158 us with copies to b and r and a cleared x).
const double* launch_start_zero64(hipStream_t s, int nb, long long zero_row, const double* rhs,
                                  const double* x, double* b, const SolverState& init,
                                  SolverState* st, SolverState* hst, double* part, double tol_b);
// The scalars of one component of SPMV_START (nb blocks, its partial sums).
void launch_start_fin(hipStream_t s, int nb, const SolverState& init, SolverState* st,
                      SolverState* hst, const double* part, double tol_b);
// part null (SPMV_PLAIN and SPMV_RESID on a grid with bMean 0 or 3, SPMV_FINAL for
// its copy): no sums are taken.
void launch_spmv64(hipStream_t s, int mode, const DevGrid<double>& g, const double* x, double* y,
                   const double* a, double* c, double* c2, SolverState* st, double* part,
                   bool fin = true, SolverState* hst = nullptr);
// K5; returns its number of partials. last: with its finalize kernel. sums: where
// those of K4 are (null: at part, a value per four blocks).
int launch_update64(hipStream_t s, const DevGrid<double>& g, const KrylovVectors<double>& v,
                    SolverState* st, double* part, int fin = FIN_KERNEL, bool last = true,
                    SolverState* hst = nullptr, unsigned long long* prog = nullptr,
                    const FinArgs* sums = nullptr);

// The caller around the solve (projection.hip): the rhs of the pressure
// equation from the velocity (and an obstacle's udef / chi, both or neither
// null), and the pressure-gradient update of the velocity ([n][3] doubles).
void launch_pressure_rhs(hipStream_t s, const DevGrid<double>& g, const double* vel,
                         const double* udef, const double* chi, double dt, double* out);
void launch_grad_p_update(hipStream_t s, const DevGrid<double>& g, const double* p, double dt,
                          double* vel);

// x -= the volume-weighted mean of x (h3 per block, inv_vol = 1 / sum 512 h^3);
// the weighted sum is left in host[0] (pinned); wsum: a word of scratch.
void launch_remove_mean(hipStream_t s, long long n, double* x, const double* h3, double inv_vol,
                        double* part, double* wsum, double* host);
// b = a over n4 float4 (the copy-rate probe of the diagnostics).
void launch_stream_copy(hipStream_t s, long long n4, const void* a, void* b);
// b = a over n4 16-byte words, one of them pinned host memory.
void launch_host_copy(hipStream_t s, long long n4, const void* a, void* b);

// Warm start from several guesses (device vectors of n doubles).
constexpr int HIST_MAX = 8;                // differences of previous pressures
constexpr int GUESS_MAXV = HIST_MAX + 2;   // r0 + the history directions + the net's
struct GuessVecs {
  const double* v[GUESS_MAXV];
};
// d = a - b, and d[row] = 0 when row >= 0 (the bMean = 1 / 3 cell that getVec
// zeroes): one direction of the warm start;
void launch_guess_direction(hipStream_t s, long long n, const double* a, const double* b,
                            long long row, double* d);
// x[row] = 0 (nothing for row < 0): the bMean = 1 / 3 cell that getVec zeroes;
void launch_zero_cell(hipStream_t s, double* x, long long row);
// dots = the upper triangle of the Gram matrix of r.v[0 .. nv), row by row,
// GUESS_MAXV (GUESS_MAXV + 1) / 2 values (those of absent vectors 0), in a
// fixed order; part holds that many partials per 2048 cells;
void launch_guess_gram(hipStream_t s, long long n, const GuessVecs& r, int nv, double* part,
                       double* dots);
// x = x0 + sum_{k < m} gt[k] (h[k-1] - h[k]) + gnet (pred - x0), h[-1] = x0,
// and x[row] = x0[row] (row >= 0); pred is not read when gnet = 0.
void launch_guess_blend(hipStream_t s, long long n, const double* x0, const GuessVecs& h,
                        const double* gt, int m, const double* pred, double gnet, long long row,
                        double* x);

}  // namespace cup3d
