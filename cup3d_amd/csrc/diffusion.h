// Implicit diffusion kernels (diffusion.hip): the DST block preconditioner
// and the velocity update of a diffusion step.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "kernels.h"
#include "poisson_internal.h"

namespace cup3d {

// mode PREC_P / PREC_S / PREC_PLAIN; h per block, sigma = 1 / (nu dt); fin and
// f: whether and from where the kernel takes its scalars' sums.
void launch_precond_dst(hipStream_t s, int mode, int nb, const double* h,
                        double sigma, const KrylovVectors<double>& v, SolverState* st,
                        int fin = FIN_KERNEL, const FinArgs& f = FinArgs());
// The same in FP32 for the mixed forms' inner solve (sigma = 0: the pressure
// equation's block inverse h^-1 P_inv).
void launch_precond_dst32(hipStream_t s, int mode, int nb, const float* h,
                          const KrylovVectors<float>& v, SolverState* st,
                          int fin = FIN_KERNEL, const FinArgs& f = FinArgs());
// vel[:, c] += x[c] (null: 0) for the three components of an [n][3] field.
void launch_diffusion_add(hipStream_t s, long long n, const double* const x[3], double* vel);


// K1 and K2 (PREC_P: v.nu and v.p to v.pw and y) or K3 and K4 (PREC_S: v.r and
// v.nu to v.s and y) in one kernel, on grids for which fused_blocks() holds; the
// outputs overlap none of the inputs. part: g.nb sums of up to three values and one
// word, other than f.part. PREC_S takes its scalars from the sums (fin is not
// FIN_KERNEL).
void launch_precond_spmv64(hipStream_t s, int mode, const DevGrid<double>& g,
                           const KrylovVectors<double>& v, double* y, SolverState* st, int fin,
                           const FinArgs& f, double* part);

}  // namespace cup3d
