// vec.h -- vector kernels of the Schur CG and the Lanczos step length.
#pragma once

#include "dev_common.h"

namespace hdk {

// slots of the device scalar array read back by the host
enum {
    CG_RNORM = 0,
    CG_BNORM = 1,
    CG_RZ = 2,
    CG_ALPHA = 3,
    LZ_R1 = 6,
    LZ_R2 = 7,
    SC_LOGDET = 8,
    SC_AUX = 9,
    CG_TRUE = 11,
    CG_TOL = 12,
    CG_STOP = 13,  // why the Jacobi iteration ended (CgStop), 0 while it runs
    CG_ITER = 14,  // iteration it ended at
    SC_SLOTS = 16
};

// CG_STOP values: converged; no progress (above a hundredth of the start after 20
// iterations); not a number; right-hand side below the tolerance
enum CgStop { CG_RUNNING = 0, CG_CONVERGED = 1, CG_STALLED = 2, CG_NAN = 3, CG_TINY = 4 };

void cg_start(hipStream_t s, int m, const double *rhs, double *r, double *x, double *sc);
void cg_jacobi(hipStream_t s, int m, const double *r, const double *jac, double *z, double *p);
void cg_step1(hipStream_t s, int m, const double *z, const double *r, const double *p, const double *Mp, double *x,
              double *rn, double *sc);
void cg_step2(hipStream_t s, int m, const double *rn, const double *z, double *p, double *r, double *sc);
// The Jacobi-preconditioned iteration with its decisions on the device, so that the host
// queues several iterations between two looks at them; once sc[CG_STOP] is set, the
// remaining ones leave x as it is.  cgj_start: r = rhs, x = 0, z = p = r / jac, the norm and
// the tolerance; cgj_iter: cg_step1, cg_jacobi and cg_step2 of iteration iter in one launch;
// cgj_half: cg_step1 alone (the iteration that restarts from the true residual).  The
// scalars go to sc and, where report is not null, to report (host memory the device can write).
void cgj_start(hipStream_t s, int m, const double *rhs, const double *jac, double relTol, double absTol, double *r,
               double *x, double *z, double *p, double *sc);
void cgj_iter(hipStream_t s, int m, int iter, const double *jac, const double *Mp, double *x, double *r, double *z,
              double *p, double *sc, double *report);
void cgj_half(hipStream_t s, int m, const double *z, const double *r, const double *p, const double *Mp, double *x,
              double *sc);
// The whole Jacobi CG of a system of m <= CGS_MAX rows in one launch: M m x m (ldm, both
// triangles), rhs in device or device-readable host memory (copied to crhs), at most
// maxIter iterations with a restart from the true residual at iter % restart == 5.  The
// scalars of cgj_iter go to report (CG_ITER: maxIter when it ran out), the solution to x
// and xHost (both written on every exit but CG_TINY).
constexpr int CGS_MAX = 256;
void cg_small(hipStream_t s, int m, const double *M, long ldm, const double *rhs, const double *jac, double relTol,
              double absTol, int maxIter, int restart, double *crhs, double *x, double *xHost, double *report);
void cg_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r);
// r = rhs - Mx and sc[CG_TRUE] = ||r||
void cg_true_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r, double *sc);

// combination coefficients of a Krylov basis, passed by value
constexpr int LZ_MAX = 30;
struct LzCoef {
    double y[LZ_MAX + 1];
};
// Step k of Lanczos on w: V_{k + 1}, v and the norm in H (zeros when the norm is 0), and
// (alpha_k, norm_k) in hist (host memory the device can write).
void lz_step(hipStream_t s, int n, int k, double *w, double *V, double *H, int ldh, double *v, double *hist);
// lz_step for n <= LZF_MAX without its v, and y = Li^T V_{k + 1} for the lower-triangular Li
// (n x n) in the same launch; w is left as it is
constexpr int LZF_MAX = 2048;
void lz_step_product(hipStream_t s, int n, int k, const double *w, double *V, double *H, int ldh, double *hist,
                     const double *Li, double *y);
// v = V_0 = x / ||x|| with x = x0, or x0 + pert where pert is not null
void lz_start(hipStream_t s, int n, const double *x0, const double *pert, double *v, double *V);
void lz_comb(hipStream_t s, int n, int kp1, const double *V, const LzCoef &y, double *z);
// n <= LZS_MAX: one workgroup runs the start (k0 = 0), the products L^-1 (-D) L^-T v and the
// steps k0 .. k1 - 1 in one launch, ...
constexpr int LZS_MAX = 160;
void lz_small_steps(hipStream_t s, int n, int k0, int k1, const double *x0, const double *pert, const double *Li,
                    const double *LiT, const double *D, double *V, double *H, int ldh, double *hist);
// ... and the two residuals of the step bound in another: with z = V y1, warm = Op z,
// report[LZ_R1] = ||Op z - e1 z|| and the same of V y2 in report[LZ_R2].
void lz_small_bound(hipStream_t s, int n, int kp1, double e1, const LzCoef &y1, const LzCoef &y2, const double *Li,
                    const double *LiT, const double *D, const double *V, double *warm, double *report);
void axpy_norm(hipStream_t s, int n, double a, const double *x, double *y, double *sc, int slot);

void axpy(hipStream_t s, long n, double a, const double *x, double *y);
void regularize(hipStream_t s, int m, double *M, long ldm, double r);
void get_diag(hipStream_t s, int m, const double *M, long ldm, double *d);
void f2d(hipStream_t s, long n, const float *x, double *y);
// y = x * sc (elementwise, with the precision conversion)
void f2d_scaled(hipStream_t s, long n, const float *x, const double *sc, double *y);
void d2f_scaled(hipStream_t s, long n, const double *x, const double *sc, float *y);
// sc[i] = 1 / sqrt(M_ii) (1 where M_ii <= 0)
void jacobi_scale(hipStream_t s, int m, const double *M, long ldm, double *sc);
void d2f(hipStream_t s, long n, const double *x, float *y);
// coef[0] = 0, coef[i + 1] = x[i] (coefficients of sum_i x_i A_i for the buffer assembly)
void shift_coef(hipStream_t s, int m, const double *x, double *coef);
// y[i] += (M_ii - ref[i]) x[i]
void diag_delta_axpy(hipStream_t s, int m, const double *M, long ldm, const double *ref, const double *x, double *y);

}  // namespace hdk
