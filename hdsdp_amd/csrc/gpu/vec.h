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
    LZ_ALPHA = 4,
    LZ_NORM = 5,
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
void cg_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r);
// r = rhs - Mx and sc[CG_TRUE] = ||r||
void cg_true_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r, double *sc);

void lz_step(hipStream_t s, int n, int k, double *w, double *V, double *H, int ldh, double *v, double *sc,
             double *hist);
void lz_start(hipStream_t s, int n, const double *x, double *v, double *V);
void lz_comb(hipStream_t s, int n, int kp1, const double *V, const double *y, double *z);
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
