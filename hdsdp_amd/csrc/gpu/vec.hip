// vec.hip -- m- and n-vector work of the Schur CG and the Lanczos step length.
//
// Vectors here have at most a few ten thousand entries, so each fused step
// runs in one workgroup of 1024 threads: the reductions are done in a fixed
// order (deterministic run to run) and no grid-wide synchronisation is needed.
// Scalars that the host controls on are written to a small device array that
// the host reads back once per step.
#include "vec.h"

#include <type_traits>

namespace hdk {

// Sum over a workgroup of 1024 threads, in every thread: each wave's tree sum, then the
// sixteen of them in order (every thread adds them up itself: one barrier per sum).  Two
// sums in a row use different halves B of red (32 doubles).
template <int B>
__device__ inline double block_sum(double v, double *red) {
    v = wave_tree_sum(v);
    if ((threadIdx.x & 63) == 0) red[16 * B + (threadIdx.x >> 6)] = v;
    __syncthreads();
    double t[16], total = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) t[w] = red[16 * B + w];
#pragma unroll
    for (int w = 0; w < 16; ++w) total += t[w];
    return total;
}

// ---- conjugate gradient (linalg/hdsdp_linsolver.c:855-997) -----------------

// r = rhs, x = 0, sc[CG_RNORM] = sc[CG_BNORM] = ||rhs||
__global__ __launch_bounds__(1024) void cg_start_kernel(int m, const double *rhs, double *r, double *x, double *sc) {
    __shared__ double red[32];
    double acc = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        double v = rhs[i];
        r[i] = v;
        x[i] = 0.0;
        acc += v * v;
    }
    double nrm = sqrt(block_sum<0>(acc, red));
    if (threadIdx.x == 0) {
        sc[CG_RNORM] = nrm;
        sc[CG_BNORM] = nrm;
    }
}

// z = r / jacobi (jacobi != NULL) else z = r; optional copy p = z
__global__ __launch_bounds__(1024) void cg_jacobi_kernel(int m, const double *r, const double *jac, double *z, double *p) {
    for (int i = threadIdx.x + blockIdx.x * blockDim.x; i < m; i += blockDim.x * gridDim.x) {
        double v = jac ? r[i] / jac[i] : r[i];
        z[i] = v;
        if (p) p[i] = v;
    }
}

// rz = z.r; pMp = p.Mp; alpha = rz / pMp; x += alpha p; rn = r - alpha Mp; sc[CG_RNORM] = ||rn||:
// the host decides on it before the preconditioner and the product of a next step
__global__ __launch_bounds__(1024) void cg_step1_kernel(int m, const double *z, const double *r, const double *p,
                                                        const double *Mp, double *x, double *rn, double *sc) {
    __shared__ double red[32];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        a += z[i] * r[i];
        b += p[i] * Mp[i];
    }
    double rz = block_sum<0>(a, red);
    double pMp = block_sum<1>(b, red);
    double alpha = rz / pMp;
    double c = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        x[i] += alpha * p[i];
        const double v = r[i] - alpha * Mp[i];
        rn[i] = v;
        c += v * v;
    }
    const double nrm = sqrt(block_sum<0>(c, red));
    if (threadIdx.x == 0) {
        sc[CG_RZ] = rz;
        sc[CG_ALPHA] = alpha;
        sc[CG_RNORM] = nrm;
    }
}

// beta = rn.z / rz; p = z + beta p; r = rn
__global__ __launch_bounds__(1024) void cg_step2_kernel(int m, const double *rn, const double *z, double *p, double *r,
                                                        double *sc) {
    __shared__ double red[32];
    double a = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) a += rn[i] * z[i];
    double beta = block_sum<0>(a, red) / sc[CG_RZ];
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        p[i] = z[i] + beta * p[i];
        r[i] = rn[i];
    }
}

// r = rhs - Mx (Mx precomputed)
__global__ void cg_residual_kernel(int m, const double *rhs, const double *Mx, double *r) {
    for (int i = threadIdx.x + blockIdx.x * blockDim.x; i < m; i += blockDim.x * gridDim.x) r[i] = rhs[i] - Mx[i];
}

__global__ __launch_bounds__(1024) void cg_true_residual_kernel(int m, const double *rhs, const double *Mx, double *r,
                                                                double *sc) {
    __shared__ double red[32];
    double acc = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        const double v = rhs[i] - Mx[i];
        r[i] = v;
        acc += v * v;
    }
    const double nrm = sqrt(block_sum<0>(acc, red));
    if (threadIdx.x == 0) sc[CG_TRUE] = nrm;
}

void cg_true_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r, double *sc) {
    cg_true_residual_kernel<<<1, 1024, 0, s>>>(m, rhs, Mx, r, sc);
}

void cg_start(hipStream_t s, int m, const double *rhs, double *r, double *x, double *sc) {
    cg_start_kernel<<<1, 1024, 0, s>>>(m, rhs, r, x, sc);
}
void cg_jacobi(hipStream_t s, int m, const double *r, const double *jac, double *z, double *p) {
    cg_jacobi_kernel<<<(m + 1023) / 1024, 1024, 0, s>>>(m, r, jac, z, p);
}
void cg_step1(hipStream_t s, int m, const double *z, const double *r, const double *p, const double *Mp, double *x,
              double *rn, double *sc) {
    cg_step1_kernel<<<1, 1024, 0, s>>>(m, z, r, p, Mp, x, rn, sc);
}
void cg_step2(hipStream_t s, int m, const double *rn, const double *z, double *p, double *r, double *sc) {
    cg_step2_kernel<<<1, 1024, 0, s>>>(m, rn, z, p, r, sc);
}
void cg_residual(hipStream_t s, int m, const double *rhs, const double *Mx, double *r) {
    cg_residual_kernel<<<(m + 1023) / 1024, 1024, 0, s>>>(m, rhs, Mx, r);
}

// The Jacobi iteration on small systems is bound by launches and host round trips: four
// launches, a copy and a synchronisation per iteration took 45 us at m = 368, of which
// the arithmetic is under 5.  One launch per iteration beside the product with M, and
// a host look every few iterations, take 12.  Same statements and reduction orders
// as the separate kernels.
__global__ __launch_bounds__(1024) void cgj_start_kernel(int m, const double *rhs, const double *jac, double relTol,
                                                         double absTol, double *r, double *x, double *z, double *p,
                                                         double *sc) {
    __shared__ double red[32];
    double acc = 0.0;
    for (int i = threadIdx.x; i < m; i += blockDim.x) {
        const double v = rhs[i], t = v / jac[i];
        r[i] = v;
        x[i] = 0.0;
        z[i] = t;
        p[i] = t;
        acc += v * v;
    }
    const double nrm = sqrt(block_sum<0>(acc, red));
    if (threadIdx.x == 0) {
        const double tol = fmax(fmin(absTol, nrm * relTol), 0.1 * absTol);
        sc[CG_RNORM] = nrm;
        sc[CG_BNORM] = nrm;
        sc[CG_TOL] = tol;
        sc[CG_STOP] = (nrm < tol) ? CG_TINY : CG_RUNNING;
        sc[CG_ITER] = 0.0;
    }
}

template <bool HALF>
__global__ __launch_bounds__(1024) void cgj_iter_kernel(int m, int iter, const double *jac, const double *Mp, double *x,
                                                        double *r, double *z, double *p, double *sc, double *report) {
    __shared__ double red[32];
    if (sc[CG_STOP] == CG_RUNNING) {  // the same for every thread: only thread 0 writes it, below
        double a = 0.0, b = 0.0;
        for (int i = threadIdx.x; i < m; i += blockDim.x) {
            a += z[i] * r[i];
            b += p[i] * Mp[i];
        }
        const double rz = block_sum<0>(a, red);
        const double pMp = block_sum<1>(b, red);
        const double alpha = rz / pMp;
        if (HALF) {
            for (int i = threadIdx.x; i < m; i += blockDim.x) x[i] += alpha * p[i];
            return;
        }
        a = 0.0;
        for (int i = threadIdx.x; i < m; i += blockDim.x) {
            x[i] += alpha * p[i];
            const double v = r[i] - alpha * Mp[i], t = v / jac[i];
            r[i] = v;
            z[i] = t;
            a += v * t;
        }
        const double beta = block_sum<0>(a, red) / rz;
        double c = 0.0;
        for (int i = threadIdx.x; i < m; i += blockDim.x) {
            p[i] = z[i] + beta * p[i];
            c += r[i] * r[i];
        }
        const double nrm = sqrt(block_sum<1>(c, red));
        if (threadIdx.x == 0) {
            const double stop = (nrm != nrm)                                   ? CG_NAN
                                : (iter > 20 && nrm > 0.01 * sc[CG_BNORM]) ? CG_STALLED
                                : (nrm < sc[CG_TOL])                           ? CG_CONVERGED
                                                                               : CG_RUNNING;
            sc[CG_RNORM] = nrm;
            sc[CG_ITER] = iter;
            sc[CG_STOP] = stop;
        }
        __threadfence_block();
    }
    if (report && threadIdx.x == 0) {
        report[CG_RNORM] = sc[CG_RNORM];
        report[CG_BNORM] = sc[CG_BNORM];
        report[CG_TOL] = sc[CG_TOL];
        report[CG_ITER] = sc[CG_ITER];
        report[CG_STOP] = sc[CG_STOP];
    }
}

// The same iteration of a vector of at most 1024 E entries, every vector read once into
// registers (E entries per thread) and written once.  The loops above wait for memory in
// each of their three passes: m = 3001 9.5 us against 6.9.  Six entries of six vectors are
// what 128 registers hold; longer vectors keep the loops.
template <int E>
__global__ __launch_bounds__(1024) void cgj_iter_reg_kernel(int m, int iter, const double *jac, const double *Mp,
                                                            double *x, double *r, double *z, double *p, double *sc,
                                                            double *report) {
    __shared__ double red[32];
    const bool running = sc[CG_STOP] == CG_RUNNING;  // the same for every thread, as above
    if (running) {
        const double bnorm = sc[CG_BNORM], tol = sc[CG_TOL];
        double vz[E], vr[E], vp[E], vM[E], vx[E], vj[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = threadIdx.x + 1024 * e;
            const bool in = i < m;
            vz[e] = in ? z[i] : 0.0;
            vr[e] = in ? r[i] : 0.0;
            vp[e] = in ? p[i] : 0.0;
            vM[e] = in ? Mp[i] : 0.0;
            vx[e] = in ? x[i] : 0.0;
            vj[e] = in ? jac[i] : 1.0;
        }
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            a += vz[e] * vr[e];
            b += vp[e] * vM[e];
        }
        const double rz = block_sum<0>(a, red);
        const double pMp = block_sum<1>(b, red);
        const double alpha = rz / pMp;
        a = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            vx[e] += alpha * vp[e];
            const double v = vr[e] - alpha * vM[e], t = v / vj[e];
            vr[e] = v;
            vz[e] = t;
            if ((int) threadIdx.x + 1024 * e < m) a += v * t;
        }
        const double beta = block_sum<0>(a, red) / rz;
        double c = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = threadIdx.x + 1024 * e;
            if (i >= m) continue;
            x[i] = vx[e];
            r[i] = vr[e];
            z[i] = vz[e];
            p[i] = vz[e] + beta * vp[e];
            c += vr[e] * vr[e];
        }
        const double nrm = sqrt(block_sum<1>(c, red));
        if (threadIdx.x == 0) {
            const double stop = (nrm != nrm)                          ? CG_NAN
                                : (iter > 20 && nrm > 0.01 * bnorm) ? CG_STALLED
                                : (nrm < tol)                         ? CG_CONVERGED
                                                                      : CG_RUNNING;
            sc[CG_RNORM] = nrm;
            sc[CG_ITER] = iter;
            sc[CG_STOP] = stop;
            if (report) {
                report[CG_RNORM] = nrm;
                report[CG_BNORM] = bnorm;
                report[CG_TOL] = tol;
                report[CG_ITER] = iter;
                report[CG_STOP] = stop;
            }
        }
    } else if (report && threadIdx.x == 0) {
        report[CG_RNORM] = sc[CG_RNORM];
        report[CG_BNORM] = sc[CG_BNORM];
        report[CG_TOL] = sc[CG_TOL];
        report[CG_ITER] = sc[CG_ITER];
        report[CG_STOP] = sc[CG_STOP];
    }
}

void cgj_start(hipStream_t s, int m, const double *rhs, const double *jac, double relTol, double absTol, double *r,
               double *x, double *z, double *p, double *sc) {
    cgj_start_kernel<<<1, 1024, 0, s>>>(m, rhs, jac, relTol, absTol, r, x, z, p, sc);
}
void cgj_iter(hipStream_t s, int m, int iter, const double *jac, const double *Mp, double *x, double *r, double *z,
              double *p, double *sc, double *report) {
#define HDK_CGJ(e)                                                                                           \
    if (m <= 1024 * e) {                                                                                     \
        cgj_iter_reg_kernel<e><<<1, 1024, 0, s>>>(m, iter, jac, Mp, x, r, z, p, sc, report);                 \
        return;                                                                                              \
    }
    HDK_CGJ(1)
    HDK_CGJ(2)
    HDK_CGJ(3)
    HDK_CGJ(4)
    HDK_CGJ(6)
#undef HDK_CGJ
    cgj_iter_kernel<false><<<1, 1024, 0, s>>>(m, iter, jac, Mp, x, r, z, p, sc, report);
}
void cgj_half(hipStream_t s, int m, const double *z, const double *r, const double *p, const double *Mp, double *x,
              double *sc) {
    cgj_iter_kernel<true><<<1, 1024, 0, s>>>(m, 0, nullptr, Mp, x, const_cast<double *>(r), const_cast<double *>(z),
                                             const_cast<double *>(p), sc, nullptr);
}

// Workgroups of eight waves that keep small matrices on the CU: wave w holds the columns
// 4 (w + 8 q) + c, c < 4, q < 2 NU, of a matrix of at most 64 NU rows, lane l the rows l,
// l + 64, ... of each.

// Sum over a workgroup whose first four waves hold the values, in every thread: each wave's
// tree sum, then the four in order, block_sum's result (its other waves add zeros).
template <int B>
__device__ inline double block_sum4(double v, double *red) {
    if (threadIdx.x < 256) {
        v = wave_tree_sum(v);
        if ((threadIdx.x & 63) == 0) red[4 * B + (threadIdx.x >> 6)] = v;
    }
    __syncthreads();
    double total = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) total += red[4 * B + w];
    return total;
}

// One workgroup: M in registers (and, of a matrix of more than 192 rows, the last quarter of
// its columns in LDS), every vector in LDS.  An iteration reads nothing from memory and takes
// 2.9 us at m = 243; with M from L2 in every iteration, at 60 GB/s to the one CU, it took 8.
// CGS_MAX is what a CU holds.  Statements and reduction orders of cgj_iter.
template <int NU>
__global__ __launch_bounds__(512, 2) void cg_small_kernel(int m, const double *M, long ldm, const double *rhs,
                                                          const double *jacG, double relTol, double absTol, int maxIter,
                                                          int restart, double *crhs, double *xG, double *xHost,
                                                          double *report) {
    constexpr int Q = 2 * NU, QR = (NU == 4) ? 6 : Q;  // column groups of a wave, those in registers
    __shared__ double red[8];
    __shared__ double b[CGS_MAX], jac[CGS_MAX], x[CGS_MAX], r[CGS_MAX], z[CGS_MAX], p[CGS_MAX], Mp[CGS_MAX];
    __shared__ double Ml[(Q > QR) ? 8 * (Q - QR) * 4 * 64 * NU : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double Mr[QR][4][NU];
    double *mine = Ml + (Q > QR ? wave * (Q - QR) * 4 * 64 * NU + lane : 0);
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int j = 4 * (wave + 8 * q) + c, i = lane + 64 * u;
                const double v = (j < m && i < m) ? M[i + j * ldm] : 0.0;
                if (q < QR) Mr[q < QR ? q : 0][c][u] = v;
                else mine[((q - QR) * 4 + c) * 64 * NU + 64 * u] = v;
            }
    // y = M p, each column summed in coldot's order
    auto symv = [&](const double *in, double *out) {
        double v[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) v[u] = (lane + 64 * u < m) ? in[lane + 64 * u] : 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            double s[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                s[c] = 0.0;
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    s[c] += ((q < QR) ? Mr[q < QR ? q : 0][c][u] : mine[((q - QR) * 4 + c) * 64 * NU + 64 * u]) * v[u];
            }
            const double t = wave_tree_sum4(s[0], s[1], s[2], s[3]);
            const int j = 4 * (wave + 8 * q) + tree_sum4_slot(lane);
            if ((lane & 15) == 0 && j < m) out[j] = t;
        }
        __syncthreads();
    };
    const int tid = threadIdx.x;
    double acc = 0.0;
    if (tid < m) {
        const double v = rhs[tid], q = jacG[tid];
        b[tid] = v;
        crhs[tid] = v;
        jac[tid] = q;
        r[tid] = v;
        x[tid] = 0.0;
        z[tid] = v / q;
        p[tid] = v / q;
        acc = 0.0 + v * v;
    }
    const double bnorm = sqrt(block_sum4<0>(acc, red));
    const double tol = fmax(fmin(absTol, bnorm * relTol), 0.1 * absTol);
    double nrm = bnorm;
    int stop = (nrm < tol) ? CG_TINY : CG_RUNNING, iter = 0;
    if (stop == CG_RUNNING) {
        symv(p, Mp);
        for (; iter < maxIter; ++iter) {
            double a = 0.0, c = 0.0;
            if (tid < m) {
                a = 0.0 + z[tid] * r[tid];
                c = 0.0 + p[tid] * Mp[tid];
            }
            const double rz = block_sum4<1>(a, red);
            const double alpha = rz / block_sum4<0>(c, red);
            if (iter % restart == 5) {
                if (tid < m) x[tid] += alpha * p[tid];
                __syncthreads();
                symv(x, Mp);
                if (tid < m) {
                    const double v = b[tid] - Mp[tid], t = v / jac[tid];
                    r[tid] = v;
                    z[tid] = t;
                    p[tid] = t;
                }
                __syncthreads();
                symv(p, Mp);
                continue;
            }
            a = 0.0;
            if (tid < m) {
                x[tid] += alpha * p[tid];
                const double v = r[tid] - alpha * Mp[tid], t = v / jac[tid];
                r[tid] = v;
                z[tid] = t;
                a = 0.0 + v * t;
            }
            const double beta = block_sum4<1>(a, red) / rz;
            c = 0.0;
            if (tid < m) {
                p[tid] = z[tid] + beta * p[tid];
                c = 0.0 + r[tid] * r[tid];
            }
            nrm = sqrt(block_sum4<0>(c, red));
            stop = (nrm != nrm)                          ? CG_NAN
                   : (iter > 20 && nrm > 0.01 * bnorm) ? CG_STALLED
                   : (nrm < tol)                         ? CG_CONVERGED
                                                         : CG_RUNNING;
            if (stop != CG_RUNNING) break;
            symv(p, Mp);
        }
    }
    if (stop != CG_TINY && tid < m) {
        xG[tid] = x[tid];
        if (xHost) xHost[tid] = x[tid];
    }
    if (tid == 0) {
        report[CG_RNORM] = nrm;
        report[CG_BNORM] = bnorm;
        report[CG_TOL] = tol;
        report[CG_ITER] = iter;
        report[CG_STOP] = stop;
    }
}

void cg_small(hipStream_t s, int m, const double *M, long ldm, const double *rhs, const double *jac, double relTol,
              double absTol, int maxIter, int restart, double *crhs, double *x, double *xHost, double *report) {
#define HDK_CGS(nu)                                                                                              \
    case nu:                                                                                                     \
        cg_small_kernel<nu><<<1, 512, 0, s>>>(m, M, ldm, rhs, jac, relTol, absTol, maxIter, restart, crhs, x,   \
                                               xHost, report);                                                   \
        break;
    switch ((m + 63) / 64) {
        HDK_CGS(1) HDK_CGS(2) HDK_CGS(3) HDK_CGS(4)
    }
#undef HDK_CGS
}

// ---- Lanczos (linalg/hdsdp_lanczos.c:196-286) ---------------------------------

// One Lanczos orthogonalisation step on w = Op(v_k):
//   w -= H(k,k-1) V_{k-1};  alp = -w.V_k;  w += alp V_k;  H(k,k) = -alp
//   norm = ||w||;  V_{k+1} = v = w / norm (or 0);  H(k+1,k) = norm
__global__ __launch_bounds__(1024) void lz_step_kernel(int n, int k, double *w, double *V, double *H, int ldh, double *v,
                                                       double *hist) {
    __shared__ double red[32];
    const double *Vk = V + (long) k * n;
    if (k > 0) {
        const double *Vkm = V + (long) (k - 1) * n;
        double h = -H[k + (k - 1) * ldh];
        for (int i = threadIdx.x; i < n; i += blockDim.x) w[i] += h * Vkm[i];
        __syncthreads();
    }
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) a += w[i] * Vk[i];
    double alp = -block_sum<0>(a, red);
    double c = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double t = w[i] + alp * Vk[i];
        w[i] = t;
        c += t * t;
    }
    double nrm = sqrt(block_sum<1>(c, red));
    double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
    double *Vn = V + (long) (k + 1) * n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double t = (nrm > 0.0) ? w[i] * inv : 0.0;
        v[i] = t;
        Vn[i] = t;
    }
    if (threadIdx.x == 0) {
        H[(k + 1) + k * ldh] = (nrm > 0.0) ? nrm : 0.0;
        hist[2 * k] = -alp;
        hist[2 * k + 1] = nrm;
    }
}

// lz_step and the first product of the next step, y_j = <Li(j:n, j), v(j:n)> in coldot's
// order.  Every workgroup takes the step by itself on its own copy of w, workgroup 0 writes its
// results, and each wave forms one column: 5 us at n = 300, 7.4 at 1000 and 10.5 at 2000, where
// the two launches take 7, 8.9 and 13 and the gap between them; LZF_MAX is as far as was measured.
__global__ __launch_bounds__(1024) void lz_step_product_kernel(int n, int k, const double *w, double *V, double *H,
                                                               int ldh, double *hist, const double *Li, double *y) {
    __shared__ double red[32];
    __shared__ double x[LZF_MAX];
    const double *Vk = V + (long) k * n;
    const double h = (k > 0) ? -H[k + (k - 1) * ldh] : 0.0;
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) {
        double t = w[i];
        if (k > 0) t += h * (Vk - n)[i];
        x[i] = t;
        a += t * Vk[i];
    }
    const double alp = -block_sum<0>(a, red);
    double c = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) {
        const double t = x[i] + alp * Vk[i];
        x[i] = t;
        c += t * t;
    }
    const double nrm = sqrt(block_sum<1>(c, red));
    const double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
    double *Vn = V + (long) (k + 1) * n;
    for (int i = threadIdx.x; i < n; i += 1024) {
        const double t = (nrm > 0.0) ? x[i] * inv : 0.0;
        x[i] = t;
        if (blockIdx.x == 0) Vn[i] = t;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        H[(k + 1) + k * ldh] = (nrm > 0.0) ? nrm : 0.0;
        hist[2 * k] = -alp;
        hist[2 * k + 1] = nrm;
    }
    __syncthreads();
    const int j = blockIdx.x * 16 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= n) return;
    const double *col = Li + (long) j * n;
    double sum = 0.0;
    int i = j + lane;
    for (; i + 7 * 64 < n; i += 8 * 64) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = col[i + 64 * u];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += v[u] * x[i + 64 * u];
    }
    for (; i + 64 < n; i += 2 * 64) {
        const double v0 = col[i], v1 = col[i + 64];
        sum += v0 * x[i];
        sum += v1 * x[i + 64];
    }
    if (i < n) sum += col[i] * x[i];
    sum = wave_tree_sum(sum);
    if (lane == 0) y[j] = sum;
}

// x = x0 (+ pert); v = V_0 = x / ||x|| (or 0)
__global__ __launch_bounds__(1024) void lz_start_kernel(int n, const double *x0, const double *pert, double *v,
                                                        double *V) {
    __shared__ double red[32];
    double c = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double x = pert ? x0[i] + pert[i] : x0[i];
        c += x * x;
    }
    double nrm = sqrt(block_sum<0>(c, red));
    double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double x = pert ? x0[i] + pert[i] : x0[i];
        double t = (nrm > 0.0) ? x * inv : 0.0;
        v[i] = t;
        V[i] = t;
    }
}

// z = V[:, 0:kp1] y
__global__ void lz_comb_kernel(int n, int kp1, const double *V, LzCoef y, double *z) {
    for (int i = threadIdx.x + blockIdx.x * blockDim.x; i < n; i += blockDim.x * gridDim.x) {
        double s = 0.0;
        for (int c = 0; c < kp1; ++c) s += V[i + (long) c * n] * y.y[c];
        z[i] = s;
    }
}

// y_j = <A(lo:hi, j), x(lo:hi)> with coldot's rows and order of summation (tri 0, 1, 2) for
// the n <= 64 NU columns, by the 16 waves of one workgroup, four columns at a time; x
// and y in LDS
template <int NU, int TRI>
__device__ inline void small_coldot(int n, const double *__restrict__ A, const double *x, double *y) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int j0 = 4 * w; j0 < n; j0 += 64) {
        double a[4][NU], s[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int j = min(j0 + c, n - 1), lo = (TRI == 1) ? j : 0, hi = (TRI == 2) ? j + 1 : n;
            const double *col = A + (long) j * n + lo + lane;
#pragma unroll
            for (int u = 0; u < NU; ++u) a[c][u] = (lo + lane + 64 * u < hi) ? col[64 * u] : 0.0;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int j = min(j0 + c, n - 1), lo = (TRI == 1) ? j : 0, hi = (TRI == 2) ? j + 1 : n;
            s[c] = 0.0;
#pragma unroll
            for (int u = 0; u < NU; ++u)
                s[c] += a[c][u] * ((lo + lane + 64 * u < hi) ? x[lo + lane + 64 * u] : 0.0);
        }
        const double q = wave_tree_sum4(s[0], s[1], s[2], s[3]);
        const int j = j0 + tree_sum4_slot(lane);
        if ((lane & 15) == 0 && j < n) y[j] = q;
    }
    __syncthreads();
}

// out = L^-1 (-D) L^-T in (in, out, t in LDS)
template <int NU>
__device__ inline void small_op(int n, const double *Li, const double *LiT, const double *D, const double *in, double *t,
                                double *out) {
    small_coldot<NU, 1>(n, Li, in, out);
    small_coldot<NU, 0>(n, D, out, t);
    if ((int) threadIdx.x < n) t[threadIdx.x] = -1.0 * t[threadIdx.x];
    __syncthreads();
    small_coldot<NU, 2>(n, LiT, t, out);
}

// A Lanczos step of a small block is bound by its four launches (three products, the
// step): about 18 us of host time at any n.  In one workgroup, with the two triangles and D
// from L2 at one CU's rate, it takes 12 us at n = 128, 15 at 160 and 22 at 200, where the
// launches cost less; hence LZS_MAX.
template <int NU>
__global__ __launch_bounds__(1024) void lz_small_steps_kernel(int n, int k0, int k1, const double *x0,
                                                              const double *pert, const double *Li, const double *LiT,
                                                              const double *D, double *V, double *H, int ldh,
                                                              double *hist) {
    __shared__ double red[32], v[LZS_MAX], w[LZS_MAX], t[LZS_MAX];
    const int i = threadIdx.x;
    double vm = 0.0;  // V_{k - 1} and its norm at the step before
    double prev = 0.0;
    if (k0 == 0) {
        double x = 0.0, c = 0.0;
        if (i < n) {
            x = pert ? x0[i] + pert[i] : x0[i];
            c = 0.0 + x * x;
        }
        const double nrm = sqrt(block_sum<0>(c, red));
        const double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
        if (i < n) {
            const double q = (nrm > 0.0) ? x * inv : 0.0;
            v[i] = q;
            V[i] = q;
        }
    } else {
        prev = H[k0 + (k0 - 1) * ldh];
        if (i < n) {
            vm = V[i + (long) (k0 - 1) * n];
            v[i] = V[i + (long) k0 * n];
        }
    }
    __syncthreads();
    for (int k = k0; k < k1; ++k) {
        small_op<NU>(n, Li, LiT, D, v, t, w);
        double q = 0.0, vk = 0.0, a = 0.0;
        if (i < n) {
            q = w[i];
            vk = v[i];
            if (k > 0) q += -prev * vm;
            a = 0.0 + q * vk;
        }
        const double alp = -block_sum<1>(a, red);
        double c = 0.0;
        if (i < n) {
            q = q + alp * vk;
            c = 0.0 + q * q;
        }
        const double nrm = sqrt(block_sum<0>(c, red));
        const double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
        vm = vk;
        prev = (nrm > 0.0) ? nrm : 0.0;
        if (i < n) {
            const double u = (nrm > 0.0) ? q * inv : 0.0;
            v[i] = u;
            V[i + (long) (k + 1) * n] = u;
        }
        if (i == 0) {
            H[(k + 1) + k * ldh] = prev;
            hist[2 * k] = -alp;
            hist[2 * k + 1] = nrm;
        }
        __syncthreads();
    }
}

// The same with L^-1, D and L^-T in the registers of eight waves (n <= 64 NU <= 128): a step
// reads nothing from memory.  n = 121: 4 us per step, 12 with the matrices from L2; n = 50: 2.5
// and 6.
template <int NU>
__global__ __launch_bounds__(512, 2) void lz_resident_steps_kernel(int n, int k0, int k1, const double *x0,
                                                                   const double *pert, const double *Li,
                                                                   const double *LiT, const double *D, double *V,
                                                                   double *H, int ldh, double *hist) {
    constexpr int Q = 2 * NU;
    // vectors padded with zeros: a column of L^-1 starts at its diagonal and runs past n
    __shared__ double red[8], v[128 * NU], w[128 * NU], t[128 * NU];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double R[3][Q][4][NU];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int j = 4 * (wave + 8 * q) + c, row = lane + 64 * u;
                R[0][q][c][u] = (j < n && j + row < n) ? Li[j + row + (long) j * n] : 0.0;
                R[1][q][c][u] = (j < n && row < n) ? D[row + (long) j * n] : 0.0;
                R[2][q][c][u] = (j < n && row < j + 1) ? LiT[row + (long) j * n] : 0.0;
            }
    for (int e = threadIdx.x; e < 128 * NU; e += 512) v[e] = w[e] = t[e] = 0.0;
    __syncthreads();
    // products with matrix f and coldot's rows and order of summation: 0 from the diagonal
    // down, 1 all rows, 2 down to the diagonal
    auto product = [&](auto f, const double *in, double *out) {
        constexpr int F = decltype(f)::value;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int j0 = 4 * (wave + 8 * q);
            double s[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                s[c] = 0.0;
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    const double x = in[(F == 0 ? min(j0 + c, n - 1) : 0) + lane + 64 * u];
                    s[c] += R[F][q][c][u] * ((F == 2 && lane + 64 * u > j0 + c) ? 0.0 : x);
                }
            }
            const double sum = wave_tree_sum4(s[0], s[1], s[2], s[3]);
            const int j = j0 + tree_sum4_slot(lane);
            if ((lane & 15) == 0 && j < n) out[j] = sum;
        }
        __syncthreads();
    };
    const int i = threadIdx.x;
    double vm = 0.0;  // V_{k - 1} and its norm at the step before
    double prev = 0.0;
    if (k0 == 0) {
        double x = 0.0, c = 0.0;
        if (i < n) {
            x = pert ? x0[i] + pert[i] : x0[i];
            c = 0.0 + x * x;
        }
        const double nrm = sqrt(block_sum4<0>(c, red));
        const double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
        if (i < n) {
            const double q = (nrm > 0.0) ? x * inv : 0.0;
            v[i] = q;
            V[i] = q;
        }
    } else {
        prev = H[k0 + (k0 - 1) * ldh];
        if (i < n) {
            vm = V[i + (long) (k0 - 1) * n];
            v[i] = V[i + (long) k0 * n];
        }
    }
    __syncthreads();
    for (int k = k0; k < k1; ++k) {
        product(std::integral_constant<int, 0>(), v, w);
        product(std::integral_constant<int, 1>(), w, t);
        if (i < n) t[i] = -1.0 * t[i];
        __syncthreads();
        product(std::integral_constant<int, 2>(), t, w);
        double q = 0.0, vk = 0.0, a = 0.0;
        if (i < n) {
            q = w[i];
            vk = v[i];
            if (k > 0) q += -prev * vm;
            a = 0.0 + q * vk;
        }
        const double alp = -block_sum4<1>(a, red);
        double c = 0.0;
        if (i < n) {
            q = q + alp * vk;
            c = 0.0 + q * q;
        }
        const double nrm = sqrt(block_sum4<0>(c, red));
        const double inv = (nrm > 0.0) ? 1.0 / nrm : 0.0;
        vm = vk;
        prev = (nrm > 0.0) ? nrm : 0.0;
        if (i < n) {
            const double u = (nrm > 0.0) ? q * inv : 0.0;
            v[i] = u;
            V[i + (long) (k + 1) * n] = u;
        }
        if (i == 0) {
            H[(k + 1) + k * ldh] = prev;
            hist[2 * k] = -alp;
            hist[2 * k + 1] = nrm;
        }
        __syncthreads();
    }
}

template <int NU>
__global__ __launch_bounds__(1024) void lz_small_bound_kernel(int n, int kp1, double e1, LzCoef y1, LzCoef y2,
                                                              const double *Li, const double *LiT, const double *D,
                                                              const double *V, double *warm, double *report) {
    __shared__ double red[32], z[LZS_MAX], w[LZS_MAX], t[LZS_MAX];
    const int i = threadIdx.x;
    double s1 = 0.0, s2 = 0.0;
    if (i < n) {
        for (int c = 0; c < kp1; ++c) {
            const double q = V[i + (long) c * n];
            s1 += q * y1.y[c];
            s2 += q * y2.y[c];
        }
        z[i] = s1;
    }
    __syncthreads();
    small_op<NU>(n, Li, LiT, D, z, t, w);
    double c = 0.0;
    if (i < n) {
        const double q = w[i];
        warm[i] = q;
        const double u = q + -e1 * s1;
        c = 0.0 + u * u;
        z[i] = s2;
    }
    const double r1 = sqrt(block_sum<0>(c, red));
    small_op<NU>(n, Li, LiT, D, z, t, w);
    c = 0.0;
    if (i < n) {
        const double u = w[i] + -e1 * s2;
        c = 0.0 + u * u;
    }
    const double r2 = sqrt(block_sum<1>(c, red));
    if (i == 0) {
        report[LZ_R1] = r1;
        report[LZ_R2] = r2;
    }
}

#define HDK_LZS(call)                      \
    switch ((n + 63) / 64) {               \
        case 1: { constexpr int NU = 1; call; break; } \
        case 2: { constexpr int NU = 2; call; break; } \
        default: { constexpr int NU = 3; call; break; } \
    }
void lz_small_steps(hipStream_t s, int n, int k0, int k1, const double *x0, const double *pert, const double *Li,
                    const double *LiT, const double *D, double *V, double *H, int ldh, double *hist) {
    if (n <= 64)
        lz_resident_steps_kernel<1><<<1, 512, 0, s>>>(n, k0, k1, x0, pert, Li, LiT, D, V, H, ldh, hist);
    else if (n <= 128)
        lz_resident_steps_kernel<2><<<1, 512, 0, s>>>(n, k0, k1, x0, pert, Li, LiT, D, V, H, ldh, hist);
    else
        lz_small_steps_kernel<3><<<1, 1024, 0, s>>>(n, k0, k1, x0, pert, Li, LiT, D, V, H, ldh, hist);
}
void lz_small_bound(hipStream_t s, int n, int kp1, double e1, const LzCoef &y1, const LzCoef &y2, const double *Li,
                    const double *LiT, const double *D, const double *V, double *warm, double *report) {
    HDK_LZS((lz_small_bound_kernel<NU><<<1, 1024, 0, s>>>(n, kp1, e1, y1, y2, Li, LiT, D, V, warm, report)))
}
#undef HDK_LZS

// y += a x; sc[slot] = ||y||
__global__ __launch_bounds__(1024) void axpy_norm_kernel(int n, double a, const double *x, double *y, double *sc, int slot) {
    __shared__ double red[32];
    double c = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double t = y[i] + a * x[i];
        y[i] = t;
        c += t * t;
    }
    double nrm = sqrt(block_sum<0>(c, red));
    if (threadIdx.x == 0) sc[slot] = nrm;
}

void lz_step(hipStream_t s, int n, int k, double *w, double *V, double *H, int ldh, double *v, double *hist) {
    lz_step_kernel<<<1, 1024, 0, s>>>(n, k, w, V, H, ldh, v, hist);
}
void lz_step_product(hipStream_t s, int n, int k, const double *w, double *V, double *H, int ldh, double *hist,
                     const double *Li, double *y) {
    lz_step_product_kernel<<<(n + 15) / 16, 1024, 0, s>>>(n, k, w, V, H, ldh, hist, Li, y);
}
void lz_start(hipStream_t s, int n, const double *x0, const double *pert, double *v, double *V) {
    lz_start_kernel<<<1, 1024, 0, s>>>(n, x0, pert, v, V);
}
void lz_comb(hipStream_t s, int n, int kp1, const double *V, const LzCoef &y, double *z) {
    lz_comb_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, kp1, V, y, z);
}
void axpy_norm(hipStream_t s, int n, double a, const double *x, double *y, double *sc, int slot) {
    axpy_norm_kernel<<<1, 1024, 0, s>>>(n, a, x, y, sc, slot);
}

// ---- generic ------------------------------------------------------------------

__global__ void axpy_kernel(long n, double a, const double *x, double *y) {
    for (long i = threadIdx.x + blockIdx.x * (long) blockDim.x; i < n; i += (long) blockDim.x * gridDim.x)
        y[i] += a * x[i];
}

void axpy(hipStream_t s, long n, double a, const double *x, double *y) {
    long blocks = (n + 255) / 256;
    axpy_kernel<<<blocks > 4096 ? 4096 : blocks, 256, 0, s>>>(n, a, x, y);
}

// M_ii += reg where reg = min(r * min_i M_ii, 1e-5), dropped below 1e-14
// (interface/hdsdp_schur.c:348-373)
__global__ __launch_bounds__(1024) void regularize_kernel(int m, double *M, long ldm, double r) {
    __shared__ double red[32];
    double mn = 1e+30;
    for (int i = threadIdx.x; i < m; i += blockDim.x) mn = fmin(mn, M[i + i * ldm]);
    for (int off = 32; off > 0; off >>= 1) mn = fmin(mn, __shfl_down(mn, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mn;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 1e+30;
        for (int w = 0; w < (int) (blockDim.x >> 6); ++w) t = fmin(t, red[w]);
        double reg = r * t;
        reg = fmin(reg, 1e-05);
        if (reg < 1e-14) reg = 0.0;
        red[16] = reg;
    }
    __syncthreads();
    double reg = red[16];
    for (int i = threadIdx.x; i < m; i += blockDim.x) M[i + i * ldm] += reg;
}

__global__ void shift_coef_kernel(int m, const double *x, double *coef) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > m) return;
    coef[i] = (i == 0) ? 0.0 : x[i - 1];
}

void shift_coef(hipStream_t s, int m, const double *x, double *coef) {
    shift_coef_kernel<<<(m + 256) / 256, 256, 0, s>>>(m, x, coef);
}

__global__ void diag_delta_axpy_kernel(int m, const double *M, long ldm, const double *ref, const double *x,
                                       double *y) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    y[i] += (M[i + i * ldm] - ref[i]) * x[i];
}

void diag_delta_axpy(hipStream_t s, int m, const double *M, long ldm, const double *ref, const double *x, double *y) {
    diag_delta_axpy_kernel<<<(m + 255) / 256, 256, 0, s>>>(m, M, ldm, ref, x, y);
}

void regularize(hipStream_t s, int m, double *M, long ldm, double r) {
    regularize_kernel<<<1, 1024, 0, s>>>(m, M, ldm, r);
}

__global__ void get_diag_kernel(int m, const double *M, long ldm, double *d) {
    for (int i = threadIdx.x + blockIdx.x * blockDim.x; i < m; i += blockDim.x * gridDim.x) d[i] = M[i + i * ldm];
}

void get_diag(hipStream_t s, int m, const double *M, long ldm, double *d) {
    get_diag_kernel<<<(m + 255) / 256, 256, 0, s>>>(m, M, ldm, d);
}

__global__ void f2d_kernel(long n, const float *x, double *y) {
    for (long i = threadIdx.x + blockIdx.x * (long) blockDim.x; i < n; i += (long) blockDim.x * gridDim.x) y[i] = x[i];
}
__global__ void d2f_kernel(long n, const double *x, float *y) {
    for (long i = threadIdx.x + blockIdx.x * (long) blockDim.x; i < n; i += (long) blockDim.x * gridDim.x)
        y[i] = (float) x[i];
}

__global__ void f2d_scaled_kernel(long n, const float *x, const double *sc, double *y) {
    for (long i = threadIdx.x + blockIdx.x * (long) blockDim.x; i < n; i += (long) blockDim.x * gridDim.x)
        y[i] = (double) x[i] * sc[i];
}
__global__ void d2f_scaled_kernel(long n, const double *x, const double *sc, float *y) {
    for (long i = threadIdx.x + blockIdx.x * (long) blockDim.x; i < n; i += (long) blockDim.x * gridDim.x)
        y[i] = (float) (x[i] * sc[i]);
}
__global__ void jacobi_scale_kernel(int m, const double *M, long ldm, double *sc) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) {
        const double d = M[i + (long) i * ldm];
        sc[i] = (d > 0.0) ? 1.0 / sqrt(d) : 1.0;
    }
}
void f2d_scaled(hipStream_t s, long n, const float *x, const double *sc, double *y) {
    f2d_scaled_kernel<<<(n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256, 256, 0, s>>>(n, x, sc, y);
}
void d2f_scaled(hipStream_t s, long n, const double *x, const double *sc, float *y) {
    d2f_scaled_kernel<<<(n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256, 256, 0, s>>>(n, x, sc, y);
}
void jacobi_scale(hipStream_t s, int m, const double *M, long ldm, double *sc) {
    jacobi_scale_kernel<<<(m + 255) / 256, 256, 0, s>>>(m, M, ldm, sc);
}

void f2d(hipStream_t s, long n, const float *x, double *y) {
    f2d_kernel<<<(n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256, 256, 0, s>>>(n, x, y);
}
void d2f(hipStream_t s, long n, const double *x, float *y) {
    d2f_kernel<<<(n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256, 256, 0, s>>>(n, x, y);
}

}  // namespace hdk
