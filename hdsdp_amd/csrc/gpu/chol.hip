// chol.hip -- Cholesky of the dual slack S and of the Schur matrix M on gfx950.
//
// The factorisation is bound by its serial chain of 64 x 64 diagonal blocks, not by
// flops: at n = 2000 the flops take 40 us of MFMA time and the matrix has 32 such
// blocks.  Two things keep the chain short:
//
//  * One launch per block column.  chol_step_kernel(k) applies panel k - 1 to every
//    remaining 64 x 64 tile, one workgroup per tile, and its workgroup 0 applies it to
//    the diagonal tile (k, k) and factors that tile at once, beside the other tiles.
//    A workgroup forms the panel blocks it needs (L(i, k - 1) = A(i, k - 1) X^T with the
//    64 x 64 inverse X of the last diagonal factor) by itself instead of waiting for
//    a panel launch; the factor goes to a matrix of its own, so no workgroup
//    overwrites a block that another still reads.
//  * A blocked leaf.  The 64 x 64 block is factored in four blocks of 16 columns: one
//    wave holds a 16-column block in registers and eliminates it column by column with
//    DPP broadcasts (no LDS and no barrier inside the 16 steps); trailing updates and
//    the products of the block's inverse are 16 x 16 x 16 MFMA products on the other
//    waves.
//
// A block column takes 20 us this way against 52 us as three launches (an eight-wave
// leaf with an LDS round trip and a barrier per column, a panel product, an update):
// n = 500: 160 us, n = 1000: 325 us, n = 2000: 680 us (1.8 ms before), m = 8084: 6.5 ms.
// Results are those of the unblocked leaf bit for bit up to n = 64 CH_FLAT; an elimination
// with reciprocals instead of correctly rounded quotients took 16 us per block column,
// but the interior-point path amplifies its rounding into other iterates.
//
// Tiles are computed transposed (MFMA rows = columns of the tile), so that a wave
// loads, stores and stages 16 consecutive rows of a column per lane group.
#include "dev_common.h"

#include <utility>

namespace hdk {

namespace {

constexpr int CH_THREADS = 512;
// LDS column of 64 rows padded to 72: the four lane groups of an operand read start
// 8 doubles apart (mod 32), two lanes per bank pair, the minimum for 512 bytes
constexpr int CH_LD = 72;

__device__ inline v4d mma(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// lane K of each group of 16 lanes to its whole group
template <int K>
__device__ inline double row_bcast(double v) {
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + K, 0xf, 0xf, true);
}

// a / p of the elimination.  Fast form: r = recip(p) from the hardware's approximation
// (relative error e below 2^-22) with the third-order step x (1 + e + e^2), half an ulp and
// 2^-13 of one off at most, and the quotient from a r with one residual step: correctly
// rounded unless a / p lies within some 2^-53 ulp of the middle of two numbers (or |a| below
// 2^-969 makes the residual underflow: an ulp then).  p and r have to be normal numbers: a tile
// with a pivot outside FAST_MIN .. FAST_MAX is factored again with divisions (DIV), which
// takes the step from 20 us to 27.
constexpr double FAST_MIN = 0x1p-960, FAST_MAX = 0x1p960;

template <bool DIV>
__device__ inline double recip(double p) {
    if (DIV) return 0.0;
    const double x = __builtin_amdgcn_rcp(p);
    const double e = __builtin_fma(-p, x, 1.0);
    return __builtin_fma(x, __builtin_fma(e, e, e), x);
}

template <bool DIV>
__device__ inline double quot(double a, double p, double r) {
    if (DIV) return a / p;
    const double u = a * r;
    return __builtin_fma(__builtin_fma(-u, p, a), r, u);
}

template <int... C>
__device__ inline void row_bcast_all(double v, double (&out)[16], std::integer_sequence<int, C...>) {
    ((out[C] = row_bcast<C>(v)), ...);
}

// Column K of a right-looking factorisation of a 16-column block: lane (j, g) = (lane mod
// 16, lane / 16) holds row j of the diagonal block (a, every group all of it) and one
// row of the 64 of the tile (z).  Every row subtracts t = z(K) / p times column K of the
// diagonal block, p = pivot K; column K keeps its values before the step (they become
// column K of the factor).  The next pivot is formed from its own two entries ahead of
// the row updates, by the operations of those updates: the chain from pivot to pivot
// has no cross-lane operation.  Entries above the diagonal are scratch.
template <int K, bool DIV>
__device__ inline void elim_step(double (&a)[16], double (&z)[16], double &p, double &piv, int j) {
    piv = (j == K) ? p : piv;
    const double r = recip<DIV>(p), pk = p;
    if (K < 15) {
        const double q = row_bcast<(K + 1) & 15>(a[K]), d = row_bcast<(K + 1) & 15>(a[(K + 1) & 15]);
        p = __builtin_fma(-quot<DIV>(q, pk, r), q, d);
    }
    double col[16];
    row_bcast_all(a[K], col, std::make_integer_sequence<int, 16>());
    const double ta = -quot<DIV>(a[K], pk, r), tz = -quot<DIV>(z[K], pk, r);
#pragma unroll
    for (int c = K + 1; c < 16; ++c) {
        a[c] = __builtin_fma(ta, col[c], a[c]);
        z[c] = __builtin_fma(tz, col[c], z[c]);
    }
}

// the 16 columns of a block; returns pivot j on the lanes (j, .)
template <bool DIV, int... K>
__device__ inline double elim(double (&a)[16], double (&z)[16], int j, std::integer_sequence<int, K...>) {
    asm volatile("" : "+v"(j));  // keeps the step masks out of the caller's registers
    double p = row_bcast<0>(a[0]), piv = 1.0;
    (elim_step<K, DIV>(a, z, p, piv, j), ...);
    return piv;
}

// P^T (columns 16 c .. 16 c + 15, rows of the operand) = X A^T for the operand rows av
// (av[q] = A(row, 4 q + g)) and the lower-triangular 64 x 64 inverse X staged as [k][row]
__device__ inline v4d panel_block(const double (*X)[CH_LD], const double (&av)[16], int c, int l, int g) {
    v4d acc = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 16; ++q)
        if (q < 4 * (c + 1)) acc = mma(X[4 * q + g][16 * c + l], av[q], acc);
    return acc;
}

// a 64 x 64 column-major block into LDS: two columns of 32 pairs per wave and load
struct Pair4 {
    double2 v[4];
};
__device__ inline Pair4 fetch64(const double *D, int tid) {
    Pair4 p;
#pragma unroll
    for (int u = 0; u < 4; ++u) p.v[u] = reinterpret_cast<const double2 *>(D)[tid + CH_THREADS * u];
    return p;
}
__device__ inline void stash64(double (*X)[CH_LD], const Pair4 &p, int tid) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + CH_THREADS * u;
        *reinterpret_cast<double2 *>(&X[e >> 5][2 * (e & 31)]) = p.v[u];
    }
}

// rows row0 + l of block column kp of A (64 columns), av[q] = A(row0 + l, 64 kp + 4 q + g)
template <typename T>
__device__ inline void load_rows(const T *A, long lda, int n, int row, int kp, int g, double (&av)[16]) {
    const T *p = A + row + (long) (64 * kp + g) * lda;
#pragma unroll
    for (int q = 0; q < 16; ++q) av[q] = (row < n) ? (double) p[(long) (4 * q) * lda] : 0.0;
}

template <typename T>
__device__ inline void store_panel(T *L, long ldl, int n, int row, int kp, int c, int g, v4d p) {
    if (row >= n) return;
    T *q = L + row + (long) (64 * kp + 16 * c + g) * ldl;
#pragma unroll
    for (int r = 0; r < 4; ++r) q[(long) (4 * r) * ldl] = (T) p[r];
}

// C^T - P1 P0^T over a 16 x 16 block: rows of P0 (tile rows, block rb), rows of P1
// (tile columns, block cb), both staged as [k][row]; the product is summed first and
// subtracted once, as a rank-64 update by GEMM rounds
__device__ inline v4d rank64(const double (*P1)[CH_LD], const double (*P0)[CH_LD], int cb, int rb, int l, int g,
                             v4d c) {
    v4d acc = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 16; ++q) acc = mma(P1[4 * q + g][16 * cb + l], P0[4 * q + g][16 * rb + l], acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) c[r] -= acc[r];
    return c;
}

// Diagonal tile k: D = A(k, k) - L(k, kp) L(k, kp)^T (kp >= 0), then D = L L^T and
// X = L^-1, in four blocks of 16 columns.  Wave 0 carries the chain: it factors a block
// column for all rows below (elim); then up to three waves apply it to the next block
// column, and while wave 0 factors that one, the others apply it to the rest, scale the
// column to L's and form the rows of X.  Every entry of L and X sees the operations of
// the unblocked right-looking factorisation and of forward substitution in their order
// (an FP64 MFMA adds its four products one after the other, each rounded as an FMA), so
// the blocking does not change a bit of them.
struct LeafScratch {
    double p[64], r[64];  // pivots and their reciprocals
    int fail, again;
};

// Returns whether the tile has to be factored again with divisions (L and X not stored).
template <typename T, bool DIV>
__device__ bool leaf_role(int n, const T *A, long lda, T *L, long ldl, double *Dinv, int k, int kp, int *info,
                          double (*B0)[CH_LD], double (*B1)[CH_LD], LeafScratch *ls) {
    // B0: the panel rows P, then X; B1: the inverse of the last diagonal factor, then the tile
    double (*P)[CH_LD] = B0, (*Xs)[CH_LD] = B0, (*As)[CH_LD] = B1;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = lane & 15,
              g = lane >> 4;
    const int k0 = 64 * k, kb = min(64, n - k0);
    // the first step of an outer block (the others read info below); this workgroup is the
    // only one that writes it, so every thread reads the same
    const int failed = (kp < 0 && k > 0) ? *info : 0;
    // entry (r, c) of the diagonal tile, identity beyond kb; only the lower triangle of A
    // is valid
    auto diag = [&](int r, int c) -> double {
        const int i = max(r, c), j = min(r, c);
        return (i < kb) ? (double) A[(k0 + i) + (long) (k0 + j) * lda] : (r == c ? 1.0 : 0.0);
    };
    // lower 16-blocks (rb, cb) of the tile: block column 0 on waves 0 - 3, before the first
    // barrier; the other six on waves 5 - 7, two each, beside wave 0's first columns
    const int rbA = (w < 4) ? w : w - 4, cbA = (w < 4) ? 0 : 1;  // (w, 0); (1, 1), (2, 1), (3, 1)
    const int rbB = (w == 5) ? 2 : 3, cbB = (w == 7) ? 3 : 2;    // (2, 2), (3, 2), (3, 3)
    v4d cA = {0, 0, 0, 0}, cB = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (w != 4) cA[r] = diag(16 * rbA + l, 16 * cbA + 4 * r + g);
        if (w > 4) cB[r] = diag(16 * rbB + l, 16 * cbB + 4 * r + g);
    }
    if (failed) return false;  // an earlier pivot was not positive
    if (kp >= 0) {
        const int rb = w & 3, ca = (w < 4) ? 0 : 1, cb = 3 - ca;
        const Pair4 xp = fetch64(Dinv + (long) kp * 4096, tid);
        double av[16];
        load_rows(A, lda, n, k0 + 16 * rb + l, kp, g, av);
        const int bad = *info;
        stash64(B1, xp, tid);
        __syncthreads();
        const v4d pa = panel_block(B1, av, ca, l, g), pb = panel_block(B1, av, cb, l, g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            P[16 * ca + 4 * r + g][16 * rb + l] = pa[r];
            P[16 * cb + 4 * r + g][16 * rb + l] = pb[r];
        }
        if (bad) return false;
        store_panel(L, ldl, n, k0 + 16 * rb + l, kp, ca, g, pa);
        store_panel(L, ldl, n, k0 + 16 * rb + l, kp, cb, g, pb);
        __syncthreads();
        if (w < 4) cA = rank64(P, P, cbA, rbA, l, g, cA);
    }
    if (w < 4)
#pragma unroll
        for (int r = 0; r < 4; ++r) As[16 * cbA + 4 * r + g][16 * rbA + l] = cA[r];
    if (tid == 0) {
        ls->fail = 64;
        ls->again = 0;
    }
    __syncthreads();
    if (w > 4) {
        if (kp >= 0) {
            cA = rank64(P, P, cbA, rbA, l, g, cA);
            cB = rank64(P, P, cbB, rbB, l, g, cB);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            As[16 * cbA + 4 * r + g][16 * rbA + l] = cA[r];
            As[16 * cbB + 4 * r + g][16 * rbB + l] = cB[r];
        }
    }
    // trailing block (i, j) of step b: a(r, c) -= sum_K t(r, K) a(c, K), t = a / pivot
    auto trail = [&](int i, int j, int b) {
        v4d c;
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r] = As[16 * j + 4 * r + g][16 * i + l];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int K = 16 * b + 4 * q + g;
            c = mma(-As[K][16 * j + l], quot<DIV>(As[K][16 * i + l], ls->p[K], ls->r[K]), c);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) As[16 * j + 4 * r + g][16 * i + l] = c[r];
    };
    // Y(b, j) = - sum_{j <= t < b} L(b, t) X(t, j) into X's place
    auto xrow_sum = [&](int b, int j) {
        v4d y = {0, 0, 0, 0};
        for (int t = j; t < b; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y = mma(-As[16 * b + l][16 * t + 4 * q + g], Xs[16 * t + 4 * q + g][16 * j + l], y);
#pragma unroll
        for (int r = 0; r < 4; ++r) Xs[16 * b + 4 * r + g][16 * j + l] = y[r];
    };
    // rows 16 b .. 16 b + 15 of X by forward substitution from Y, lane = column
    auto xrow_solve = [&](int b) {
        double x[16];
#pragma unroll
        for (int k = 0; k < 16; ++k)
            x[k] = (lane < 16 * b) ? Xs[16 * b + k][lane] : (lane == 16 * b + k ? 1.0 : 0.0);
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const double d = As[16 * b + k][16 * b + k];
            x[k] = quot<DIV>(x[k], d, recip<DIV>(d));
#pragma unroll
            for (int i = k + 1; i < 16; ++i) x[i] = __builtin_fma(-As[16 * b + k][16 * b + i], x[k], x[i]);
        }
        if (lane < 16 * (b + 1))
#pragma unroll
            for (int k = 0; k < 16; ++k) Xs[16 * b + k][lane] = x[k];
    };
    // L(r, c) = a(r, c) / sqrt(pivot c) of block column b, 16-row block i: the diagonal
    // block in its place, the others in the mirrored block above the diagonal (lane
    // (l, g): row l, columns g, g + 4, ...)
    auto scale = [&](int i, int b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = 16 * b + 4 * q + g;
            const double s = sqrt(ls->p[c]), v = quot<DIV>(As[c][16 * i + l], s, recip<DIV>(s));
            if (i > b) As[16 * i + l][c] = v;
            else As[c][16 * i + l] = (4 * q + g == l) ? s : v;
        }
    };
    for (int b = 0; b < 4; ++b) {
        double z[16], piv = 1.0;
        const int zb = (b + g < 4) ? b + g : b;  // 16-row block of this lane's row
        if (w == 0) {
            double a[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                a[c] = As[16 * b + c][16 * b + l];
                z[c] = As[16 * b + c][16 * zb + l];
            }
            piv = elim<DIV>(a, z, l, std::make_integer_sequence<int, 16>());
        }
        if (b == 0) __syncthreads();  // every wave is done with P
        if (w == 0) {
            if (b + g < 4)
#pragma unroll
                for (int c = 0; c < 16; ++c) As[16 * b + c][16 * zb + l] = z[c];
            if (lane < 16) {
                ls->p[16 * b + l] = piv;
                ls->r[16 * b + l] = recip<DIV>(piv);
            }
            // the first pivot that is not positive, or that the fast quotients are not made for
            const unsigned long long odd = __ballot(DIV ? !(piv > 0.0) : !(piv >= FAST_MIN && piv <= FAST_MAX));
            if (odd && lane == __ffsll(odd) - 1 && ls->fail == 64 && !ls->again) {
                if (!DIV && piv > 0.0) ls->again = 1;
                else ls->fail = 16 * b + lane;
            }
        } else if (b > 0 && w < 4) {
            // the rest of step b - 1: block columns beyond b, and the column's L
            int q = 0;
            for (int j = b + 1; j < 4; ++j)
                for (int i = j; i < 4; ++i)
                    if (q++ % 3 == w - 1) trail(i, j, b - 1);
            if (b - 1 + w < 4) scale(b - 1 + w, b - 1);
        } else if (b > 0 && w == 5) {
            for (int j = 0; j < b - 1; ++j) xrow_sum(b - 1, j);
            xrow_solve(b - 1);
        }
        __syncthreads();
        if (ls->fail < 64 || ls->again) break;  // the same for every thread: wave 0 wrote them before the barrier
        if (w < 3 - b) trail(b + 1 + w, b + 1, b);
        else if (w == 4) scale(b, b);
        else if (b == 3 && w > 0 && w < 4) xrow_sum(3, w - 1);
        __syncthreads();
    }
    if (!DIV && ls->again) return true;
    if (ls->fail < 64) {
        if (tid == 0) *info = k0 + ls->fail + 1;
        return false;
    }
    if (w == 0) xrow_solve(3);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int c = w + 8 * u;
        const double v = ((lane >> 4) == (c >> 4)) ? As[c][lane] : As[lane][c];
        if (lane >= c && lane < kb && c < kb) L[(k0 + lane) + (long) (k0 + c) * ldl] = (T) v;
    }
    __syncthreads();
    double *D = Dinv + (long) k * 4096;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int c = w + 8 * u;
        D[lane + 64 * c] = (lane >= c) ? Xs[lane][c] : 0.0;
    }
    return false;
}

// Step k of the factorisation of the lower triangle of A (destroyed) into L: workgroup 0
// factors the diagonal tile (k, k); the others apply panel kp = k - 1 to the tiles (i, j),
// k <= j < jEnd, j <= i, and write L(i, kp).  kp < 0: nothing to apply (grid of one).
// One workgroup per CU (214 registers); capped at 128 registers, for two per CU, the leaf
// spills and the step takes 23 us.
template <typename T>
__global__ __launch_bounds__(CH_THREADS, 2) void chol_step_kernel(int n, T *A, long lda, T *L, long ldl, double *Dinv,
                                                                  int k, int kp, int jEnd, int *info) {
    __shared__ __attribute__((aligned(16))) double P0[64][CH_LD], P1[64][CH_LD];
    __shared__ LeafScratch ls;
    __shared__ int bad;
    if (blockIdx.x == 0) {
        if (k == 0 && threadIdx.x == 0) *info = 0;
        if (leaf_role<T, false>(n, A, lda, L, ldl, Dinv, k, kp, info, P0, P1, &ls)) {
            __syncthreads();
            leaf_role<T, true>(n, A, lda, L, ldl, Dinv, k, kp, info, P0, P1, &ls);
        }
        return;
    }
    const int nb = (n + 63) / 64;
    int t = blockIdx.x, j = k;
    while (t >= nb - j) {  // tile t of the trapezoid, column by column
        t -= nb - j;
        ++j;
    }
    const int i = j + t;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = lane & 15,
              g = lane >> 4;
    const int rb = w & 3;
    const int crow = 64 * i + 16 * rb + l;  // C rows of this lane: block rb of tile i
    const int cb0 = 2 * (w >> 2);           // two column blocks per wave
    const Pair4 xp = fetch64(Dinv + (long) kp * 4096, tid);
    // waves 0 - 3: L(i, kp) into P0; waves 4 - 7: L(j, kp) into P1
    const int prow = 64 * (w < 4 ? i : j) + 16 * rb + l;
    double av[16];
    load_rows(A, lda, n, prow, kp, g, av);
    double cin[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = 64 * j + 16 * (cb0 + h) + 4 * r + g;
            cin[h][r] = (crow < n && col < n && crow >= col) ? (double) A[crow + (long) col * lda] : 0.0;
        }
    // workgroup 0 may write info while this one runs: one read for all threads, so that they
    // leave together
    if (tid == 0) bad = *info;
    stash64(P1, xp, tid);
    __syncthreads();
    {
        v4d p[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) p[c] = panel_block(P1, av, c, l, g);
        if (bad) return;
        __syncthreads();
        double(*P)[CH_LD] = (w < 4) ? P0 : P1;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int r = 0; r < 4; ++r) P[16 * c + 4 * r + g][16 * rb + l] = p[c][r];
            if (j == k && w < 4) store_panel(L, ldl, n, prow, kp, c, g, p[c]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int cb = cb0 + h;
        if (i == j && cb > rb) continue;
        const v4d c = rank64(P1, P0, cb, rb, l, g, (v4d){cin[h][0], cin[h][1], cin[h][2], cin[h][3]});
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = 64 * j + 16 * cb + 4 * r + g;
            if (crow < n && col < n && crow >= col) A[crow + (long) col * lda] = (T) c[r];
        }
    }
}

// L(i, kp) = A(i, kp) X^T for the tiles i = kp + 1 + blockIdx.x: the last panel of an
// outer block
template <typename T>
__global__ __launch_bounds__(CH_THREADS) void chol_panel_kernel(int n, const T *A, long lda, T *L, long ldl,
                                                                const double *Dinv, int kp, const int *info) {
    __shared__ __attribute__((aligned(16))) double X[64][CH_LD];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l = lane & 15, g = lane >> 4;
    const int row = 64 * (kp + 1 + blockIdx.x) + 16 * (w & 3) + l, ca = (w < 4) ? 0 : 1, cb = 3 - ca;
    const Pair4 xp = fetch64(Dinv + (long) kp * 4096, tid);
    double av[16];
    load_rows(A, lda, n, row, kp, g, av);
    const int bad = *info;
    stash64(X, xp, tid);
    __syncthreads();
    if (bad) return;
    store_panel(L, ldl, n, row, kp, ca, g, panel_block(X, av, ca, l, g));
    store_panel(L, ldl, n, row, kp, cb, g, panel_block(X, av, cb, l, g));
}

}  // namespace

// Matrices of up to CH_FLAT block columns are factored step by step over all their tiles;
// larger ones in outer blocks of CH_OUTER block columns, whose trailing update is one
// rank-(64 CH_OUTER) product: the part on the next outer block on s, the rest on the
// second stream beside the next block's steps.  The line lies where the step by step
// form's tiles (a rank-64 update each, with its panel blocks formed again) outgrow the
// chip: m = 2300 takes 1.0 ms in outer blocks and 0.8 ms flat, m = 8084 6.5 ms in outer
// blocks, where one flat step alone would hold 8000 tiles of 7 us on 256 CUs.  At
// m = 20000 the outer blocks take 55 ms (48 TF; 61 ms with outer blocks of 4, 57 of 6, 56
// of 8 and of 16), the paired rank-64 updates before them 105 ms.
constexpr int CH_FLAT = 48, CH_OUTER = 12;

template <typename T>
void potrf(hipStream_t s, int n, T *A, int lda, T *L, int ldl, double *Dinv, int *info, const LookAhead *la) {
    const int nb = (n + 63) / 64;
    auto step = [&](int k, int kp, int jEnd) {
        int tiles = 1;
        if (kp >= 0) {
            tiles = 0;
            for (int j = k; j < jEnd; ++j) tiles += nb - j;
        }
        chol_step_kernel<T><<<tiles, CH_THREADS, 0, s>>>(n, A, lda, L, ldl, Dinv, k, kp, jEnd, info);
    };
    if (nb <= CH_FLAT) {
        for (int k = 0; k < nb; ++k) step(k, k - 1, nb);
        return;
    }
    int ring = 0;
    bool s2dirty = false;
    hipEvent_t evB = nullptr;
    for (int o = 0; o < nb; o += CH_OUTER) {
        const int e = std::min(o + CH_OUTER, nb), e2 = std::min(e + CH_OUTER, nb);
        for (int k = o; k < e; ++k) step(k, (k > o) ? k - 1 : -1, e);
        if (e == nb) break;
        chol_panel_kernel<T><<<nb - e, CH_THREADS, 0, s>>>(n, A, lda, L, ldl, Dinv, e - 1, info);
        const int r0 = 64 * e, r2 = 64 * e2, c0 = 64 * o, K = 64 * (e - o);
        auto update = [&](hipStream_t st, int r, int cols) {
            gemm<T>(st, false, true, true, n - r, cols, K, (T) -1, L + r + (long) c0 * ldl, ldl, 0,
                    L + r + (long) c0 * ldl, ldl, 0, (T) 1, A + r + (long) r * lda, lda, 0, 1);
        };
        if (r2 < n && la) {
            hipEvent_t evP = la->ev[ring++ % LA_EVENTS];
            hipEventRecord(evP, s);
            hipStreamWaitEvent(la->s2, evP, 0);
        }
        if (s2dirty) {
            hipStreamWaitEvent(s, evB, 0);  // the previous update of these columns
            s2dirty = false;
        }
        update(s, r0, std::min(n, r2) - r0);
        if (r2 < n) {
            update(la ? la->s2 : s, r2, n - r2);
            if (la) {
                evB = la->ev[ring++ % LA_EVENTS];
                hipEventRecord(evB, la->s2);
                s2dirty = true;
            }
        }
    }
    if (s2dirty) hipStreamWaitEvent(s, evB, 0);
}

template void potrf<double>(hipStream_t, int, double *, int, double *, int, double *, int *, const LookAhead *);
template void potrf<float>(hipStream_t, int, float *, int, float *, int, double *, int *, const LookAhead *);

}  // namespace hdk
