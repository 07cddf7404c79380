// dev_common.h -- shared declarations of the gfx950 kernels and launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <cstdio>

#define HIP_OK(expr)                                                                    \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess) {                                                         \
            fprintf(stderr, "[hdsdp_amd] HIP error %s at %s:%d\n", hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                                \
            return HDSDP_RETCODE_FAILED;                                                \
        }                                                                               \
    } while (0)

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

namespace hdk {

// Sum over the 64 lanes of a wave, valid in lane 0: the additions of a shuffle-down tree
// (32, 16, 8, 4, 2, 1) with the lane exchanges of the VALU instead of LDS permutes (0.1 us a
// sum against 0.3).
__device__ inline double wave_tree_sum(double v) {
    auto half = [](double x, int step) {
        const unsigned lo = (unsigned) __double2loint(x), hi = (unsigned) __double2hiint(x);
        if (step == 32)
            return __hiloint2double((int) __builtin_amdgcn_permlane32_swap(hi, hi, false, false)[1],
                                    (int) __builtin_amdgcn_permlane32_swap(lo, lo, false, false)[1]);
        return __hiloint2double((int) __builtin_amdgcn_permlane16_swap(hi, hi, false, false)[1],
                                (int) __builtin_amdgcn_permlane16_swap(lo, lo, false, false)[1]);
    };
    v += half(v, 32);
    v += half(v, 16);
#define HDK_ROW_SHL(n)                                                                                       \
    v += __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x100 + n, 0xf, 0xf, true),            \
                          __builtin_amdgcn_mov_dpp(__double2loint(v), 0x100 + n, 0xf, 0xf, true))
    HDK_ROW_SHL(8);
    HDK_ROW_SHL(4);
    HDK_ROW_SHL(2);
    HDK_ROW_SHL(1);
#undef HDK_ROW_SHL
    return v;
}

// Four such sums at once, in lane 0 of each row of 16: s0, s2, s1, s3.  Two values share a
// register after the first exchange and all four after the second: 21 instructions
// instead of 72, the additions those of wave_tree_sum.
__device__ inline double wave_tree_sum4(double s0, double s1, double s2, double s3) {
    auto join32 = [](double x, double y) {  // lanes < 32: x(l) + x(l + 32), lanes >= 32 the same of y
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned) __double2loint(x), (unsigned) __double2loint(y), false,
                                                         false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned) __double2hiint(x), (unsigned) __double2hiint(y), false,
                                                         false);
        return __hiloint2double((int) hi[0], (int) lo[0]) + __hiloint2double((int) hi[1], (int) lo[1]);
    };
    const double x = join32(s0, s1), y = join32(s2, s3);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned) __double2loint(x), (unsigned) __double2loint(y), false,
                                                     false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned) __double2hiint(x), (unsigned) __double2hiint(y), false,
                                                     false);
    double v = __hiloint2double((int) hi[0], (int) lo[0]) + __hiloint2double((int) hi[1], (int) lo[1]);
#define HDK_ROW_SHL(n)                                                                                       \
    v += __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x100 + n, 0xf, 0xf, true),            \
                          __builtin_amdgcn_mov_dpp(__double2loint(v), 0x100 + n, 0xf, 0xf, true))
    HDK_ROW_SHL(8);
    HDK_ROW_SHL(4);
    HDK_ROW_SHL(2);
    HDK_ROW_SHL(1);
#undef HDK_ROW_SHL
    return v;
}
// which of the four sums a lane of wave_tree_sum4's result holds (lanes 0, 16, 32, 48)
__device__ inline int tree_sum4_slot(int lane) { return ((lane >> 5) & 1) | ((lane >> 3) & 2); }

__device__ inline float wave_tree_sum(float v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    return v;
}

constexpr int KSTEP = 16;  // k slab of the 128-wide GEMM tiles, granularity of skipped k ranges
constexpr int NB = 64;     // Cholesky / triangular-inverse block

// C = alpha * op(A) * op(B) + beta * C over `batch` problems (column-major).
// lower != 0 restricts the output to i >= j (tiles above the diagonal skipped).
// tri = 1 when op(B) is lower triangular, 2 when op(A) is, 3 when op(B) is upper
// triangular, 5 when op(A) is, 4 when op(A) is upper and op(B) lower: the k ranges that
// multiply the zero triangle are skipped (the stored zeros must be present).
template <typename T>
void gemm(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha,
          const T *A, int lda, long strideA, const T *B, int ldb, long strideB, T beta, T *C,
          int ldc, long strideC, int batch = 1, int tri = 0);

// W = Li^T Li, both triangles, for a lower-triangular n x n Li with zeros above the diagonal
void gram_lower(hipStream_t s, int n, const double *Li, double *W);

// gemm with the k range split into parts whose partial products go to work (P x M x N)
// and are summed in a fixed order, for products with few output tiles and long k
// (128-wide tiles fill the chip only with enough of them).  Falls back to gemm when
// work is null or too small for two parts.
// number of k parts gemm_splitk uses for this shape (1: no split)
int splitk_parts(int M, int N, long K, bool lower, int most = 32);
template <typename T>
void gemm_splitk(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha, const T *A,
                 int lda, const T *B, int ldb, T beta, T *C, int ldc, T *work, size_t workLen);

// P_z = alpha X_z^T X_z (lower, r x r, ld r, stride r^2) over `parts` k slices of kc (the
// last one kLast wide; multiples of 16) of the k panels X: entry (k, p) at (k / 16) slab +
// 16 p + k % 16, p up to whole tiles of 128.
void gram_panels(hipStream_t s, int r, int kc, int kLast, int parts, double alpha, const double *X, long slab,
                 double *P);
// A_z B_z^T (z < batch), operands of `rows` >= n rows: of the first n rows
// and columns the strictly lower part, packed by columns, and the diagonal, into dg + z sDg.
// slab = 0: packed entries into off + z K1; slab > 0: entry e into off[(e / 16) slab + 16 z +
// e % 16] (operands 16-byte aligned, even ld, whole tiles of rows).  tri as in gemm.
void gemm_nt_packed(hipStream_t s, int rows, int n, const double *A, int lda, long sA, const double *B, int ldb,
                    long sB, double *off, long K1, long slab, double *dg, long sDg, int batch, int tri);
// C = alpha * X^T Y + beta * C from bf16 split products on the matrix cores: each FP32
// operand split into `terms` bf16 terms (2: three products, ~16 bits; 3: six products,
// ~24 bits, FP32-equivalent), FP32 accumulation flushed into FP64 every 256 k.
// X: K x M (ldx), Y: K x N (ldy), column-major FP32; lower restricts C to i >= j.
// tri = 1 when Y(k, j) = 0 for k > j, 2 when X(k, i) = 0 for k > i (those k are skipped).
template <typename Tout>
void gemm_bf16s_tn(hipStream_t s, int terms, bool lower, int M, int N, int K, double alpha, const float *X, int ldx,
                   long sX, const float *Y, int ldy, long sY, double beta, Tout *C, int ldc, long sC, int batch = 1,
                   int tri = 0);

// A second stream and a ring of events for look-ahead factorisations.
constexpr int LA_EVENTS = 16;
struct LookAhead {
    hipStream_t s2;
    hipEvent_t ev[LA_EVENTS];
};

// Lower Cholesky A = L L^T of the n x n matrix A (lower triangle, destroyed), blocked by
// NB.  L (n x n, lower triangle written) and A are distinct.  Dinv: chol_dinv_len(n)
// doubles, the inverses of L's 64 x 64 diagonal blocks (column-major, zeros above the
// diagonal, the last one padded with the identity).  info: device int, set to 0 on
// success else failing column + 1.  With la, the bulk of each trailing update of a large
// matrix runs on la->s2 while the next block columns are factored on s; s has waited for
// s2 when the call returns.
inline size_t chol_dinv_len(size_t n) { return (n + NB - 1) / NB * NB * NB; }
template <typename T>
void potrf(hipStream_t s, int n, T *A, int lda, T *L, int ldl, double *Dinv, int *info, const LookAhead *la = nullptr);

// Linv = L^-1 for the lower-triangular n x n factor L (upper of Linv zeroed) with the
// inverses Dinv of its diagonal blocks.  work: n * n scratch.  With span (a power-of-two
// multiple of NB), only the diagonal blocks of span rows are inverted, each in its place.
template <typename T>
void trtri(hipStream_t s, int n, const T *L, int ldl, const double *Dinv, T *Linv, int ldi, T *work, int span = 0);

// A Cholesky factor L (lower triangle of an m x m matrix, whose upper triangle it may
// overwrite) as a preconditioner: prepare fills Li and LiT (m x m each, ld as L's), apply
// computes z = L^-T L^-1 r with tmp of m entries; r, z and tmp distinct.
template <typename T>
void solve_prepare(hipStream_t s, int m, T *L, int ld, const double *Dinv, T *Li, T *LiT);
template <typename T>
void solve_apply(hipStream_t s, int m, const T *L, int ld, const T *Li, const T *LiT, const T *r, T *z, T *tmp,
                 bool complete = false);
// Where prepare inverts diagonal blocks only, solve_complete extends Li and LiT to the whole
// inverse (m^3 / 3 flops) for apply with complete: half the launches per solve.
bool solve_in_blocks(int m);
template <typename T>
void solve_complete(hipStream_t s, int m, const T *L, int ld, T *Li, T *LiT);

// In-place LU with partial pivoting, P A = L U (L unit lower, U upper, both in A),
// blocked by 64 columns.  ipiv (device, m ints): row interchanged with row c at step c,
// 0-based; info (device int, cleared by the caller): 0, or the first zero-pivot column + 1.
void lu_factor(hipStream_t s, int m, double *A, int lda, int *ipiv, int *info);
// x = A^-1 b from lu_factor's factors and perm, the composed interchanges (P b = b[perm]).
// x and b are distinct m-vectors.
void lu_solve(hipStream_t s, int m, const double *A, int lda, const int *perm, const double *b, double *x);

// y[j] = alpha * sum_{i in rows(j)} A[i + j*lda] x[i] + beta * y[j] for j < ncols,
// rows(j) = [0, m) (tri 0), [j, m) (tri 1, lower), [0, j] (tri 2, upper).
template <typename T>
void coldot(hipStream_t s, int m, int ncols, int tri, T alpha, const T *A, int lda, const T *x, T beta, T *y);

// y = M x for symmetric M read only in its lower triangle (one pass, tile partials
// added in a fixed order); work: symv_lower_work(m) doubles.
constexpr int SYMV_R = 512, SYMV_C = 256;
size_t symv_lower_work(int m);
void symv_lower(hipStream_t s, int m, const double *M, long ldm, const double *x, double *y, double *work);

// A[upper] = A[lower]^T for the n x n matrix.
template <typename T>
void mirror_lower(hipStream_t s, int n, T *A, int lda);
// B = A^T (n x n).
template <typename T>
void transpose(hipStream_t s, int n, const T *A, int lda, T *B, int ldb);
// Zero the strictly upper triangle.
template <typename T>
void zero_upper(hipStream_t s, int n, T *A, int lda);

void fill(hipStream_t s, double *x, long n, double v);
void fill_f(hipStream_t s, float *x, long n, float v);
void copy_lower(hipStream_t s, int n, const double *A, int lda, double *B, int ldb);
void convert_lower_to_float(hipStream_t s, int n, const double *A, int lda, float *B, int ldb);
// B = lower(diag(sc) A diag(sc) + shift I) in FP32, zeros above the diagonal
void convert_lower_scaled(hipStream_t s, int n, const double *A, int lda, const double *sc, double shift, float *B,
                          int ldb);
void add_diag(hipStream_t s, int n, double *A, int lda, const double *d, double scalar);
// out[0] = 2 * sum log A_jj
void logdet_diag(hipStream_t s, int n, const double *A, int lda, double *out);

}  // namespace hdk
