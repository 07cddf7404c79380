// dense.hip -- dense linear algebra for the dual slack S and the Schur matrix M
// on gfx950: MFMA GEMM, blocked Cholesky, recursive triangular inverse, GEMV.
//
// GEMM tiles are 32, 64 or 128 wide per workgroup of four 64-wide waves; each wave owns a
// quadrant as MFMA 16x16 accumulators and the k-dimension is staged through LDS in
// slabs.  FP64 uses v_mfma_f64_16x16x4_f64, FP32
// v_mfma_f32_16x16x4_f32; both take one A and one B element per lane,
//   A[i][k] at lane i + 16 k,  B[k][j] at lane j + 16 k,
// and return four accumulator elements per lane in different row orders
// (measured on gfx950):
//   FP32: D[i][j] at lane j + 16 (i / 4), element i % 4;
//   FP64: D[i][j] at lane j + 16 (i % 4), element i / 4.
#include "dev_common.h"

namespace hdk {

template <typename T>
struct Mfma;

template <>
struct Mfma<double> {
    typedef v4d acc_t;
    // row of accumulator element r held by lane group g = lane / 16
    __device__ static inline int row(int g, int r) { return 4 * r + g; }
    __device__ static inline acc_t op(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};

template <>
struct Mfma<float> {
    typedef v4f acc_t;
    __device__ static inline int row(int g, int r) { return 4 * g + r; }
    __device__ static inline acc_t op(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// k range of one output tile when an operand is triangular: tri 1 = op(B) lower
// (B(k, j) = 0 for k < j), tri 2 = op(A) lower (A(i, k) = 0 for k > i), tri 3 = op(B) upper
// (B(k, j) = 0 for k > j), tri 4 = op(A) upper and op(B) lower (zero for k < max(i, j)),
// tri 5 = op(A) upper.  Only exact zeros are skipped, so the result is the same as
// the full product.
__device__ inline void tri_krange(int tri, int i0, int j0, int tile, int K, int &kLo, int &kHi) {
    kLo = 0;
    kHi = K;
    if (tri == 1) kLo = (j0 / KSTEP) * KSTEP;
    if (tri == 4) kLo = (max(i0, j0) / KSTEP) * KSTEP;
    if (tri == 5) kLo = (i0 / KSTEP) * KSTEP;
    if (tri == 2) kHi = (i0 + tile < K) ? i0 + tile : K;
    if (tri == 3) kHi = (j0 + tile < K) ? j0 + tile : K;
}

// Output tile of this workgroup.  With lin != 0 (lower products with as many tile rows
// as tile columns) blockIdx.x runs over the lower tiles only, t = x (x + 1) / 2 + y with
// y <= x: consecutive workgroups go to consecutive XCDs, so every XCD gets the same
// share of the triangle (a 2-D grid gives tile column x to XCD x mod 8, and the
// columns near the diagonal end hold unequal work).
//
// With tri == 2 (op(A) lower: the work of a tile grows with its row; 4 and 5 shrink with it) the tile row of
// a 2-D grid is rotated by the other grid coordinates: workgroup x + gridDim.x (y + ...)
// goes to XCD (x + ...) mod 8, so with 8k tile rows XCD x would receive every tile of
// row x (the heaviest rows all on one XCD); the rotation gives each XCD every row.
__device__ inline void tile_xy(int lin, int &bx, int &by, int tri = 0) {
    if (!lin) {
        bx = blockIdx.x;
        by = blockIdx.y;
        if (tri == 2 || tri >= 4) bx = (int) ((blockIdx.x + blockIdx.y + blockIdx.z) % gridDim.x);
        return;
    }
    // a triangular operand makes the later tiles the longer ones (tri 4: the earlier): those go first
    const int t = (tri && tri != 4) ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    int x = (int) ((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((x + 1) * (x + 2) / 2 <= t) ++x;
    while (x * (x + 1) / 2 > t) --x;
    bx = x;
    by = t - x * (x + 1) / 2;
}

// 128 x 128 tiles for large products: four waves, each a 64 x 64 quadrant as 4 x 4
// MFMA 16x16 accumulators; k slabs of 16 double-buffered in LDS so the global
// loads of slab s + 1 are in flight while slab s is multiplied (one barrier per slab).
constexpr int BT = 128, BPAD = 16;
static_assert(4 * 16 * 65 <= 2 * KSTEP * (BT + BPAD), "epilogue staging must fit in the k-slab buffers");

template <typename T, bool TA, bool TB, bool CHECK>
__device__ inline void big_load(const T *A, int lda, const T *B, int ldb, int M, int N, int K, int i0, int j0,
                                int k0, int tid, T (&ra)[8], T (&rb)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        int i, k;
        if (!TA) { k = tid >> 4; i = (tid & 15) * 8 + u; } else { i = tid >> 1; k = (tid & 1) * 8 + u; }
        const int gi = i0 + i, gk = k0 + k;
        const T *pa = TA ? A + gk + (long) gi * lda : A + gi + (long) gk * lda;
        ra[u] = (!CHECK || (gi < M && gk < K)) ? *pa : (T) 0;
        int j, kb;
        if (TB) { kb = tid >> 4; j = (tid & 15) * 8 + u; } else { j = tid >> 1; kb = (tid & 1) * 8 + u; }
        const int gj = j0 + j, gkb = k0 + kb;
        const T *pb = TB ? B + gj + (long) gkb * ldb : B + gkb + (long) gj * ldb;
        rb[u] = (!CHECK || (gj < N && gkb < K)) ? *pb : (T) 0;
    }
}

// Interior slab with 16-byte loads (FP64; leading dimensions, strides and base
// addresses even, checked by the launcher).  Each thread moves 8 elements of each
// operand as 4 pairs:
//   k-contiguous operand (A with TA, B without TB): row tid / 2, k = 8 (tid % 2) + 2u
//   row-contiguous operand: k = tid / 16, rows 2 (tid % 16) + 32u, so that the 16
//   lanes of one k read 256 consecutive bytes per instruction.
typedef double dpair __attribute__((ext_vector_type(2)));

template <bool TA, bool TB>
__device__ inline void big_load_vec(const double *A, int lda, const double *B, int ldb, int i0, int j0, int k0,
                                    int tid, double (&ra)[8], double (&rb)[8]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        dpair va, vb;
        if (TA) {
            const int i = tid >> 1, k = (tid & 1) * 8 + 2 * u;
            va = *reinterpret_cast<const dpair *>(A + (k0 + k) + (long) (i0 + i) * lda);
        } else {
            const int k = tid >> 4, i = 2 * (tid & 15) + 32 * u;
            va = *reinterpret_cast<const dpair *>(A + (i0 + i) + (long) (k0 + k) * lda);
        }
        if (!TB) {
            const int j = tid >> 1, k = (tid & 1) * 8 + 2 * u;
            vb = *reinterpret_cast<const dpair *>(B + (k0 + k) + (long) (j0 + j) * ldb);
        } else {
            const int k = tid >> 4, j = 2 * (tid & 15) + 32 * u;
            vb = *reinterpret_cast<const dpair *>(B + (j0 + j) + (long) (k0 + k) * ldb);
        }
        ra[2 * u] = va.x;
        ra[2 * u + 1] = va.y;
        rb[2 * u] = vb.x;
        rb[2 * u + 1] = vb.y;
    }
}

template <bool TA, bool TB>
__device__ inline void big_store_vec(double (*As)[BT + BPAD], double (*Bs)[BT + BPAD], int tid, const double (&ra)[8],
                                     const double (&rb)[8]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (TA) {
            const int i = tid >> 1, k = (tid & 1) * 8 + 2 * u;
            As[k][i] = ra[2 * u];
            As[k + 1][i] = ra[2 * u + 1];
        } else {
            const int k = tid >> 4, i = 2 * (tid & 15) + 32 * u;
            *reinterpret_cast<dpair *>(&As[k][i]) = (dpair){ra[2 * u], ra[2 * u + 1]};
        }
        if (!TB) {
            const int j = tid >> 1, k = (tid & 1) * 8 + 2 * u;
            Bs[k][j] = rb[2 * u];
            Bs[k + 1][j] = rb[2 * u + 1];
        } else {
            const int k = tid >> 4, j = 2 * (tid & 15) + 32 * u;
            *reinterpret_cast<dpair *>(&Bs[k][j]) = (dpair){rb[2 * u], rb[2 * u + 1]};
        }
    }
}

// one k slab of the tile into registers (returns whether the vector layout was used);
// the bounds checks are dropped for interior slabs
template <typename T, bool TA, bool TB, bool VEC>
__device__ inline bool big_fetch(const T *A, int lda, const T *B, int ldb, int M, int N, int K, int i0, int j0,
                                 int k0, int tid, T (&ra)[8], T (&rb)[8]) {
    if (i0 + BT <= M && j0 + BT <= N && k0 + KSTEP <= K) {
        if constexpr (VEC) {
            big_load_vec<TA, TB>(A, lda, B, ldb, i0, j0, k0, tid, ra, rb);
            return true;
        }
        big_load<T, TA, TB, false>(A, lda, B, ldb, M, N, K, i0, j0, k0, tid, ra, rb);
    } else {
        big_load<T, TA, TB, true>(A, lda, B, ldb, M, N, K, i0, j0, k0, tid, ra, rb);
    }
    return false;
}

template <typename T, bool TA, bool TB>
__device__ inline void big_store(T (*As)[BT + BPAD], T (*Bs)[BT + BPAD], int tid, const T (&ra)[8],
                                 const T (&rb)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        int i, k;
        if (!TA) { k = tid >> 4; i = (tid & 15) * 8 + u; } else { i = tid >> 1; k = (tid & 1) * 8 + u; }
        As[k][i] = ra[u];
        int j, kb;
        if (TB) { kb = tid >> 4; j = (tid & 15) * 8 + u; } else { j = tid >> 1; kb = (tid & 1) * 8 + u; }
        Bs[kb][j] = rb[u];
    }
}

// PACK 1 (square lower products with beta = 0): the strictly lower part of the result's
// first ldc rows and columns goes to C packed by columns and the diagonal to dg (stride
// sDg), as pack_lower stores them.
// PANEL: both operands are read from k panels of 16, entry (k, i) at (k / 16) slab + 16 i +
// k % 16, so that a slab of a tile is 16 KB of consecutive memory; K a multiple of 16,
// rows of whole tiles present.
template <typename T, bool TA, bool TB, bool LOWER, bool VEC, int PACK = 0, bool PANEL = false>
__global__ __launch_bounds__(256) void gemm_big_kernel(int M, int N, int K, T alpha, const T *A, int lda, long sA,
                                                       const T *B, int ldb, long sB, T beta, T *C, int ldc,
                                                       long sC, int tri, int lin, int kLast, T *dg = nullptr,
                                                       long sDg = 0, long slab = 0) {
    typedef typename Mfma<T>::acc_t acc_t;
    if (kLast > 0 && blockIdx.z == gridDim.z - 1) K = kLast;  // ragged last k part of a split product
    int bx, by;
    tile_xy(lin, bx, by, tri);
    const int i0 = bx * BT, j0 = by * BT;
    if (LOWER && i0 + BT - 1 < j0) return;
    int kLo, kHi;
    tri_krange(tri, i0, j0, BT, K, kLo, kHi);
    A += (long) blockIdx.z * sA;
    B += (long) blockIdx.z * sB;
    C += (long) blockIdx.z * sC;
    __shared__ __attribute__((aligned(16))) T As[2][KSTEP][BT + BPAD];
    __shared__ __attribute__((aligned(16))) T Bs[2][KSTEP][BT + BPAD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 64, wj = (wave >> 1) * 64;
    const int lr = lane & 15, lk = lane >> 4;
    acc_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = (acc_t){0, 0, 0, 0};
    T ra[8], rb[8];
    auto stash = [&](int buf, bool vec) {
        if constexpr (VEC) {
            if (vec) {
                big_store_vec<TA, TB>(As[buf], Bs[buf], tid, ra, rb);
                return;
            }
        }
        big_store<T, TA, TB>(As[buf], Bs[buf], tid, ra, rb);
    };
    auto fetch = [&](int k0) {
        if constexpr (PANEL) {
            const long at = (long) (k0 / KSTEP) * slab;
            big_load_vec<TA, TB>(A + at, KSTEP, B + at, KSTEP, i0, j0, 0, tid, ra, rb);
            return true;
        } else {
            return big_fetch<T, TA, TB, VEC>(A, lda, B, ldb, M, N, K, i0, j0, k0, tid, ra, rb);
        }
    };
    bool vec = fetch(kLo);
    stash(0, vec);
    __syncthreads();
    const int nslab = (kHi - kLo + KSTEP - 1) / KSTEP;
    // the quadrants that start a half tile earlier have a triangular operand's zeros in the
    // last half tile of the k range: those waves skip its products
    const int kWave = __builtin_amdgcn_readfirstlane((tri == 2 && wi == 0) ? i0 + 64 : (tri == 3 && wj == 0) ? j0 + 64
                                                                                                             : K);
    for (int sl = 0; sl < nslab; ++sl) {
        const int cur = sl & 1;
        const bool more = sl + 1 < nslab;
        if (more) vec = fetch(kLo + (sl + 1) * KSTEP);
        if (kLo + sl * KSTEP < kWave)
#pragma unroll
        for (int kk = 0; kk < KSTEP; kk += 4) {
            T af[4], bf[4];
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                af[f] = As[cur][kk + lk][wi + 16 * f + lr];
                bf[f] = Bs[cur][kk + lk][wj + 16 * f + lr];
            }
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = Mfma<T>::op(af[a], bf[b], acc[a][b]);
        }
        if (more) stash(cur ^ 1, vec);
        __syncthreads();
    }
    // Epilogue: each wave stages its 64 x 64 quadrant through LDS (the k-slab buffers,
    // free after the last barrier) 16 columns at a time, so that lane q reads and
    // writes row q of C: 64 consecutive rows per column, coalesced.
    T (*stage)[65] = reinterpret_cast<T (*)[65]>(&As[0][0][0]) + wave * 16;
    const int i = i0 + wi + lane;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) stage[lr][a * 16 + Mfma<T>::row(lk, r)] = acc[a][b][r];
        if constexpr (PACK != 0) {
            const long n = ldc;
#pragma unroll
            for (int cc = 0; cc < 16; ++cc) {
                const long j = j0 + wj + b * 16 + cc;
                if (i >= n || j >= n || i < j) continue;
                const T v = alpha * stage[cc][lane];
                const long e = j * n - j * (j + 1) / 2 + (i - j - 1);
                if (i == j) dg[(long) blockIdx.z * sDg + i] = v;
                else C[e] = v;
            }
            continue;
        }
        // all loads of the strip are issued before any store (C may alias nothing,
        // but the compiler cannot know that)
        T cin[16];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
            const int j = j0 + wj + b * 16 + cc;
            const bool ok = i < M && j < N && (!LOWER || i >= j);
            cin[cc] = (ok && beta != (T) 0) ? C[i + (long) j * ldc] : (T) 0;
        }
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
            const int j = j0 + wj + b * 16 + cc;
            if (i < M && j < N && (!LOWER || i >= j)) C[i + (long) j * ldc] = alpha * stage[cc][lane] + beta * cin[cc];
        }
    }
}

// 16-byte loads need even leading dimensions, strides and addresses
template <typename T>
static bool vec_ok(const T *A, long lda, long sA, const T *B, long ldb, long sB) {
    return sizeof(T) == 8 && lda % 2 == 0 && ldb % 2 == 0 && sA % 2 == 0 && sB % 2 == 0 &&
           ((uintptr_t) A % 16) == 0 && ((uintptr_t) B % 16) == 0;
}

// 128-wide tile launch; batch z multiplies K-wide slices at strides sA, sB (the last
// one kLast wide when kLast > 0)
template <typename T>
static void gemm_big(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha, const T *A,
                     int lda, long strideA, const T *B, int ldb, long strideB, T beta, T *C, int ldc, long strideC,
                     int batch, int tri, int kLast) {
    const int mt = (M + BT - 1) / BT, nt = (N + BT - 1) / BT;
    const int lin = (lower && mt == nt) ? 1 : 0;
    dim3 bgrid(lin ? mt * (mt + 1) / 2 : mt, lin ? 1 : nt, batch);
    const bool vec = vec_ok<T>(A, lda, strideA, B, ldb, strideB);
#define HDK_GEMM_BIG(ta, tb, lo)                                                                                 \
    if (transA == ta && transB == tb && lower == lo) {                                                           \
        if (vec)                                                                                                 \
            gemm_big_kernel<T, ta, tb, lo, sizeof(T) == 8><<<bgrid, 256, 0, s>>>(                                \
                M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, tri, lin, kLast);       \
        else                                                                                                     \
            gemm_big_kernel<T, ta, tb, lo, false><<<bgrid, 256, 0, s>>>(M, N, K, alpha, A, lda, strideA, B, ldb, \
                                                                        strideB, beta, C, ldc, strideC, tri,     \
                                                                        lin, kLast);                             \
        return;                                                                                                  \
    }
    HDK_GEMM_BIG(false, false, false)
    HDK_GEMM_BIG(false, true, false)
    HDK_GEMM_BIG(true, false, false)
    HDK_GEMM_BIG(true, true, false)
    HDK_GEMM_BIG(false, false, true)
    HDK_GEMM_BIG(false, true, true)
    HDK_GEMM_BIG(true, false, true)
    HDK_GEMM_BIG(true, true, true)
#undef HDK_GEMM_BIG
}

// 64- and 32-wide tiles (TI) of four waves, each a quadrant of F x F MFMA blocks, F = TI / 32,
// with slabs of 32 or 64 k.
//
// 32-wide tiles serve products that leave CUs idle on 64-wide ones (the levels of a
// triangular inverse, S^-1 of a small block, the k parts of a rank-m update with few
// tiles): on 64-wide tiles such a product is bound by the MFMA chain of its few tiles, 0.43 us
// per 16 k whatever the rest of the chip does; a 32-wide tile takes a quarter of it on four
// times the workgroups, and pays a load latency once per 64 k.
//
// MFMA rows are tile columns, so that a wave loads and stores 16 consecutive rows.  Each
// operand is staged in its own order: rows consecutive as [k][TI + 16], k consecutive as
// [row][slab + 2], both free of bank conflicts in the fragment reads.  The slab sits in LDS
// once (40 to 50 KB, three workgroups per CU); the next one is in flight in registers
// while it is multiplied.  Every output sums its k in ascending order whatever the tile, so
// the choice of one does not change a bit.  The last batch entry may have fewer rows
// (mLast > 0) and a shorter k (kLast > 0).  PACK: the strictly lower part of a square result
// goes to C packed by columns (1) or in k panels (2: packed entry e of matrix z at
// C[(e / 16) slab + 16 z + e % 16]) and its diagonal to dg (beta = 0).
template <int TI>
struct MidTile {
    static constexpr int TK = (TI == 32) ? 64 : 32, LR = TI + 16, LK = TK + 2, F = TI / 32;
    static constexpr int PER = TI * TK / 256;  // elements of a slab per thread
};

template <typename T, bool KC, int TI>
__device__ inline void mid_fetch(const T *X, long ldx, int rows, int K, int r0, int k0, int tid,
                                 T (&v)[MidTile<TI>::PER]) {
    constexpr int TK = MidTile<TI>::TK;
#pragma unroll
    for (int u = 0; u < MidTile<TI>::PER; ++u) {
        // addresses clamped into the operand; the k beyond K are zeroed in mid_stash
        const int r = min(r0 + (KC ? tid / TK + 256 / TK * u : tid % TI), rows - 1);
        const int k = min(k0 + (KC ? tid % TK : tid / TI + 256 / TI * u), K - 1);
        v[u] = KC ? X[k + r * ldx] : X[r + k * ldx];
    }
}

template <typename T, bool KC, int TI>
__device__ inline void mid_stash(T *S, int K, int k0, int tid, const T (&v)[MidTile<TI>::PER]) {
    constexpr int TK = MidTile<TI>::TK;
#pragma unroll
    for (int u = 0; u < MidTile<TI>::PER; ++u) {
        const int r = KC ? tid / TK + 256 / TK * u : tid % TI, k = KC ? tid % TK : tid / TI + 256 / TI * u;
        S[KC ? r * MidTile<TI>::LK + k : k * MidTile<TI>::LR + r] = (k0 + k < K) ? v[u] : (T) 0;
    }
}

template <typename T, bool TA, bool TB, bool LOWER, int TI, int PACK = 0>
__global__ __launch_bounds__(256) void gemm_mid_kernel(int M, int N, int K, T alpha, const T *A, int lda, long sA,
                                                       const T *B, int ldb, long sB, T beta, T *C, int ldc, long sC,
                                                       int tri, int lin, int mLast, int kLast, T *dg = nullptr,
                                                       long sDg = 0, long slab = 0) {
    typedef MidTile<TI> G;
    constexpr int F = G::F, TK = G::TK, LR = G::LR, LK = G::LK;
    constexpr bool KCA = TA, KCB = !TB;  // operand consecutive along k
    __shared__ T As[KCA ? TI * LK : TK * LR], Bs[KCB ? TI * LK : TK * LR];
    if (blockIdx.z == gridDim.z - 1) {
        if (mLast > 0) M = mLast;
        if (kLast > 0) K = kLast;
    }
    int bx, by;
    tile_xy(lin, bx, by, tri);
    const int i0 = bx * TI, j0 = by * TI;
    if (i0 >= M || j0 >= N || (LOWER && i0 + TI - 1 < j0)) return;
    int kLo, kHi;
    tri_krange(tri, i0, j0, TI, K, kLo, kHi);
    A += (long) blockIdx.z * sA;
    B += (long) blockIdx.z * sB;
    C += (long) blockIdx.z * sC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * (TI / 2), wj = (wave >> 1) * (TI / 2), lr = lane & 15, lk = lane >> 4;
    typename Mfma<T>::acc_t acc[F][F];
    T cin[F][F][4];
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
        for (int b = 0; b < F; ++b) {
            acc[a][b] = (typename Mfma<T>::acc_t){0, 0, 0, 0};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + wi + 16 * a + lr, j = j0 + wj + 16 * b + Mfma<T>::row(lk, r);
                cin[a][b][r] = (beta != (T) 0 && i < M && j < N && (!LOWER || i >= j)) ? C[i + (long) j * ldc] : (T) 0;
            }
        }
    T ra[G::PER], rb[G::PER];
    if (kLo < kHi) {
        mid_fetch<T, KCA, TI>(A, lda, M, K, i0, kLo, tid, ra);
        mid_fetch<T, KCB, TI>(B, ldb, N, K, j0, kLo, tid, rb);
    }
    for (int k0 = kLo; k0 < kHi; k0 += TK) {
        mid_stash<T, KCA, TI>(As, K, k0, tid, ra);
        mid_stash<T, KCB, TI>(Bs, K, k0, tid, rb);
        __syncthreads();
        if (k0 + TK < kHi) {
            mid_fetch<T, KCA, TI>(A, lda, M, K, i0, k0 + TK, tid, ra);
            mid_fetch<T, KCB, TI>(B, ldb, N, K, j0, k0 + TK, tid, rb);
        }
#pragma unroll
        for (int kk = 0; kk < TK; kk += 4) {
            T af[F], bf[F];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const int i = wi + 16 * f + lr, j = wj + 16 * f + lr, k = kk + lk;
                af[f] = As[KCA ? i * LK + k : k * LR + i];
                bf[f] = Bs[KCB ? j * LK + k : k * LR + j];
            }
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int b = 0; b < F; ++b) acc[a][b] = Mfma<T>::op(bf[b], af[a], acc[a][b]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
        for (int b = 0; b < F; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + wi + 16 * a + lr, j = j0 + wj + 16 * b + Mfma<T>::row(lk, r);
                if (i >= M || j >= N || (LOWER && i < j)) continue;
                if (PACK) {
                    if (i == j) dg[blockIdx.z * sDg + i] = alpha * acc[a][b][r];
                    else {
                        const long q = (long) j * N - (long) j * (j + 1) / 2 + (i - j - 1);
                        C[PACK == 1 ? q : (q >> 4) * slab + 16 * blockIdx.z + (q & 15)] = alpha * acc[a][b][r];
                    }
                } else {
                    C[i + (long) j * ldc] = alpha * acc[a][b][r] + beta * cin[a][b][r];
                }
            }
}

template <int TI, typename T>
static void gemm_mid(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha, const T *A,
                     int lda, long strideA, const T *B, int ldb, long strideB, T beta, T *C, int ldc, long strideC,
                     int batch, int tri, int mLast = 0, int kLast = 0) {
    const int mt = (M + TI - 1) / TI, nt = (N + TI - 1) / TI;
    const int lin = (lower && mt == nt) ? 1 : 0;
    const dim3 grid(lin ? mt * (mt + 1) / 2 : mt, lin ? 1 : nt, batch);
#define HDK_GEMM_MID(ta, tb, lo)                                                                               \
    if (transA == ta && transB == tb && lower == lo) {                                                         \
        gemm_mid_kernel<T, ta, tb, lo, TI><<<grid, 256, 0, s>>>(M, N, K, alpha, A, lda, strideA, B, ldb,       \
                                                                strideB, beta, C, ldc, strideC, tri, lin,      \
                                                                mLast, kLast);                                 \
        return;                                                                                                \
    }
    HDK_GEMM_MID(false, false, false)
    HDK_GEMM_MID(false, true, false)
    HDK_GEMM_MID(true, false, false)
    HDK_GEMM_MID(true, true, false)
    HDK_GEMM_MID(false, false, true)
    HDK_GEMM_MID(false, true, true)
    HDK_GEMM_MID(true, false, true)
    HDK_GEMM_MID(true, true, true)
#undef HDK_GEMM_MID
}

// Tile width of a product: the least modelled time
//   k per tile x time per k and tile x tiles per CU (rounded up)
// over the three widths.  A CU's workgroups share its matrix cores, so the time of a width
// grows with the tiles per CU and not below what its latencies take alone (1.3, 1.7, 2.2
// tiles' worth); a tile of a triangular product walks half its k and half a tile on average;
// prologue and epilogue cost as much as 96 and 32 k; the bounds-checked loads of ragged
// 128-wide tiles cost 0.8 of a tile more, unaligned operands a fifth.  Measured on MI355X,
// us at 32, 64 and 128: 500^3 14.6, 34.5, 109; 1000^3 67, 67, 218; 1300^3 137, 127, 262;
// 4000^3 2967, 2473, 2231; lower 4000^3 1480, 1218, 1670; lower 8000^2 x 768 1177, 951, 863;
// 8000 x 768 x 768 lower 241, 208, 237; 450 triangular products of n = 300 540, 433, 709, of
// n = 200 211, 238, 334; 16 lower k parts 450^2 x 2800 268, 338, 484.
static int pick_tile(int M, int N, int K, bool lower, int batch, int tri, bool vec) {
    const int width[3] = {32, 64, 128};
    const double perK[3] = {0.0137, 0.041, 0.125}, alone[3] = {2.2, 1.7, 1.3}, extra[3] = {32, 32, 96};
    int best = 64;
    double tBest = 1e300;
    for (int v = 0; v < 3; ++v) {
        const int t = width[v];
        const long mt = (M + t - 1) / t, nt = (N + t - 1) / t, c = std::min(mt, nt);
        const long tiles = (lower ? mt * nt - c * (c - 1) / 2 : mt * nt) * batch;
        const double depth = std::max(alone[v], (double) ((tiles + 255) / 256));
        const double k = (tri == 0) ? K : (tri == 4) ? (K + t) / 3.0 : std::min<double>(K, (K + t) / 2.0);
        double time = perK[v] * depth * (k + extra[v]);
        if (t == 128) {
            const double ragged = 1.0 - (double) (M / t) * (N / t) / (double) (mt * nt);
            time *= (1.0 + 0.8 * ragged) * (vec ? 1.0 : 1.2);
        }
        if (time < tBest) {
            tBest = time;
            best = t;
        }
    }
    return best;
}

template <typename T>
void gemm(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha, const T *A,
          int lda, long strideA, const T *B, int ldb, long strideB, T beta, T *C, int ldc, long strideC,
          int batch, int tri) {
    if (M <= 0 || N <= 0 || batch <= 0) return;
    const int t = pick_tile(M, N, K, lower, batch, tri, vec_ok<T>(A, lda, strideA, B, ldb, strideB));
    if (t == 128)
        gemm_big<T>(s, transA, transB, lower, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc,
                    strideC, batch, tri, 0);
    else if (t == 64)
        gemm_mid<64, T>(s, transA, transB, lower, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc,
                        strideC, batch, tri);
    else
        gemm_mid<32, T>(s, transA, transB, lower, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc,
                        strideC, batch, tri);
}

template void gemm<double>(hipStream_t, bool, bool, bool, int, int, int, double, const double *, int, long,
                           const double *, int, long, double, double *, int, long, int, int);
template void gemm<float>(hipStream_t, bool, bool, bool, int, int, int, float, const float *, int, long,
                          const float *, int, long, float, float *, int, long, int, int);

// W = Li^T Li for a lower-triangular Li (n x n, zeros above): entry (i, j) sums k >= max(i, j)
// only, n^3 / 3 multiply-adds, and is symmetric to the bit, so beyond the 32-wide tiles the
// lower half is formed and mirrored (n^3 / 6).  n = 2000: 83 us, the full product 366.
void gram_lower(hipStream_t s, int n, const double *Li, double *W) {
    const bool half = pick_tile(n, n, n, false, 1, 4, n % 2 == 0) > 32;
    gemm<double>(s, true, false, half, n, n, n, 1.0, Li, n, 0, Li, n, 0, 0.0, W, n, 0, 1, 4);
    if (half) mirror_lower<double>(s, n, W, n);
}

// P_z = alpha X_z^T X_z (lower, r x r, ld r, stride r^2) over the k slices z of kc (the
// last one kLast wide) of the k panels X (PANEL above; slab doubles per 16 k)
void gram_panels(hipStream_t s, int r, int kc, int kLast, int parts, double alpha, const double *X, long slab,
                 double *P) {
    const int nt = (r + BT - 1) / BT;
    gemm_big_kernel<double, true, false, true, true, 0, true><<<dim3(nt * (nt + 1) / 2, 1, parts), 256, 0, s>>>(
        r, r, kc, alpha, X, 0, kc / KSTEP * slab, X, 0, kc / KSTEP * slab, 0.0, P, r, (long) r * r, 0, 1, kLast,
        nullptr, 0, slab);
}

// C_z = A_z B_z^T for z < batch, lower triangle, packed (PACK above); tri as in gemm.  k panels
// (operands of whole 128-wide tiles, n >= 512) are stored by the 64-wide tiles, whose triangle
// of tiles and k ranges wastes less: T_p = U_p L^-T, us at 64 and 128: 60 of n = 512 119 and 151,
// of 1024 599 and 691, 28 of 1536 804 and 887, 16 of 2048 1038 and 1134.
void gemm_nt_packed(hipStream_t s, int rows, int n, const double *A, int lda, long sA, const double *B, int ldb,
                    long sB, double *off, long K1, long slab, double *dg, long sDg, int batch, int tri) {
    const bool vec = vec_ok<double>(A, lda, sA, B, ldb, sB);
    const int t = (slab > 0) ? 64 : pick_tile(n, n, n, true, batch, tri, vec);
    if (t < 128) rows = n;
    const int nt = (rows + t - 1) / t, K = std::min(rows, (n + KSTEP - 1) / KSTEP * KSTEP);
    const dim3 grid(nt * (nt + 1) / 2, 1, batch);
    if (slab > 0)
        gemm_mid_kernel<double, false, true, true, 64, 2><<<grid, 256, 0, s>>>(
            n, n, n, 1.0, A, lda, sA, B, ldb, sB, 0.0, off, n, 0, tri, 1, 0, 0, dg, sDg, slab);
    else if (t == 32)
        gemm_mid_kernel<double, false, true, true, 32, 1><<<grid, 256, 0, s>>>(
            n, n, n, 1.0, A, lda, sA, B, ldb, sB, 0.0, off, n, K1, tri, 1, 0, 0, dg, sDg);
    else if (t == 64)
        gemm_mid_kernel<double, false, true, true, 64, 1><<<grid, 256, 0, s>>>(
            n, n, n, 1.0, A, lda, sA, B, ldb, sB, 0.0, off, n, K1, tri, 1, 0, 0, dg, sDg);
    else if (vec)
        gemm_big_kernel<double, false, true, true, true, 1><<<grid, 256, 0, s>>>(
            rows, rows, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, off, n, K1, tri, 1, 0, dg, sDg);
    else
        gemm_big_kernel<double, false, true, true, false, 1><<<grid, 256, 0, s>>>(
            rows, rows, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, off, n, K1, tri, 1, 0, dg, sDg);
}

// ---- split-K ---------------------------------------------------------------------

// C(i, j) = alpha sum_p P_p(i, j) + beta C(i, j) over the P partial products (ld M),
// i >= j only when lower.  Partials are summed in index order.
template <typename T>
__global__ void splitk_reduce_kernel(int M, int N, int P, T alpha, const T *W, T beta, T *C, int ldc, int lower) {
    const long total = (long) M * N, mn = total;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < total; e += (long) gridDim.x * blockDim.x) {
        const int i = (int) (e % M), j = (int) (e / M);
        if (lower && i < j) continue;
        T acc = W[e];
        for (int p = 1; p < P; ++p) acc += W[e + p * mn];
        T *c = C + i + (long) j * ldc;
        *c = (beta == (T) 0) ? alpha * acc : alpha * acc + beta * *c;
    }
}

static int cu_count() {
    static int cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] <= 0) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
        cache[dev] = v;
    }
    return cache[dev];
}

// Parts P (k ranges of at least 1024) minimising the modelled time: the 128-wide FP64
// kernel holds two workgroups per CU, so P parts of T output tiles take
// ceil(T P / (2 CUs)) rounds of a k range K / P each, plus the partial-sum traffic
// (written by the product, read by the reduction) per part.  Ties go to fewer parts.
int splitk_parts(int M, int N, long K, bool lower, int most) {
    const long mt = (M + BT - 1) / BT, nt = (N + BT - 1) / BT;
    const long tiles = std::max<long>(1, lower ? (mt == nt ? mt * (mt + 1) / 2 : mt * nt / 2) : mt * nt);
    const long slots = 2L * cu_count();
    const double secPerK = 2.0 * BT * BT * (double) slots / 68e12;           // one round, one k
    const double secPerPart = (double) M * N * 8.0 * (lower ? 1.0 : 2.0) / 5e12;  // partials out and in
    int best = 1;
    double tBest = 1e300;
    for (int P = 1; P <= most && P <= K / 1024; ++P) {
        const long kc = ((K + P - 1) / P + KSTEP - 1) / KSTEP * KSTEP;
        const int parts = (int) ((K + kc - 1) / kc);
        const long rounds = (tiles * parts + slots - 1) / slots;
        const double t = rounds * (double) kc * secPerK + (parts > 1 ? parts * secPerPart : 0.0);
        if (t < 0.97 * tBest) {
            tBest = t;
            best = parts;
        }
    }
    return best;
}

template <typename T>
void gemm_splitk(hipStream_t s, bool transA, bool transB, bool lower, int M, int N, int K, T alpha, const T *A,
                 int lda, const T *B, int ldb, T beta, T *C, int ldc, T *work, size_t workLen) {
    if (M <= 0 || N <= 0) return;
    const size_t mn = (size_t) M * N;
    long P = splitk_parts(M, N, K, lower);
    if (work) P = std::min<long>(P, (long) (workLen / mn));
    if (!work || P <= 1) {
        gemm<T>(s, transA, transB, lower, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, 0);
        return;
    }
    // parts of kc (a multiple of the k slab), the last one K - (parts - 1) kc, in one launch
    const int kc = (int) (((K + P - 1) / P + KSTEP - 1) / KSTEP * KSTEP);
    const int parts = (K + kc - 1) / kc;
    const int kLast = K - (parts - 1) * kc;
    const long sA = transA ? kc : (long) kc * lda, sB = transB ? (long) kc * ldb : kc;
    const int t = pick_tile(M, N, kc, lower, parts, 0, vec_ok<T>(A, lda, sA, B, ldb, sB));
    if (t == 128)
        gemm_big<T>(s, transA, transB, lower, M, N, kc, (T) 1, A, lda, sA, B, ldb, sB, (T) 0, work, M, (long) mn,
                    parts, 0, kLast);
    else if (t == 64)
        gemm_mid<64, T>(s, transA, transB, lower, M, N, kc, (T) 1, A, lda, sA, B, ldb, sB, (T) 0, work, M, (long) mn,
                        parts, 0, 0, kLast);
    else
        gemm_mid<32, T>(s, transA, transB, lower, M, N, kc, (T) 1, A, lda, sA, B, ldb, sB, (T) 0, work, M, (long) mn,
                        parts, 0, 0, kLast);
    splitk_reduce_kernel<T><<<4096, 256, 0, s>>>(M, N, parts, alpha, work, beta, C, ldc, lower ? 1 : 0);
}

template void gemm_splitk<double>(hipStream_t, bool, bool, bool, int, int, int, double, const double *, int,
                                  const double *, int, double, double *, int, double *, size_t);

// ---- triangular inverse ------------------------------------------------------

// Linv = the inverses of the 64 x 64 diagonal blocks, zero elsewhere in the diagonal blocks
// of `span` rows (the rest of Linv is left alone).  The columns run over grid x: there may be
// more of them than the 65535 workgroups of grid y.
template <typename T>
__global__ void place_diag_kernel(int n, int span, const double *Dinv, T *Linv, long ldi) {
    const int j = blockIdx.x, t = blockIdx.y * blockDim.x + threadIdx.x;
    const int i = j / span * span + t;
    if (t >= span || i >= n) return;
    const bool in = (i >> 6) == (j >> 6);
    Linv[i + j * ldi] = in ? (T) Dinv[(long) (j >> 6) * NB * NB + (i & 63) + 64 * (j & 63)] : (T) 0;
}

// inv([[A, 0], [B, C]]) = [[A^-1, 0], [-C^-1 B A^-1, C^-1]], applied level by level
// with every pair of one level batched into two GEMMs.  Below the 128-wide tiles a
// shorter last pair is in the same two launches; n = 500 takes 40 us (129 on 64-wide tiles
// with launches of its own for that pair), n = 2000 172 (442).
template <typename T>
static void trtri_levels(hipStream_t s, int n, const T *L, int ldl, T *Linv, int ldi, T *work, int from, int to) {
    for (int sz = from; sz < to; sz *= 2) {
        int npair = n / (2 * sz);
        long strideL = 2L * sz * (ldl + 1), strideI = 2L * sz * (ldi + 1), strideW = (long) sz * sz;
        const int o = npair * 2 * sz, sc = std::max(0, n - o - sz);  // rows of a last, shorter pair
        // W = L21 Linv11 (Linv11 lower), then Linv21 = -Linv22 W (Linv22 lower)
        const int cnt = npair + (sc > 0 ? 1 : 0);
        if (cnt == 0) continue;
        const int t = pick_tile(sz, sz, sz, false, cnt, 1, false);
        if (t < 128) {
            const auto mid = (t == 32) ? gemm_mid<32, T> : gemm_mid<64, T>;
            mid(s, false, false, false, sz, sz, sz, (T) 1, L + sz, ldl, strideL, Linv, ldi, strideI, (T) 0, work, sz,
                strideW, cnt, 1, sc, 0);
            mid(s, false, false, false, sz, sz, sz, (T) -1, Linv + (long) sz * (ldi + 1), ldi, strideI, work, sz,
                strideW, (T) 0, Linv + sz, ldi, strideI, cnt, 2, sc, sc);
            continue;
        }
        if (npair > 0) {
            gemm<T>(s, false, false, false, sz, sz, sz, (T) 1, L + sz, ldl, strideL, Linv, ldi, strideI, (T) 0,
                    work, sz, strideW, npair, 1);
            gemm<T>(s, false, false, false, sz, sz, sz, (T) -1, Linv + (long) sz * (ldi + 1), ldi, strideI, work,
                    sz, strideW, (T) 0, Linv + sz, ldi, strideI, npair, 2);
        }
        if (sc > 0) {
            gemm<T>(s, false, false, false, sc, sz, sz, (T) 1, L + (o + sz) + (long) o * ldl, ldl, 0,
                    Linv + o + (long) o * ldi, ldi, 0, (T) 0, work, sc, 0, 1, 1);
            gemm<T>(s, false, false, false, sc, sz, sc, (T) -1, Linv + (long) (o + sz) * (ldi + 1), ldi, 0, work,
                    sc, 0, (T) 0, Linv + (o + sz) + (long) o * ldi, ldi, 0, 1, 2);
        }
    }
}

template <typename T>
void trtri(hipStream_t s, int n, const T *L, int ldl, const double *Dinv, T *Linv, int ldi, T *work, int span) {
    if (span <= 0 || span > n) span = n;
    place_diag_kernel<T><<<dim3(n, (span + 255) / 256), 256, 0, s>>>(n, span, Dinv, Linv, ldi);
    trtri_levels<T>(s, n, L, ldl, Linv, ldi, work, NB, span);
}

template void trtri<double>(hipStream_t, int, const double *, int, const double *, double *, int, double *, int);
template void trtri<float>(hipStream_t, int, const float *, int, const double *, float *, int, float *, int);

// ---- matrix-vector ------------------------------------------------------------

// Sums over one U-row group for NC columns: lane rows i, i + 64, ..., i + (U-1) 64,
// all 2U..(NC+1)U loads issued before the FMAs, each column's FMAs in row order.
template <typename T, int U, int NC>
__device__ inline void coldot_group(const T *const (&col)[NC], const T *__restrict__ x, int i, T (&sum)[NC]) {
    T a[NC][U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        b[u] = x[i + u * 64];
#pragma unroll
        for (int c = 0; c < NC; ++c) a[c][u] = col[c][i + u * 64];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int u = 0; u < U; ++u) sum[c] += a[c][u] * b[u];
}

// y_j = alpha <A(lo:hi, j), x(lo:hi)> + beta y_j with (lo, hi) = (0, m), (j, m) for tri 1
// and (0, j + 1) for tri 2.  One wave per NC adjacent columns (NC > 1 only for tri 0 and
// 2, where the columns share the x rows and one x load serves all of them).  Each lane
// accumulates rows lo + lane, lo + lane + 64, ... in order and the wave adds its lanes by a
// fixed shuffle tree, so the result does not depend on NC or on the unrolling.
template <typename T, int NC>
__global__ __launch_bounds__(256) void coldot_kernel(int m, int ncols, int tri, T alpha, const T *__restrict__ A,
                                                     int lda, const T *__restrict__ x, T beta, T *y) {
    const int j0 = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * NC;
    const int lane = threadIdx.x & 63;
    if (j0 >= ncols) return;
    const T *col[NC];
    int hic[NC];
    T sum[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int j = min(j0 + c, ncols - 1);  // a ragged last wave repeats the last column
        col[c] = A + (long) j * lda;
        hic[c] = (tri == 2) ? j + 1 : m;
        sum[c] = 0;
    }
    const int hmin = hic[0];  // hic is nondecreasing in c
    int i = ((NC == 1 && tri == 1) ? j0 : 0) + lane;
    for (; i + 7 * 64 < hmin; i += 8 * 64) coldot_group<T, 8, NC>(col, x, i, sum);
    if (i + 3 * 64 < hmin) {
        coldot_group<T, 4, NC>(col, x, i, sum);
        i += 4 * 64;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
        for (int k = i; k < hic[c]; k += 64) sum[c] += col[c][k] * x[k];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        sum[c] = wave_tree_sum(sum[c]);
        if (lane == 0 && j0 + c < ncols) y[j0 + c] = alpha * sum[c] + ((beta != (T) 0) ? beta * y[j0 + c] : (T) 0);
    }
}

template <typename T, int NC>
static void coldot_launch(hipStream_t s, int m, int ncols, int tri, T alpha, const T *A, int lda, const T *x, T beta,
                          T *y) {
    const int waves = (ncols + NC - 1) / NC;
    coldot_kernel<T, NC><<<(waves + 3) / 4, 256, 0, s>>>(m, ncols, tri, alpha, A, lda, x, beta, y);
}

// Columns per wave: shared x loads pay once there are enough waves to fill the chip
// (measured on 20000^2 FP64: 4.4 TB/s at one column per wave, 5.8 TB/s at four).
template <typename T>
void coldot(hipStream_t s, int m, int ncols, int tri, T alpha, const T *A, int lda, const T *x, T beta, T *y) {
    if (ncols <= 0) return;
    if (tri != 1 && ncols >= 8192)
        coldot_launch<T, 4>(s, m, ncols, tri, alpha, A, lda, x, beta, y);
    else if (tri != 1 && ncols >= 1024)
        coldot_launch<T, 2>(s, m, ncols, tri, alpha, A, lda, x, beta, y);
    else
        coldot_launch<T, 1>(s, m, ncols, tri, alpha, A, lda, x, beta, y);
}

template void coldot<double>(hipStream_t, int, int, int, double, const double *, int, const double *, double,
                             double *);
template void coldot<float>(hipStream_t, int, int, int, float, const float *, int, const float *, float, float *);

// ---- solves with a Cholesky factor ---------------------------------------------------

// The factor as a preconditioner: L is applied by block substitution over blocks of
// solve_span(m) rows with inverted diagonal blocks.  The full inverse costs m^3 / 3 flops
// after the m^3 / 3 of the factorisation (m = 20000: 47 ms after 55; m = 8084: 5.5 after
// 6.7); the inverses of the diagonal blocks cost m span^2 / 3, and a solve reads the same
// triangle once, in 2 m / span dependent pairs of launches per direction.  Up to 2048 rows
// the block is the whole matrix; beyond, the span keeps a solve to five blocks or so.
// Measured, one interior-point iteration (one factorisation, four solves): m = 8084
// 16.0 ms with the full inverse, 13.2, 12.3, 11.9 and 13.1 with spans 512, 1024, 2048 and 4096;
// m = 20000 147 ms, 107, 103, 100 and 102, where the FP32 factor's many more CG steps decide
// (whole mixed solve 9.9, 9.1, 8.6 and 8.5 s).
static int solve_span(int m) {
    int span = 2048;
    while ((long) span * 5 < m) span *= 2;
    return span;
}

// L is mirrored into the upper triangle of its matrix when it has more than one block
// (column j of the upper triangle is row j of L); Li and LiT hold the inverses of the
// diagonal blocks and their transposes in place.
template <typename T>
void solve_prepare(hipStream_t s, int m, T *L, int ld, const double *Dinv, T *Li, T *LiT) {
    const int span = solve_span(m);
    trtri<T>(s, m, L, ld, Dinv, Li, ld, LiT, span);
    for (int b0 = 0; b0 < m; b0 += span) {
        const long at = (long) b0 * (ld + 1);
        transpose<T>(s, std::min(span, m - b0), Li + at, ld, LiT + at, ld);
    }
    if (m > span) mirror_lower<T>(s, m, L, ld);
}

bool solve_in_blocks(int m) { return m > solve_span(m); }

template <typename T>
void solve_complete(hipStream_t s, int m, const T *L, int ld, T *Li, T *LiT) {
    zero_upper<T>(s, m, Li, ld);
    trtri_levels<T>(s, m, L, ld, Li, ld, LiT, solve_span(m), m);
    transpose<T>(s, m, Li, ld, LiT, ld);
}

// z = L^-T L^-1 r; tmp: m entries; r, z and tmp distinct
template <typename T>
void solve_apply(hipStream_t s, int m, const T *L, int ld, const T *Li, const T *LiT, const T *r, T *z, T *tmp,
                 bool complete) {
    const int span = complete ? m : solve_span(m);
    if (m > span) (void) hipMemcpyAsync(z, r, sizeof(T) * m, hipMemcpyDeviceToDevice, s);
    const T *rhs = (m > span) ? z : r;
    int b0 = 0;
    for (; b0 < m; b0 += span) {
        // tmp_b = L_bb^-1 (r_b - sum over earlier blocks)
        const int cnt = std::min(span, m - b0);
        if (b0 > 0) coldot<T>(s, b0, cnt, 0, (T) -1, L + (long) b0 * ld, ld, tmp, (T) 1, z + b0);
        coldot<T>(s, cnt, cnt, 2, (T) 1, LiT + (long) b0 * (ld + 1), ld, rhs + b0, (T) 0, tmp + b0);
    }
    for (b0 -= span; b0 >= 0; b0 -= span) {
        // z_b = L_bb^-T (tmp_b - sum over later blocks)
        const int cnt = std::min(span, m - b0), e0 = b0 + cnt;
        if (e0 < m) coldot<T>(s, m - e0, cnt, 0, (T) -1, L + e0 + (long) b0 * ld, ld, z + e0, (T) 1, tmp + b0);
        coldot<T>(s, cnt, cnt, 1, (T) 1, Li + (long) b0 * (ld + 1), ld, tmp + b0, (T) 0, z + b0);
    }
}

template void solve_prepare<double>(hipStream_t, int, double *, int, const double *, double *, double *);
template void solve_prepare<float>(hipStream_t, int, float *, int, const double *, float *, float *);
template void solve_apply<double>(hipStream_t, int, const double *, int, const double *, const double *,
                                  const double *, double *, double *, bool);
template void solve_apply<float>(hipStream_t, int, const float *, int, const float *, const float *, const float *,
                                 float *, float *, bool);
template void solve_complete<double>(hipStream_t, int, const double *, int, double *, double *);

// ---- symmetric product from the lower triangle -----------------------------------

// y = M x for symmetric M (column-major, ldm) reading only its lower triangle, in one
// pass.  One wave per tile of SYMV_R rows x SYMV_C columns on or below the diagonal;
// lane l owns rows r0 + l + 64 q (q < RPT = SYMV_R / 64).  For each column j of the tile the wave
// forms the column sum over its rows i >= j, sum_i M(i, j) x(i) (the (L^T x)(j)
// share, L the lower triangle), and reduces it over the lanes into P1[R][j]; each
// lane also accumulates the row sums over its columns j < i, sum_j M(i, j) x(j) (the
// strictly-lower (L x)(i) share), stored as P2[C][i].  A second kernel adds the
// partials in a fixed order, so the result is deterministic.  The triangle is read
// once: half the bytes of the column-dot product over the full matrix.  (Tile shape
// measured at m = 20000: 512 x 256 with 4 columns per pass, 0.36 ms; 512 x 128 with 2,
// 0.40 ms; wider or taller tiles leave too few waves.)
template <int RPT, int CP>
__global__ __launch_bounds__(256) void symv_lower_tile_kernel(int m, const double *__restrict__ M, long ldm,
                                                              const double *__restrict__ x, double *P1, double *P2) {
    constexpr int TR = 64 * RPT;  // rows per tile
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int R = blockIdx.x * 4 + w, C = blockIdx.y;
    const int r0 = R * TR, c0 = C * SYMV_C;
    if (r0 >= m || r0 + TR - 1 < c0) return;  // no entry of this tile on or below the diagonal
    double xi[RPT], acc2[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int i = r0 + lane + 64 * q;
        xi[q] = (i < m) ? x[i] : 0.0;
        acc2[q] = 0.0;
    }
    const int cEnd = min(min(c0 + SYMV_C, m), r0 + TR);
    // CP columns per pass, the next pass's loads issued before this pass's lane
    // reductions (software pipelining: the loop is otherwise load-latency bound)
    double v[CP][RPT];
    auto fetch = [&](int j) {
#pragma unroll
        for (int c = 0; c < CP; ++c) {
            const double *col = M + (long) (j + c) * ldm;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int i = r0 + lane + 64 * q;
                v[c][q] = (j + c < cEnd && i < m && i >= j + c) ? col[i] : 0.0;
            }
        }
    };
    fetch(c0);
    for (int j = c0; j < cEnd; j += CP) {
        double a[CP], xj[CP];
#pragma unroll
        for (int c = 0; c < CP; ++c) {
            xj[c] = (j + c < cEnd) ? x[j + c] : 0.0;
            a[c] = 0.0;
        }
#pragma unroll
        for (int c = 0; c < CP; ++c)
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int i = r0 + lane + 64 * q;
                a[c] += v[c][q] * xi[q];
                if (i > j + c) acc2[q] += v[c][q] * xj[c];
            }
        if (j + CP < cEnd) fetch(j + CP);
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int c = 0; c < CP; ++c) a[c] += __shfl_down(a[c], off);
        if (lane == 0)
#pragma unroll
            for (int c = 0; c < CP; ++c)
                if (j + c < cEnd) P1[(long) R * m + j + c] = a[c];
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int i = r0 + lane + 64 * q;
        if (i < m) P2[(long) C * m + i] = acc2[q];
    }
}

// y(i) = sum over the row chunks R >= i / SYMV_R of P1[R][i] + sum over the column
// blocks C <= (row chunk start of i + SYMV_R - 1) / SYMV_C of P2[C][i], in that order
__global__ void symv_lower_reduce_kernel(int m, int nR, int nC, const double *P1, const double *P2, double *y) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    double s = 0.0;
    for (int R = i / SYMV_R; R < nR; ++R) s += P1[(long) R * m + i];
    const int cLast = min(nC - 1, ((i / SYMV_R) * SYMV_R + SYMV_R - 1) / SYMV_C);
    for (int C = 0; C <= cLast; ++C) s += P2[(long) C * m + i];
    y[i] = s;
}

size_t symv_lower_work(int m) {
    const size_t nR = (m + SYMV_R - 1) / SYMV_R, nC = (m + SYMV_C - 1) / SYMV_C;
    return (nR + nC) * (size_t) m;
}

void symv_lower(hipStream_t s, int m, const double *M, long ldm, const double *x, double *y, double *work) {
    if (m <= 0) return;
    const int nR = (m + SYMV_R - 1) / SYMV_R, nC = (m + SYMV_C - 1) / SYMV_C;
    double *P1 = work, *P2 = work + (size_t) nR * m;
    symv_lower_tile_kernel<SYMV_R / 64, 4><<<dim3((nR + 3) / 4, nC), 256, 0, s>>>(m, M, ldm, x, P1, P2);
    symv_lower_reduce_kernel<<<(m + 255) / 256, 256, 0, s>>>(m, nR, nC, P1, P2, y);
}

// ---- layout helpers --------------------------------------------------------------

template <typename T>
__global__ void mirror_kernel(int n, T *A, int lda) {
    __shared__ T tile[32][33];
    const int bi = blockIdx.x, bj = blockIdx.y;
    if (bi < bj) return;
    const int i0 = bi * 32, j0 = bj * 32, tx = threadIdx.x, ty = threadIdx.y;
    for (int r = ty; r < 32; r += 8) {
        int i = i0 + tx, j = j0 + r;
        tile[r][tx] = (i < n && j < n) ? A[i + (long) j * lda] : (T) 0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        int i = i0 + r, j = j0 + tx;  // source (i, j), destination (j, i)
        if (i < n && j < n && i > j) A[j + (long) i * lda] = tile[tx][r];
    }
}

template <typename T>
void mirror_lower(hipStream_t s, int n, T *A, int lda) {
    int nb = (n + 31) / 32;
    mirror_kernel<T><<<dim3(nb, nb), dim3(32, 8), 0, s>>>(n, A, lda);
}

template void mirror_lower<double>(hipStream_t, int, double *, int);
template void mirror_lower<float>(hipStream_t, int, float *, int);

template <typename T>
__global__ void transpose_kernel(int n, const T *A, int lda, T *B, int ldb) {
    __shared__ T tile[32][33];
    const int i0 = blockIdx.x * 32, j0 = blockIdx.y * 32, tx = threadIdx.x, ty = threadIdx.y;
    for (int r = ty; r < 32; r += 8) {
        int i = i0 + tx, j = j0 + r;
        tile[r][tx] = (i < n && j < n) ? A[i + (long) j * lda] : (T) 0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        int i = i0 + r, j = j0 + tx;
        if (i < n && j < n) B[j + (long) i * ldb] = tile[tx][r];
    }
}

template <typename T>
void transpose(hipStream_t s, int n, const T *A, int lda, T *B, int ldb) {
    int nb = (n + 31) / 32;
    transpose_kernel<T><<<dim3(nb, nb), dim3(32, 8), 0, s>>>(n, A, lda, B, ldb);
}

template void transpose<double>(hipStream_t, int, const double *, int, double *, int);
template void transpose<float>(hipStream_t, int, const float *, int, float *, int);

template <typename T>
__global__ void zero_upper_kernel(int n, T *A, int lda) {
    long total = (long) n * n;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < total; e += (long) gridDim.x * blockDim.x) {
        long i = e % n, j = e / n;
        if (i < j) A[i + j * lda] = 0;
    }
}

template <typename T>
void zero_upper(hipStream_t s, int n, T *A, int lda) {
    zero_upper_kernel<T><<<1024, 256, 0, s>>>(n, A, lda);
}

template void zero_upper<double>(hipStream_t, int, double *, int);
template void zero_upper<float>(hipStream_t, int, float *, int);

__global__ void fill_kernel(double *x, long n, double v) {
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < n; e += (long) gridDim.x * blockDim.x) x[e] = v;
}

void fill(hipStream_t s, double *x, long n, double v) {
    if (n <= 0) return;
    long blocks = (n + 255) / 256;
    fill_kernel<<<blocks > 4096 ? 4096 : blocks, 256, 0, s>>>(x, n, v);
}

__global__ void fill_f_kernel(float *x, long n, float v) {
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < n; e += (long) gridDim.x * blockDim.x) x[e] = v;
}

void fill_f(hipStream_t s, float *x, long n, float v) {
    if (n <= 0) return;
    long blocks = (n + 255) / 256;
    fill_f_kernel<<<blocks > 4096 ? 4096 : blocks, 256, 0, s>>>(x, n, v);
}

__global__ void copy_lower_kernel(int n, const double *A, int lda, double *B, int ldb) {
    long total = (long) n * n;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < total; e += (long) gridDim.x * blockDim.x) {
        long i = e % n, j = e / n;
        if (i >= j) B[i + j * ldb] = A[i + j * lda];
    }
}

void copy_lower(hipStream_t s, int n, const double *A, int lda, double *B, int ldb) {
    copy_lower_kernel<<<2048, 256, 0, s>>>(n, A, lda, B, ldb);
}

__global__ void convert_lower_kernel(int n, const double *A, int lda, float *B, int ldb) {
    long total = (long) n * n;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < total; e += (long) gridDim.x * blockDim.x) {
        long i = e % n, j = e / n;
        B[i + j * ldb] = (i >= j) ? (float) A[i + j * lda] : 0.0f;
    }
}

void convert_lower_to_float(hipStream_t s, int n, const double *A, int lda, float *B, int ldb) {
    convert_lower_kernel<<<2048, 256, 0, s>>>(n, A, lda, B, ldb);
}

__global__ void convert_lower_scaled_kernel(int n, const double *A, int lda, const double *sc, double shift, float *B,
                                            int ldb) {
    long total = (long) n * n;
    for (long e = blockIdx.x * (long) blockDim.x + threadIdx.x; e < total; e += (long) gridDim.x * blockDim.x) {
        long i = e % n, j = e / n;
        float v = 0.0f;
        if (i >= j) v = (float) (A[i + j * lda] * sc[i] * sc[j] + ((i == j) ? shift : 0.0));
        B[i + j * ldb] = v;
    }
}

void convert_lower_scaled(hipStream_t s, int n, const double *A, int lda, const double *sc, double shift, float *B,
                          int ldb) {
    convert_lower_scaled_kernel<<<2048, 256, 0, s>>>(n, A, lda, sc, shift, B, ldb);
}

__global__ void add_diag_kernel(int n, double *A, int lda, const double *d, double scalar) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) A[i + (long) i * lda] += (d ? d[i] : 0.0) + scalar;
}

void add_diag(hipStream_t s, int n, double *A, int lda, const double *d, double scalar) {
    add_diag_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, A, lda, d, scalar);
}

__global__ void logdet_kernel(int n, const double *A, int lda, double *out) {
    __shared__ double red[256];
    double sum = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) sum += log(A[i + (long) i * lda]);
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int) threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = 2.0 * red[0];
}

void logdet_diag(hipStream_t s, int n, const double *A, int lda, double *out) {
    logdet_kernel<<<1, 256, 0, s>>>(n, A, lda, out);
}

}  // namespace hdk
