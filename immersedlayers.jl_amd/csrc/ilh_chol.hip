// ilh_chol.hip -- the dense FP64 algebra of the Schur complements on the
// matrix cores: a v_mfma_f64_16x16x4f64 GEMM, and the blocked Cholesky
// factorisation of the symmetrised Schur matrix with its multi-right-hand-side
// solves.
//
// The reference solves S x = b with `S\b` (LAPACK LU on every call,
// test/literate/problems.jl:291, test/literate/dirichlet.jl:99).  For the
// Schur matrices built from an interpolation E and a regularization R of the
// same grid kind (create_RTLinvR, src/matrix_operators.jl:9-30, and the
// integrating-factor stage matrices E H R), GridScaling makes R = E^T diag(d)
// (d = ds / dx^2), so
//     S = M diag(d),   M = E K E^T  symmetric,
// with K the kernel (-L^-1 or the heat kernel).  -L^-1 is only conditionally
// positive definite: M is positive definite on the vectors orthogonal to the
// constant one and has a single negative eigenvalue along it.  A Householder
// reflection H (H u = e_1, u = 1/sqrt(n)) moves that direction to the first
// coordinate:
//     H M H = [alpha  beta^T ]      Mt = (n-1) x (n-1), positive definite,
//             [beta   Mt     ]
// Mt is factored by blocked Cholesky (no pivoting), the first coordinate is
// eliminated through its scalar Schur complement sigma = alpha - beta^T Mt^-1 beta.
// An exactly singular direction (points whose windows coincide) shows as a
// non-positive pivot; the caller then falls back to LU.
#include "ilh_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace ilh {

typedef double double4_t __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ GEMM
// C (M x Nc) = beta C + alpha opA(A) B, column-major, beta in {0, 1} (BETA0: C
// is not read).  opA(A)[m][k] = A[m + lda k] (TA = 0) or A[k + lda m] (TA = 1),
// B[k][n] at k + ldb n.  tri restricts the K range of each tile to where a
// triangular operand is nonzero (entries of its other triangle outside its
// 64 x 64 diagonal blocks are never read): TRI_A_LOWER opA(A)[m][k] = 0 for
// k > m, TRI_B_LOWER B[k][n] = 0 for k < n.
//
// 64 x 64 tile per work-group of four waves, each wave a 32 x 32 quadrant of
// 2 x 2 blocks of 16 x 16.  K runs in chunks of 16 through two LDS buffers:
// the next chunk's global loads are in flight while the current one feeds the
// matrix cores, and all of a chunk's LDS fragments are read before its 16
// matrix instructions, so that they issue back to back (1024 of a chunk's
// cycles; the wave's LDS wait is paid once per chunk).  The product is formed
// transposed (the B tile as the MFMA's first operand), so a lane's result
// entries run down a column of C and the stores of 16 lanes cover 128
// contiguous bytes.  The bound is the matrix cores' FP64 rate (32 FMA cycles
// per 16 x 16 x 4 product); the tiles with the longest K range of a triangular
// operand are dispatched first.
// v_mfma_f64_16x16x4f64 lane layout (checked on gfx950): first operand
// X[i][k] at lane i + 16 k, second Y[k][j] at lane j + 16 k; lane l, item r
// of the result holds D[l / 16 + 4 r][l % 16].
static constexpr int GT = 64, GKC = 16;
enum { TRI_NONE = 0, TRI_A_LOWER = 1, TRI_B_LOWER = 2 };

// A batch runs over blockIdx.z: operands at z times the strides, M (and K,
// when k_is_m) clipped to what is left of m_total rows z m_step on.
struct GemmBatch {
    size_t sa = 0, sb = 0, sc = 0;
    int m_total = 0, m_step = 0;
    int k_is_m = 0;
};
// With DOT, also the sums of C[m, n] v[n] over each 32 columns of a tile, at
// dots + M (2 n-tile + half) (gridDim.z = 1).
struct GemmDots {
    const double* v = nullptr;
    double* dots = nullptr;
};

template <int TA, bool BETA0, bool DOT>
// (A or B may be C itself when every work-group reads all the entries it
// overwrites; hence no __restrict__.)
__global__ void __launch_bounds__(256) k_dgemm(int M, int Nc, int K, double alpha, const double* A, int lda,
                                               const double* B, int ldb, double* C, int ldc, int tri, GemmBatch bt,
                                               GemmDots ep)
{
    __shared__ double As[2][GKC][GT + 2];   // As[k][m]
    __shared__ double Bs[2][GKC][GT + 2];   // Bs[k][n]
    const int z = blockIdx.z;
    A += bt.sa * z;
    B += bt.sb * z;
    C += bt.sc * z;
    if (bt.m_step) {
        M = min(M, bt.m_total - z * bt.m_step);
        if (bt.k_is_m) K = min(K, M);
    }
    // triangular operands: tiles by falling K range, every second round of
    // 256 (one per CU) backwards, so that the rounds' sums come out even
    int bx = blockIdx.x, by = blockIdx.y;
    if (tri != TRI_NONE) {
        const int total = gridDim.x * gridDim.y;
        int t = blockIdx.x + gridDim.x * blockIdx.y;
        const int r0 = t & ~255;
        if (r0 & 256) t = r0 + min(256, total - r0) - 1 - (t - r0);
        if (tri == TRI_A_LOWER) {
            bx = gridDim.x - 1 - t / gridDim.y;
            by = t % gridDim.y;
        } else {
            by = t / gridDim.x;
            bx = t % gridDim.x;
        }
    }
    const int m0 = bx * GT, n0 = by * GT;
    if (m0 >= M || n0 >= Nc) return;
    int klo = 0, khi = K;
    if (tri == TRI_A_LOWER) khi = min(K, m0 + GT);
    else if (tri == TRI_B_LOWER) klo = n0;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
    // this thread's four elements of each operand's chunk.  Rows and columns
    // past the end load the last one's entries (their products are not
    // stored), and k past the end an entry that exists, zeroed on its way to
    // LDS: the loads themselves carry no branch or use, so that three chunks
    // of them stay in flight
    const int am = TA == 0 ? tid & 63 : tid >> 4, ak = TA == 0 ? tid >> 6 : tid & 15;
    const int bn = tid >> 4, bk = tid & 15;
    const double *pa[4], *pb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = min(m0 + am + (TA == 0 ? 0 : 16 * j), M - 1), n = min(n0 + bn + 16 * j, Nc - 1);
        const int k = klo + ak + (TA == 0 ? 4 * j : 0);
        pa[j] = TA == 0 ? A + m + (size_t)lda * k : A + k + (size_t)lda * m;
        pb[j] = B + (klo + bk) + (size_t)ldb * n;
    }
    const size_t step_a = TA == 0 ? (size_t)lda * GKC : GKC;
    double pre[3][8];   // three chunks on the way: [0..3] of A, [4..7] of B
    auto load = [&](int k0, double* r) {   // the chunk at k0 (in order: the pointers advance with it)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r[j] = *(k0 + ak + (TA == 0 ? 4 * j : 0) < khi ? pa[j] : A);
            r[4 + j] = *(k0 + bk < khi ? pb[j] : B);
            pa[j] += step_a;
            pb[j] += GKC;
        }
    };
    auto store = [&](int k0, int buf, const double* r) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double va = k0 + ak + (TA == 0 ? 4 * j : 0) < khi ? r[j] : 0.0;
            const double vb = k0 + bk < khi ? r[4 + j] : 0.0;
            if (TA == 0) As[buf][(tid >> 6) + 4 * j][tid & 63] = va;
            else As[buf][tid & 15][(tid >> 4) + 16 * j] = va;
            Bs[buf][tid & 15][(tid >> 4) + 16 * j] = vb;
        }
    };
    double4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};
    const int nch = khi > klo ? (khi - klo + GKC - 1) / GKC : 0;
    if (nch > 0) {
        // chunk c is loaded three ahead, into the registers that chunk c - 3 left
#pragma unroll
        for (int q = 0; q < 3; ++q) load(klo + q * GKC, pre[q]);
        store(klo, 0, pre[0]);
        lds_sync();
    }
    for (int c0 = 0; c0 < nch; c0 += 3) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int c = c0 + q;
            if (c >= nch) break;
            const int buf = c & 1;
            double a[4][2], b[4][2];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int kr = 4 * kk + (lane >> 4);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[kk][i] = As[buf][kr][wm + 16 * i + (lane & 15)];
                    b[kk][i] = Bs[buf][kr][wn + 16 * i + (lane & 15)];
                }
            }
            load(klo + (c + 3) * GKC, pre[q]);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[kk][j], a[kk][i], acc[i][j], 0, 0, 0);
            store(klo + (c + 1) * GKC, buf ^ 1, pre[(q + 1) % 3]);
            lds_sync();
        }
    }
    // acc[i][j] item r of lane l: C row m0 + wm + 16 i + l % 16, column n0 + wn + 16 j + l / 16 + 4 r
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int gm = m0 + wm + 16 * i + (lane & 15);
        if (DOT) {
            double q = 0.0;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int gn = n0 + wn + 16 * j + (lane >> 4) + 4 * r;
                    if (gn < Nc) q = __builtin_fma(acc[i][j][r], ep.v[gn], q);
                }
            q += __shfl_xor(q, 16, 64);
            q += __shfl_xor(q, 32, 64);
            if (lane < 16 && gm < M) ep.dots[gm + (size_t)M * (2 * by + (wave >> 1))] = q;
        }
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gn = n0 + wn + 16 * j + (lane >> 4) + 4 * r;
                if (gn >= Nc) continue;
                double* p = C + gm + (size_t)ldc * gn;
                *p = BETA0 ? alpha * acc[i][j][r] : *p + alpha * acc[i][j][r];
            }
    }
}

void gemm_sub(hipStream_t st, int M, int Nc, int K, const double* A, int lda, const double* B, int ldb, double* C, int ldc)
{
    if (M <= 0 || Nc <= 0 || K <= 0) return;
    k_dgemm<0, false, false><<<dim3((M + GT - 1) / GT, (Nc + GT - 1) / GT), 256, 0, st>>>(
        M, Nc, K, -1.0, A, lda, B, ldb, C, ldc, TRI_NONE, GemmBatch(), GemmDots());
    ILH_HIP(hipGetLastError());
}

// ------------------------------------------------------------- Cholesky
static constexpr int CB = 64;   // block size of the factorisation
static constexpr int SB = 16;   // sub-block of a diagonal block: one matrix-core product

__device__ __forceinline__ double readlane_d(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// 1 / sqrt(x), x > 0 and of ordinary size: the hardware estimate and two
// coupled Newton steps (Goldschmidt), to within an ulp or two
__device__ __forceinline__ double rsqrt_nr(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double r = __builtin_fma(-g, h, 0.5);
        g = __builtin_fma(g, r, g);
        h = __builtin_fma(h, r, h);
    }
    return 2.0 * h;
}

// 64 x 64 blocks in LDS, row-major with one pad entry per row
typedef double Block[CB][CB + 1];

// X_bb = L_bb^-1 of the 16 x 16 diagonal sub-block b (lane c % 16 forms column
// c by forward substitution; rd: reciprocals of L's diagonal).  Every wave that
// needs X_bb calls this itself and then reads back only what it wrote (equal
// values in the same places), so no barrier is needed.
__device__ __forceinline__ void sub_inverse(const Block& T, const double* rd, Block& X, int b, int lane)
{
    const int o = b * SB, c = lane & 15;
    double x[SB];
#pragma unroll
    for (int r = 0; r < SB; ++r) {
        double v = r == c ? 1.0 : 0.0, v2 = 0.0;
#pragma unroll
        for (int k = 0; k < r; ++k) {
            if (k & 1) v2 = __builtin_fma(-T[o + r][o + k], x[k], v2);
            else v = __builtin_fma(-T[o + r][o + k], x[k], v);
        }
        x[r] = (v + v2) * rd[o + r];
    }
    if (lane < SB)
#pragma unroll
        for (int r = 0; r < SB; ++r) X[o + r][o + c] = x[r];
}

// X_ij = -X_ii sum_{k=j}^{i-1} L_ik X_kj for 16 x 16 sub-blocks, by one wave:
// the inner sum's result layout is the second operand's layout of the outer
// product, so nothing is exchanged in between
__device__ __forceinline__ void sub_inverse_off(const Block& T, Block& X, int i, int j, int lane)
{
    const int lr = lane & 15, lk = lane >> 4;
    double4_t y = (double4_t){0.0, 0.0, 0.0, 0.0};
    for (int k = j; k < i; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            y = __builtin_amdgcn_mfma_f64_16x16x4f64(T[i * SB + lr][k * SB + 4 * q + lk], X[k * SB + 4 * q + lk][j * SB + lr],
                                                     y, 0, 0, 0);
    double4_t x = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
        x = __builtin_amdgcn_mfma_f64_16x16x4f64(X[i * SB + lr][i * SB + 4 * q + lk], y[q], x, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) X[i * SB + lk + 4 * r][j * SB + lr] = -x[r];
}

// T_ij -= L_ib L_jb^T for 16 x 16 sub-blocks, by one wave
__device__ __forceinline__ void sub_update(Block& T, int i, int j, int b, int lane)
{
    const int lr = lane & 15, lk = lane >> 4;
    double4_t acc = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(T[i * SB + lr][b * SB + 4 * q + lk], T[j * SB + lr][b * SB + 4 * q + lk],
                                                   acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) T[i * SB + lk + 4 * r][j * SB + lr] -= acc[r];
}

// Cholesky of the 64 x 64 block in T (its lower triangle) by a work-group of
// four waves, and the inverse of the factor in X's lower sub-blocks.  Column
// panels of 16: wave 0 holds all 64 rows of the panel (lane = row) and factors
// it alone, the pivot and the multipliers of each step broadcast with
// readlane, so the rows below the diagonal sub-block cost nothing extra; the
// next panel's update comes first, and everything else (the remaining
// updates, the inverse's finished rows) runs on the other waves beside the
// next panel.  Eight barriers; the chain of 64 pivot steps bounds it.
// A pivot that is not positive records its 1-based column col0 + ... in *info
// (the first one only) and is replaced by 1, so that the kernel still runs to
// its end.
__device__ __forceinline__ void chol_block(Block& T, Block& X, double* rd, int col0, int* info)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto finish_row = [&](int b) {   // waves 1..3: row b of the inverse
        sub_inverse(T, rd, X, b, lane);
        if (wave - 1 < b) sub_inverse_off(T, X, b, wave - 1, lane);
    };
#pragma unroll
    for (int b = 0; b < CB / SB; ++b) {
        const int o = b * SB;
        if (wave == 0) {
            double d[SB];
#pragma unroll
            for (int c = 0; c < SB; ++c) d[c] = T[lane][o + c];
            // the next pivot's reciprocal root is formed beside the rest of a
            // step's updates; the scheduling barriers keep a step's broadcast
            // values from piling up in scalar registers
            double piv = readlane_d(d[0], o), rdv = 1.0;
            int bad = 0;
            double ri = 1.0;
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                if (j == 0) {
                    bad = piv > 0.0 ? 0 : 1;
                    piv = piv > 0.0 ? piv : 1.0;
                    ri = rsqrt_nr(piv);
                }
                const double l = d[j] * ri;
                d[j] = lane > o + j ? l : (lane == o + j ? piv * ri : 0.0);
                rdv = lane == j ? ri : rdv;
                if (j + 1 < SB) {
                    d[j + 1] = __builtin_fma(-l, readlane_d(l, o + j + 1), d[j + 1]);
                    piv = readlane_d(d[j + 1], o + j + 1);
                    bad = bad == 0 && !(piv > 0.0) ? j + 2 : bad;
                    piv = piv > 0.0 ? piv : 1.0;
                    ri = rsqrt_nr(piv);
#pragma unroll
                    for (int c = j + 2; c < SB; ++c) d[c] = __builtin_fma(-l, readlane_d(l, o + c), d[c]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (bad && lane == 0) atomicCAS(info, 0, col0 + o + bad);
            if (lane < SB) rd[o + lane] = rdv;
            if (lane >= o)
#pragma unroll
                for (int c = 0; c < SB; ++c) T[lane][o + c] = d[c];
        } else if (b > 0) {
            // updates by panel b - 1 beyond panel b: (2,2) (3,2) (3,3), then (3,3)
            if (b == 1) sub_update(T, wave == 1 ? 2 : 3, wave == 3 ? 3 : 2, 0, lane);
            if (b == 2 && wave == 1) sub_update(T, 3, 3, 1, lane);
            finish_row(b - 1);
        }
        lds_sync();
        if (b + 1 < CB / SB) {
            if (b + 1 + wave < CB / SB) sub_update(T, b + 1 + wave, b + 1, b, lane);
            lds_sync();
        }
    }
    if (wave > 0) finish_row(CB / SB - 1);
    lds_sync();
}

// One step of the right-looking blocked Cholesky of the m x m matrix A (lower
// triangle): block column k is eliminated from every 64 x 64 tile (i, j),
// k < j <= i, one work-group each,
//     A_ij -= L_ik L_jk^T,   L_ik = A_ik W_kk^T,  W_kk = L_kk^-1,
// and the work-group of tile (k+1, k+1) goes on to factor it and to invert the
// factor (W_{k+1,k+1}), so that a step is one launch and the diagonal chain
// runs beside the other tiles.  Every work-group forms the two panel blocks it
// needs itself (the panel is small next to a separate launch for it); the one
// of column k+1 keeps L_ik in Lb.  k = -1: tile (0, 0) is factored only.
// Each wave forms 16 rows of both panel blocks, operands straight from memory
// (16 rows are 128 contiguous bytes); a result item's layout is the operand
// layout of one K step, so the blocks pass through LDS as they are.
// Bound by the diagonal chain (update, 64 pivot steps, inverse); N = 1885
// (30 steps): 22 us per step; the recursive form this replaced, three to
// five launches per block around a 39 us diagonal kernel, took 85 us per block.
__global__ void __launch_bounds__(256) k_chol_step(double* __restrict__ A, int lda, int m, int k, double* __restrict__ W,
                                                   int ldw, double* __restrict__ Lb, int ldl, int* __restrict__ info)
{
    __shared__ double sm[2 * CB * (CB + 1)];
    __shared__ double rd[CB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int wm = (wave & 1) * 2, wn = (wave >> 1) * 2;   // quadrant, in 16-blocks
    int ti = 0, tj = 0;
    if (k >= 0) {
        const int t = blockIdx.x;
        ti = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
        while (ti * (ti + 1) / 2 > t) --ti;
        while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
        tj = t - ti * (ti + 1) / 2;
    }
    const int i0 = (k + 1 + ti) * CB, j0 = (k + 1 + tj) * CB;
    double4_t c[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = i0 + 16 * (wm + x) + lr, col = j0 + 16 * (wn + y) + lk + 4 * r;
                c[x][y][r] = row < m && col < m ? A[row + (size_t)lda * col] : 0.0;
            }
    if (k >= 0) {
        const int k0 = k * CB;
        const double* Wk = W + k0 + (size_t)ldw * k0;
        // W_kk's fragments (its lower sub-blocks), then the wave's 16 rows of both panel blocks
        double w[40], a[2][16];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int q = 0; q < 4 * (cb + 1); ++q)
                w[2 * cb * (cb + 1) + q] = Wk[16 * cb + lr + (size_t)ldw * (4 * q + lk)];
        const bool two = ti != tj;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (p == 1 && !two) break;
            const int row = min((p ? j0 : i0) + 16 * wave + lr, m - 1);   // rows past the end: copies of the last
#pragma unroll
            for (int q = 0; q < 16; ++q) a[p][q] = A[row + (size_t)lda * (k0 + 4 * q + lk)];
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (p == 1 && !two) break;
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                double4_t l = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 4 * (cb + 1); ++q)
                    l = __builtin_amdgcn_mfma_f64_16x16x4f64(w[2 * cb * (cb + 1) + q], a[p][q], l, 0, 0, 0);
                // item r: row lr of the wave's 16, column 16 cb + 4 r + lk = the operand of K step 4 cb + r
#pragma unroll
                for (int r = 0; r < 4; ++r) sm[p * CB * CB + (wave * 16 + 4 * cb + r) * 64 + lane] = l[r];
                const int row = i0 + 16 * wave + lr;
                if (p == 0 && tj == 0 && row < m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) Lb[row + (size_t)ldl * (k0 + 16 * cb + 4 * r + lk)] = l[r];
            }
        }
        lds_sync();
        const double* sj = sm + (two ? CB * CB : 0);
        double4_t u[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) u[x][y] = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            double fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                fa[x] = sm[((wm + x) * 16 + q) * 64 + lane];
                fb[x] = sj[((wn + x) * 16 + q) * 64 + lane];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) u[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[y], fa[x], u[x][y], 0, 0, 0);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) c[x][y] -= u[x][y];
        if (blockIdx.x != 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = i0 + 16 * (wm + x) + lr, col = j0 + 16 * (wn + y) + lk + 4 * r;
                        if (row < m && col < m) A[row + (size_t)lda * col] = c[x][y][r];
                    }
            return;
        }
        lds_sync();   // the panel blocks are read: their LDS becomes T and X
    }
    Block& T = *(Block*)sm;
    Block& X = *(Block*)(sm + CB * (CB + 1));
    const int nb = min(CB, m - i0);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * (wm + x) + lr, col = 16 * (wn + y) + lk + 4 * r;
                T[row][col] = row < nb && col < nb ? c[x][y][r] : (row == col ? 1.0 : 0.0);
            }
    lds_sync();
    chol_block(T, X, rd, i0, info);
    double* Wd = W + i0 + (size_t)ldw * i0;
    for (int e = threadIdx.x; e < CB * CB; e += 256) {
        const int r = e % CB, cc = e / CB;
        if (r < nb && cc < nb) Wd[r + (size_t)ldw * cc] = r >= cc ? X[r][cc] : 0.0;
    }
}

// W = L^-1 of the m x m matrix A = L L^T (lower triangle read; A is scratch
// afterwards): the diagonal blocks' inverses from the factorisation's steps,
// then W21 = -W22 (L21 W11) for pairs of neighbouring diagonal blocks of 64,
// 128, 256, ... rows, two batched products per size.  W's entries above its
// 64 x 64 diagonal blocks are not written; Lb, T: m x m scratch.
// *info (device, cleared by the caller): the 1-based column of the first
// non-positive pivot.
static void chol_factor(hipStream_t st, double* A, int lda, int m, double* W, double* Lb, double* T, int* info)
{
    const int nbk = (m + CB - 1) / CB;
    for (int k = -1; k < nbk - 1; ++k) {
        const int t = nbk - 1 - k;
        k_chol_step<<<k < 0 ? 1 : t * (t + 1) / 2, 256, 0, st>>>(A, lda, m, k, W, m, Lb, m, info);
    }
    ILH_HIP(hipGetLastError());
    for (int s = CB; s < m; s *= 2) {
        const int pairs = (m - s + 2 * s - 1) / (2 * s);
        const size_t dd = (size_t)2 * s * (m + 1), off = s;   // from one pair's blocks to the next; row offset of 21
        GemmBatch bt;
        bt.sa = bt.sb = bt.sc = dd;
        bt.m_total = m - s;
        bt.m_step = 2 * s;
        const dim3 grid((std::min(s, m - s) + GT - 1) / GT, s / GT, pairs);
        // T21 = L21 W11
        k_dgemm<0, true, false><<<grid, 256, 0, st>>>(std::min(s, m - s), s, s, 1.0, Lb + off, m, W, m, T + off, m,
                                                           TRI_B_LOWER, bt, GemmDots());
        // W21 = -W22 T21
        bt.k_is_m = 1;
        k_dgemm<0, true, false><<<grid, 256, 0, st>>>(std::min(s, m - s), s, s, -1.0, W + off + (size_t)m * s, m,
                                                           T + off, m, W + off, m, TRI_A_LOWER, bt, GemmDots());
    }
    ILH_HIP(hipGetLastError());
}

// ---------------------------------------------- products of W with a vector
// Y[r] = sum_{k <= r} W[r + m k] X[k]: one work-group of 16 waves per 16 rows; a
// wave takes four columns of 16 rows at a time, every 64th, and the 64 partial
// sums are added in a fixed order.  (One wave per 64 rows and column: 79 us at
// m = 1884, two vectors, too few work-groups and loads in flight.)
__global__ void __launch_bounds__(1024) k_wmv(const double* __restrict__ W, int m, const double* __restrict__ X,
                                              double* __restrict__ Y)
{
    __shared__ double part[64][17];
    const int tid = threadIdx.x, lr = tid & 15, kq = tid >> 4;   // kq: column of the round, 0..63
    const int r = blockIdx.x * 16 + lr, rc = min(r, m - 1), kend = min(m, (int)(blockIdx.x * 16 / 64 + 1) * 64);
    double acc = 0.0;
#pragma unroll 8
    for (int k = kq; k < kend; k += 64) acc = __builtin_fma(W[rc + (size_t)m * k], X[k], acc);
    part[kq][lr] = acc;
    __syncthreads();
    if (tid < 16) {
        double t = 0.0;
        for (int q = 0; q < 64; ++q) t += part[q][lr];
        if (r < m) Y[r] = t;
    }
}

// Z[p] = sum_{k >= p} W[k + m p] T[k], one wave per column p
__global__ void __launch_bounds__(256) k_wtmv(const double* __restrict__ W, int m, const double* __restrict__ T,
                                              double* __restrict__ Z)
{
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= m) return;
    const double* col = W + (size_t)m * p;
    double acc = 0.0;
#pragma unroll 8
    for (int k = p + lane; k < m; k += 64) acc = __builtin_fma(col[k], T[k], acc);
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) Z[p] = acc;
}

// --------------------------------------------------- deflated symmetric solve
// w: the Householder vector of H = I - 2 w w^T with H (1/sqrt(n)) = e_1
// (w = 0, H = I without deflation); clears the pivot flag of the factorisation
// that follows
__global__ void k_house_vec(double* __restrict__ w, int n, bool deflate, int* __restrict__ info)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *info = 0;
    if (i >= n) return;
    if (n == 1 || !deflate) {
        w[i] = 0.0;
        return;
    }
    const double u = 1.0 / sqrt((double)n);
    const double nrm = sqrt(2.0 - 2.0 * u);
    w[i] = (i == 0 ? u - 1.0 : u) / nrm;
}

// y = A x (A n x n column-major, symmetric: one wave per row reads the row
// through the column, i.e. y_i = sum_j A[j + lda i] x_j)
__global__ void k_symv(const double* __restrict__ A, int n, int lda, const double* __restrict__ x,
                       double* __restrict__ y)
{
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const double* col = A + (size_t)lda * i;
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s += col[j] * x[j];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) y[i] = s;
}

// p = 2 (y - (w.y) w), y = A w: one work-group
__global__ void __launch_bounds__(1024) k_house_p(const double* __restrict__ w, const double* __restrict__ y, int n,
                                                  double* __restrict__ p)
{
    __shared__ double red[1024];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) s += w[i] * y[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    const double t = red[0];
    for (int i = threadIdx.x; i < n; i += 1024) p[i] = 2.0 * (y[i] - t * w[i]);
}

// A <- H A H = A - w p^T - p w^T
__global__ void k_rank2(double* __restrict__ A, int n, int lda, const double* __restrict__ w,
                        const double* __restrict__ p)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= n) return;
    A[i + (size_t)lda * j] -= w[i] * p[j] + p[i] * w[j];
}

// sig = {alpha - beta . wt, w1 . wt}; a pivot of Mt of at most tol (1 / W_ii^2)
// sets *info if no pivot did
__global__ void __launch_bounds__(1024) k_sigma(const double* __restrict__ A, const double* __restrict__ w,
                                                const double* __restrict__ wt, const double* __restrict__ W, double tol,
                                                int m, double* __restrict__ sig, int* __restrict__ info)
{
    __shared__ double red[2][1024];
    double s[2] = {0.0, 0.0};
    for (int i = threadIdx.x; i < m; i += 1024) {
        s[0] += A[1 + i] * wt[i];
        s[1] += w[1 + i] * wt[i];
        const double r = W[i + (size_t)m * i];
        if (r * r * tol >= 1.0) atomicCAS(info, 0, i + 1);
    }
    for (int v = 0; v < 2; ++v) red[v][threadIdx.x] = s[v];
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off)
            for (int v = 0; v < 2; ++v) red[v][threadIdx.x] += red[v][threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        sig[0] = A[0] - red[0][0];
        sig[1] = red[1][0];
    }
}

bool sym_factor(ilh_plan* pl, SymFactor& F, int n, double* scratch, bool deflate)
{
    hipStream_t st = pl->ctx->stream;
    F.n = n;
    F.ok = false;
    const int m = n - 1, mc = std::max(m, 1);
    F.w.ensure(sizeof(double) * (size_t)n);
    F.vec.ensure(sizeof(double) * (size_t)(2 * n + mc));
    F.W.ensure(sizeof(double) * (size_t)mc * mc);
    F.T.ensure(sizeof(double) * (size_t)mc * n);   // also the product W B of a full solve
    F.info.ensure(3 * sizeof(double));   // {sigma, w1.wt}, then the pivot flag
    double* A = F.A.as<double>();
    double* w = F.w.as<double>();
    double* y = F.vec.as<double>();
    double* p = y + n;
    double* sig = F.info.as<double>();
    int* info = (int*)(sig + 2);
    k_house_vec<<<(n + 255) / 256, 256, 0, st>>>(w, n, deflate, info);
    if (deflate) {
        k_symv<<<(n + 3) / 4, 256, 0, st>>>(A, n, n, w, y);
        k_house_p<<<1, 1024, 0, st>>>(w, y, n, p);
        k_rank2<<<dim3((n + 255) / 256, n), 256, 0, st>>>(A, n, n, w, p);
    }
    ILH_HIP(hipGetLastError());
    if (m > 0) {
        chol_factor(st, A + 1 + (size_t)n, n, m, F.W.as<double>(), scratch, F.T.as<double>(), info);
        // wt = Mt^-1 beta (y is free)
        k_wmv<<<(m + 15) / 16, 1024, 0, st>>>(F.W.as<double>(), m, A + 1, y);
        k_wtmv<<<(m + 3) / 4, 256, 0, st>>>(F.W.as<double>(), m, y, F.wt());
    }
    // without the deflation every pivot, sigma the last of them, has to stand
    // clear of rounding (M's entries are at most about 1): a pivot of coinciding
    // points comes out as rounding of either sign
    const double tol = deflate ? 0.0 : n * 2.220446049250313e-16;
    k_sigma<<<1, 1024, 0, st>>>(A, w, F.wt(), F.W.as<double>(), tol, m, sig, info);
    ILH_HIP(hipGetLastError());
    double h[3];
    ILH_HIP(hipMemcpyAsync(h, sig, sizeof(h), hipMemcpyDeviceToHost, st));
    ILH_HIP(hipStreamSynchronize(st));
    int bad;
    std::memcpy(&bad, h + 2, sizeof(bad));
    if (bad || !std::isfinite(h[0]) || (deflate ? h[0] == 0.0 : h[0] <= tol)) return false;
    F.ok = true;
    return true;
}

// The deflated solve's first reflection, X' = B - 2 w (w . B) in place, and its
// first coordinate y1 = (X'0 - wt . X'1) / sigma; a work-group per column of B
// (n rows), its first 2048 entries kept in registers between the two dots.
// Bound by the latency of one round of loads and two reductions; N = 1885:
// 12 us (a wave per column that read it twice: 26).
__global__ void __launch_bounds__(256) k_defl_cols(const double* __restrict__ w, const double* __restrict__ wt,
                                                   const double* __restrict__ sig, double* __restrict__ B, int n,
                                                   double* __restrict__ y1v)
{
    constexpr int E = 8;
    __shared__ double red[2][4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    double* col = B + (size_t)n * blockIdx.x;
    auto total = [&](double a, double* q) {
        for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
        if (lane == 0) q[wave] = a;
        __syncthreads();
        return (q[0] + q[1]) + (q[2] + q[3]);
    };
    double x[E], ww[E], r = 0.0;
#pragma unroll
    for (int u = 0; u < E; ++u) {
        const int i = t + 256 * u;
        x[u] = i < n ? col[i] : 0.0;
        ww[u] = i < n ? w[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < E; ++u) r = __builtin_fma(ww[u], x[u], r);
    for (int i = t + 256 * E; i < n; i += 256) r = __builtin_fma(w[i], col[i], r);
    r = total(r, red[0]);
    double s = 0.0, x0 = 0.0;   // x0: the first entry, thread 0's
    auto reflect = [&](int i, double wi, double b) {
        const double v = __builtin_fma(-2.0 * wi, r, b);
        col[i] = v;
        if (i == 0) x0 = v;
        else s = __builtin_fma(wt[i - 1], v, s);
    };
#pragma unroll
    for (int u = 0; u < E; ++u)
        if (t + 256 * u < n) reflect(t + 256 * u, ww[u], x[u]);
    for (int i = t + 256 * E; i < n; i += 256) reflect(i, w[i], col[i]);
    s = total(s, red[1]);
    if (t == 0) y1v[blockIdx.x] = (x0 - s) / sig[0];
}

// The last step of the deflated solve: the second reflection, of [y1; Z - wt y1],
// with its scalar t = w . [y1; Z - wt y1] taken from the stored Z itself,
//     t = w0 y1 + w1 . Z - (w1 . wt) y1:
// the reflection then leaves the constant mode at y1 whatever Z's rounding is.
// (From the right-hand side, w1 . Z = (Mt^-1 w1) . X'1, the error of Z in that
// direction stays in the solution as net charge: 150 to 20000 eps |x| for
// smooth data on 245 to 1885 points, against 1 to 75 eps |x|.)
// Out[j + ldo p] = ([y1; Z - wt y1] - 2 w t) / (c d[p]), Z in Out's rows 1..m;
// nd sums of w1 . Z at dots + ncols k.  A thread takes DR rows of a column j.
constexpr int DR = 32;

__global__ void __launch_bounds__(256) k_defl_rows(const double* __restrict__ w, const double* __restrict__ wt,
                                                   const double* __restrict__ sig, const double* __restrict__ y1v,
                                                   const double* __restrict__ dots, int nd, int n, int ncols,
                                                   const double* __restrict__ d, double c, double* __restrict__ Out,
                                                   int ldo)
{
    const int j = blockIdx.x * 256 + threadIdx.x, p0 = blockIdx.y * DR;
    if (j >= ncols) return;
    double q = 0.0;
#pragma unroll 8
    for (int k = 0; k < nd; ++k) q += dots[j + (size_t)ncols * k];
    const double y1 = y1v[j], w0 = w[0];
    const double t = w0 * y1 + q - sig[1] * y1;
    if (p0 == 0) Out[j] = (y1 - 2.0 * w0 * t) / (c * d[0]);
    const int p1 = min(p0 + DR, n);
#pragma unroll 8
    for (int p = max(p0, 1); p < p1; ++p) {
        double* o = Out + j + (size_t)ldo * p;
        *o = (*o - y1 * wt[p - 1] - 2.0 * t * w[p]) / (c * d[p]);
    }
}

// the same for a single column, in one work-group
__global__ void __launch_bounds__(1024) k_defl_vec(const double* __restrict__ w, const double* __restrict__ wt,
                                                   const double* __restrict__ sig, const double* __restrict__ y1v, int n,
                                                   const double* __restrict__ d, double c, double* __restrict__ Out)
{
    __shared__ double red[16];
    double q = 0.0;
    for (int p = 1 + threadIdx.x; p < n; p += 1024) q = __builtin_fma(w[p], Out[p], q);
    for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
    __syncthreads();
    q = 0.0;
    for (int k = 0; k < 16; ++k) q += red[k];
    const double y1 = y1v[0], w0 = w[0];
    const double t = w0 * y1 + q - sig[1] * y1;
    if (threadIdx.x == 0) Out[0] = (y1 - 2.0 * w0 * t) / (c * d[0]);
    for (int p = 1 + threadIdx.x; p < n; p += 1024) Out[p] = (Out[p] - y1 * wt[p - 1] - 2.0 * t * w[p]) / (c * d[p]);
}

// Out[j + ldo p] = (M^-1 B)[p, j] / (c d[p]) for B (n x ncols, leading
// dimension n, overwritten): the rows of diag(1 / (c d)) M^-1 B, each
// contiguous.  The second reflection needs the whole of W^T W X' (its dots come
// with the product, 32 columns of a tile at a time) and is a pass over the
// result.  A single column (ldo = 1) goes through the vector products instead
// of 64-wide tiles, and Out may be B then.  The reflections are 12 and 20 of a
// solve's 370 us at N = 1885, all columns.
void sym_solve_rows(ilh_plan* pl, SymFactor& F, double* B, int ncols, const double* d, double c, double* Out, int ldo)
{
    if (!F.ok) fail(ILH_ERR_STATE, "symmetric factor not built");
    if (ncols <= 0) return;
    hipStream_t st = pl->ctx->stream;
    const int n = F.n, m = n - 1;
    const bool vec = ncols == 1 && ldo == 1;
    const int nt = (m + GT - 1) / GT, nd = vec ? 0 : 2 * nt;
    F.r.ensure(sizeof(double) * (size_t)(1 + nd) * ncols);
    double *y1 = F.r.as<double>(), *dots = y1 + ncols;
    const double* w = F.w.as<double>();
    const double* sig = F.info.as<double>();
    k_defl_cols<<<ncols, 256, 0, st>>>(w, F.wt(), sig, B, n, y1);
    ILH_HIP(hipGetLastError());
    const double* W = F.W.as<double>();
    if (m > 0) {
        F.T.ensure(sizeof(double) * (size_t)m * ncols);
        double* T = F.T.as<double>();
        if (vec) {
            k_wmv<<<(m + 15) / 16, 1024, 0, st>>>(W, m, B + 1, T);
            k_wtmv<<<(m + 3) / 4, 256, 0, st>>>(W, m, T, Out + 1);
        } else {
            GemmDots e;
            e.v = w + 1;
            e.dots = dots;
            k_dgemm<0, true, false><<<dim3(nt, (ncols + GT - 1) / GT), 256, 0, st>>>(
                m, ncols, m, 1.0, W, m, B + 1, n, T, m, TRI_A_LOWER, GemmBatch(), GemmDots());
            k_dgemm<1, true, true><<<dim3((ncols + GT - 1) / GT, nt), 256, 0, st>>>(
                ncols, m, m, 1.0, T, m, W, m, Out + ldo, ldo, TRI_B_LOWER, GemmBatch(), e);
        }
        ILH_HIP(hipGetLastError());
    }
    if (vec) k_defl_vec<<<1, 1024, 0, st>>>(w, F.wt(), sig, y1, n, d, c, Out);
    else
        k_defl_rows<<<dim3((ncols + 255) / 256, (n + DR - 1) / DR), 256, 0, st>>>(w, F.wt(), sig, y1, dots, nd, n, ncols,
                                                                                d, c, Out, ldo);
    ILH_HIP(hipGetLastError());
}

// Minv (row-major, leading dimension solve_ld(n), the padding columns zero) =
// (M diag(c d))^-1 for the factor of sym_factor
__global__ void k_identity_cm(double* __restrict__ A, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= n) return;
    A[i + (size_t)n * j] = i == j ? 1.0 : 0.0;
}

__global__ void k_zero_pad(double* __restrict__ A, int n, int ld)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, pad = ld - n;
    if (i < n * pad) A[n + i % pad + (size_t)ld * (i / pad)] = 0.0;
}

void zero_pad_columns(hipStream_t st, double* A, int n, int ld)
{
    if (ld <= n || n <= 0) return;
    k_zero_pad<<<((unsigned)n * (ld - n) + 255) / 256, 256, 0, st>>>(A, n, ld);
    ILH_HIP(hipGetLastError());
}

void sym_inverse_rowmajor(ilh_plan* pl, SymFactor& F, const double* d, double c, double* Minv)
{
    hipStream_t st = pl->ctx->stream;
    const int n = F.n, ld = solve_ld(n);
    // A's storage holds the identity
    k_identity_cm<<<dim3((n + 255) / 256, n), 256, 0, st>>>(F.A.as<double>(), n);
    ILH_HIP(hipGetLastError());
    sym_solve_rows(pl, F, F.A.as<double>(), n, d, c, Minv, ld);
    zero_pad_columns(st, Minv, n, ld);
    ILH_HIP(hipStreamSynchronize(st));   // F may be released on return
}

}  // namespace ilh
