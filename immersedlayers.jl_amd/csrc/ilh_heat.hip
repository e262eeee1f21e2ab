// ilh_heat.hip -- unbounded heat conduction with Dirichlet bodies, advanced by
// the integrating-factor half-explicit Runge-Kutta method (IF-HERK).
//
// The reference poses the problem as the constrained ODE system
//   dT/dt = kappa L T + r1 + R sigma,   E T = r2
// (test/literate/heatconduction.jl:88-130: r1 = surface_divergence!(-kappa [T]),
// constraint force regularize!(-(-sigma)), bc_op interpolate!, bc_rhs the
// surface average) and marches it with ConstrainedSystems' LiskaIFHERK
// (src/timemarching.jl:5, integrating factor for lin_op = kappa L).  IF-HERK
// applies a half-explicit RK scheme to v = exp(-(t - t_n) kappa L) T, so the
// stiff diffusion is integrated exactly; the 3-stage tableau (Liska & Colonius
// 2016) is
//   c = (0, 1/3, 1),  a21 = 1/3,  a31 = -1, a32 = 2,  b = (0, 3/4, 1/4),
// and the multiplier of each stage solves a Schur system
//   E exp((c_i - c_{i-1}) dt kappa L) R sigma = E Yhat_i - r2
// with the factors exp(dt/3 kappa L), exp(2dt/3 kappa L) and the identity.
//
// exp(tau kappa L) on the unbounded lattice is separable:
//   [exp(tau kappa L) u](i,j) = sum_{p,q} K(p) K(q) u(i-p, j-q),
//   K(p) = e^{-2a} I_p(2a),  a = tau kappa / dx^2,
// applied here as an x and a y pass of a (2M+1)-tap filter (zero outside the
// grid), in one kernel for filters of at most 16 taps a side.  The three Schur
// matrices are assembled directly from K(p)K(q) like the LGF ones and inverted
// once; their inverses decay away from the diagonal of the bodies' curves, and
// only the entries that count are kept and applied.
//
// The step (H13, H23 the two factors, W_i = F + R sigma_i, F = r1):
//   G  = H13 T                                            whole grid
//   E G + dt a21 E H13 F = r2 + ...      -> sigma_1        (E H13 F kept)
//   A  = G + dt a31 H13 W_1 + dt a32 F                     tiles near the bodies
//   Y  = H23 A                                             tiles near the bodies
//   E Y = r2 + ...                       -> sigma_2
//   T  = H23 (G + dt b2 W_2) + dt b3 F                     whole grid
//   E T = r2 + ...                       -> sigma_3,  T += dt b3 R sigma_3
// the scheme's stages with the filter's linearity used: F and the W_i are zero
// away from the bodies, and the intermediate stages are needed only where E
// reads them, so two passes over the grid serve a step (of five).  With a filter
// of more than 16 taps a side a step keeps the five passes (ilh_heat_advance).
#include "ilh_internal.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace ilh {
// An inverse stage matrix, row p as the 32-column chunks of it that count:
// chunk k of row p (ptr[p] <= k < ptr[p + 1]) holds columns 32 idx[k] .. + 31
// at val + 32 k.  Entries below eps / (16 N) of their row's largest are left
// out (all of them together below eps / 16 of it): the stage matrices couple
// points a few filter widths apart, so their inverses decay by about a digit
// every two or three points along a curve.
struct StageInverse {
    DevBuf ptr, idx, val;
};
}  // namespace ilh

struct ilh_heat {
    ilh_plan* pl = nullptr;
    unsigned gen = 0;
    double kappa = 0.0, dt = 0.0;
    int M13 = 0, M23 = 0;                 // filter half-widths
    ilh::DevBuf k13, k23;                 // K(0..M) of exp(dt/3 kL), exp(2dt/3 kL)
    ilh::StageInverse S13, S23, S0;       // inverse stage Schur matrices
    ilh::DevBuf F, A, Bt, Y, W1, W2;  // grid fields
    ilh::DevBuf e, sg, r2, r2s;           // surface vectors; r2s = r2 - dt a21 E H13 F
    // the 64 x 64 tiles near the bodies.  near[t]: F or a W_i may be nonzero
    // within 16 cells of tile t; the lists hold those tiles and the ones E reads
    // (touch)
    ilh::DevBuf near, near_list, touch_list;
    int n_near = 0, n_touch = 0;
    bool have_bc = false;
};

namespace ilh {

// K(p) = e^{-x} I_p(x), x = 2a, p = 0..M, by backward recurrence normalised
// with e^{x} = I_0(x) + 2 sum_{p>=1} I_p(x) (so sum over all p of K(p) = 1);
// truncated after the last p with K(p) > 1e-17 K(0).
static std::vector<double> heat_kernel_1d(double a)
{
    if (a <= 0.0) return {1.0};
    const double x = 2.0 * a;
    const int top = (int)(2.0 * x + 60.0 + 10.0 * std::sqrt(x));
    std::vector<double> v(top + 2, 0.0);
    v[top + 1] = 0.0;
    v[top] = 1e-280;
    for (int p = top; p >= 1; --p) {
        v[p - 1] = (2.0 * p / x) * v[p] + v[p + 1];
        if (v[p - 1] > 1e250)   // rescale to stay in range
            for (int q = p - 1; q <= top + 1; ++q) v[q] *= 1e-250;
    }
    double sum = v[0];
    for (int p = 1; p <= top; ++p) sum += 2.0 * v[p];
    std::vector<double> K;
    for (int p = 0; p <= top; ++p) {
        const double k = v[p] / sum;
        if (p > 0 && k <= 1e-17 * (v[0] / sum)) break;
        K.push_back(k);
    }
    return K;
}

namespace {

constexpr int HX = 64, HY = 4;          // naive kernels (long filters)
constexpr int XT = 256, XR = 8;          // x pass: 256-wide row segments, 8 rows per work-group
constexpr int YC = 64, YR = 64;          // y pass: columns x rows of outputs per work-group
constexpr int MX_LDS = 64, MY_LDS = 32;  // longest filters the tiled passes take

// x pass: out(i,j) = sum_{|p|<=M} K(|p|) u(i-p, j), u = a + c b (b may be
// null), zero outside [0, nx).  Eight row segments and their halos are
// staged in LDS; every thread issues all of its loads before the first store.
__global__ void __launch_bounds__(XT) k_heat_x(const double* __restrict__ a, double c, const double* __restrict__ b,
                                               int nx, int ny, const double* __restrict__ K, int M,
                                               double* __restrict__ out)
{
    constexpr int W = XT + 2 * MX_LDS;
    __shared__ double buf[XR][W];
    const int j0 = blockIdx.y * XR, x0 = blockIdx.x * XT, t = threadIdx.x;
    const int w = XT + 2 * M;
    double va[XR][2], vb[XR][2];
#pragma unroll
    for (int r = 0; r < XR; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e = t + XT * q, x = x0 - M + e, j = j0 + r;
            const bool in = e < w && x >= 0 && x < nx && j < ny;
            va[r][q] = in ? a[x + (size_t)nx * j] : 0.0;
            vb[r][q] = in && b ? b[x + (size_t)nx * j] : 0.0;
        }
#pragma unroll
    for (int r = 0; r < XR; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e = t + XT * q;
            if (e < w) buf[r][e] = b ? va[r][q] + c * vb[r][q] : va[r][q];
        }
    __syncthreads();
    const int i = x0 + t;
    if (i >= nx) return;
#pragma unroll
    for (int r = 0; r < XR; ++r) {
        const int j = j0 + r;
        if (j >= ny) break;
        const double* row = buf[r] + t + M;
        double acc = K[0] * row[0];
        for (int p = 1; p <= M; ++p) acc += K[p] * (row[-p] + row[p]);
        out[i + (size_t)nx * j] = acc;
    }
}

// y pass: out(i,j) = sum_{|p|<=M} K(|p|) in(i, j-p) + c add(i,j) (add may be
// null), zero outside [0, ny).  A 64-column strip of YR + 2M rows is staged
// in LDS (dynamic, (YR + 2M) x 64 doubles); loads, including those of `add`,
// are all issued before the strip is stored.
__global__ void __launch_bounds__(256) k_heat_y(const double* __restrict__ in, int nx, int ny,
                                                const double* __restrict__ K, int M, double c,
                                                const double* __restrict__ add, double* __restrict__ out)
{
    extern __shared__ double strip[];   // [YR + 2M][YC]
    constexpr int QMAX = (YR + 2 * MY_LDS) / 4;
    const int tx = threadIdx.x & (YC - 1), ty = threadIdx.x / YC;   // 64 x 4
    const int i = blockIdx.x * YC + tx, y0 = blockIdx.y * YR;
    const int rows = YR + 2 * M;
    double v[QMAX], ad[YR / 4];
#pragma unroll
    for (int q = 0; q < QMAX; ++q) {
        const int r = ty + 4 * q, y = y0 - M + r;
        v[q] = (r < rows && i < nx && y >= 0 && y < ny) ? in[i + (size_t)nx * y] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < YR / 4; ++q) {
        const int y = y0 + ty + 4 * q;
        ad[q] = (add && i < nx && y < ny) ? add[i + (size_t)nx * y] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < QMAX; ++q) {
        const int r = ty + 4 * q;
        if (r < rows) strip[r * YC + tx] = v[q];
    }
    __syncthreads();
    if (i >= nx) return;
#pragma unroll
    for (int q = 0; q < YR / 4; ++q) {
        const int r = ty + 4 * q, y = y0 + r;
        if (y >= ny) break;
        const double* col = strip + (r + M) * YC + tx;
        double acc = K[0] * col[0];
        for (int p = 1; p <= M; ++p) acc += K[p] * (col[-p * YC] + col[p * YC]);
        out[i + (size_t)nx * y] = add ? acc + c * ad[q] : acc;
    }
}

constexpr int YMB = 16;   // longest filter (taps a side) of the one-kernel pass

// the same passes for filters longer than the tiled ones take
__global__ void k_heat_x_long(const double* __restrict__ a, double c, const double* __restrict__ b, int nx, int ny,
                              const double* __restrict__ K, int M, double* __restrict__ out)
{
    const int i = blockIdx.x * HX + threadIdx.x, j = blockIdx.y * HY + threadIdx.y;
    if (i >= nx || j >= ny) return;
    const double* ra = a + (size_t)nx * j;
    const double* rb = b ? b + (size_t)nx * j : nullptr;
    auto u = [&](int x) { return rb ? ra[x] + c * rb[x] : ra[x]; };
    double acc = K[0] * u(i);
    for (int p = 1; p <= M; ++p) {
        const double l = i - p >= 0 ? u(i - p) : 0.0;
        const double r = i + p < nx ? u(i + p) : 0.0;
        acc += K[p] * (l + r);
    }
    out[i + (size_t)nx * j] = acc;
}

__global__ void k_heat_y_long(const double* __restrict__ in, int nx, int ny, const double* __restrict__ K, int M,
                              double c, const double* __restrict__ add, double* __restrict__ out)
{
    const int i = blockIdx.x * HX + threadIdx.x, j = blockIdx.y * HY + threadIdx.y;
    if (i >= nx || j >= ny) return;
    double acc = K[0] * in[i + (size_t)nx * j];
    for (int p = 1; p <= M; ++p) {
        const double l = j - p >= 0 ? in[i + (size_t)nx * (j - p)] : 0.0;
        const double r = j + p < ny ? in[i + (size_t)nx * (j + p)] : 0.0;
        acc += K[p] * (l + r);
    }
    const size_t o = i + (size_t)nx * j;
    out[o] = add ? acc + c * add[o] : acc;
}

// One tile's pass of the whole 2-D filter: out = H(cin in + cb b) + g + cadd add
// (b, g, add may be null; b and add are read in the tiles that near marks, in
// all of them without near), zero outside the grid.  out must not be in or b.
struct TilePass {
    const double* in = nullptr;
    double cin = 1.0;
    const double* b = nullptr;
    double cb = 0.0;
    const double* g = nullptr;
    const double* add = nullptr;
    double cadd = 0.0;
    const unsigned char* near = nullptr;
    const double* K = nullptr;
    int M = 0;
    double* out = nullptr;
    int nx = 0, ny = 0;
    const int* list = nullptr;   // tiles to do (null: all of them)
};
constexpr int HT = 64;   // tile edge
constexpr int HTH = 512; // threads per tile

// A work-group filters one 64 x 64 tile: the tile and a halo of MB cells are
// staged in LDS (MB >= M, taps past M zero); the x pass takes eight
// neighbouring outputs of one row per task from a register window of 8 + 2 MB
// values, consecutive lanes on consecutive rows (odd row stride: no bank
// conflicts), and writes back over the stage; the y pass takes 8 rows of one
// column per thread the same way.  One read of the field (its halo mostly from
// L2: neighbouring tiles run on one XCD) and one write, where an x and a y
// kernel read and write it twice.  2048^2: 23 us at M = 10, 27 us at M = 12
// (an x and a y kernel: 41 us), of which memory's share (33.5 MB in and out)
// is about 12 us and FP64 issue's about 8; two work-groups of eight waves per
// CU overlap them (of four waves each: 28 and 33 us).  The forms for 14 and 16
// taps spill 15 and 38 registers under that cap; a step at 2048^2 with 3000
// points takes 105 us at 12 taps, 114 at 14 and 130 at 16.
template <int MB>
__global__ void __launch_bounds__(HTH, 4) k_heat_xy(TilePass P)
{
    constexpr int W = HT + 2 * MB, WS = W + 1, NT = (W * (HT / 8) + HTH - 1) / HTH, NL = (W * W + HTH - 1) / HTH;
    __shared__ double buf[W][WS];
    const int t = threadIdx.x, tiles_x = (P.nx + HT - 1) / HT, ntiles = tiles_x * ((P.ny + HT - 1) / HT);
    int tile;
    if (P.list) {
        tile = P.list[blockIdx.x];
    } else {   // each XCD takes a run of neighbouring tiles
        const int per = (ntiles + 7) / 8;
        tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if (tile >= ntiles) return;
    }
    const int x0 = tile % tiles_x * HT, y0 = tile / tiles_x * HT;
    const bool near = !P.near || P.near[tile];
    const bool use_b = P.b && near, use_add = P.add && near;
    // the whole stage's loads go out together: one memory round trip
    {
        double v[NL];
        auto load = [&](const double* f, int q) {
            const int e = t + HTH * q, r = e / W, x = x0 - MB + e - r * W, y = y0 - MB + r;
            const bool in = e < W * W && x >= 0 && x < P.nx && y >= 0 && y < P.ny;
            return in ? f[x + (size_t)P.nx * y] : 0.0;
        };
#pragma unroll
        for (int q = 0; q < NL; ++q) v[q] = load(P.in, q);
        if (use_b) {
#pragma unroll
            for (int h = 0; h < NL; h += 8) {   // eight at a time (registers); near tiles only
                double vb[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) vb[q] = h + q < NL ? load(P.b, h + q) : 0.0;
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (h + q < NL) v[h + q] = __builtin_fma(P.cb, vb[q], P.cin * v[h + q]);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NL; ++q) v[q] *= P.cin;
        }
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int e = t + HTH * q, r = e / W;
            if (e < W * W) buf[r][e - r * W] = v[q];
        }
    }
    double kk[MB + 1];
#pragma unroll
    for (int p = 0; p <= MB; ++p) kk[p] = p <= P.M ? P.K[p] : 0.0;
    __syncthreads();
    double o[NT][8];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int task = t + HTH * q, r = task % W, c0 = task / W * 8;
        if (task < W * (HT / 8)) {
            double w[8 + 2 * MB];
#pragma unroll
            for (int k = 0; k < 8 + 2 * MB; ++k) w[k] = buf[r][c0 + k];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                double acc = kk[0] * w[c + MB];
#pragma unroll
                for (int p = 1; p <= MB; ++p) acc = __builtin_fma(kk[p], w[c + MB - p] + w[c + MB + p], acc);
                o[q][c] = acc;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int task = t + HTH * q, r = task % W, c0 = task / W * 8;
        if (task < W * (HT / 8))
#pragma unroll
            for (int c = 0; c < 8; ++c) buf[r][c0 + c] = o[q][c];
    }
    __syncthreads();
    constexpr int YO = HT * HT / HTH;   // rows per thread
    const int tx = t & 63, ty = t >> 6, x = x0 + tx, yb = y0 + YO * ty;
    if (x >= P.nx) return;
    double g[YO], ad[YO], w[YO + 2 * MB];
#pragma unroll
    for (int u = 0; u < YO; ++u) {
        const int y = yb + u;
        const size_t at = y < P.ny ? x + (size_t)P.nx * y : 0;
        g[u] = P.g && y < P.ny ? P.g[at] : 0.0;
        ad[u] = use_add && y < P.ny ? P.add[at] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < YO + 2 * MB; ++k) w[k] = buf[YO * ty + k][tx];
#pragma unroll
    for (int u = 0; u < YO; ++u) {
        const int y = yb + u;
        double acc = kk[0] * w[u + MB];
#pragma unroll
        for (int p = 1; p <= MB; ++p) acc = __builtin_fma(kk[p], w[u + MB - p] + w[u + MB + p], acc);
        if (y < P.ny) P.out[x + (size_t)P.nx * y] = __builtin_fma(P.cadd, ad[u], acc + g[u]);
    }
}

// near[t] = 1 for the tiles within 16 cells of a cell that D_s or R of some
// point touches, touch[t] = 1 for those that E reads (windows of four cells
// from the term's corner on; D_s reaches one cell further on each side)
__global__ void k_heat_mark(const Term* __restrict__ t, int N, int nx, int ny, unsigned char* __restrict__ near,
                            unsigned char* __restrict__ touch)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int bx = t[p].bx, by = t[p].by, tx = (nx + HT - 1) / HT;
    auto mark = [&](int lo, int hi, unsigned char* f) {
        for (int j = max(by + lo, 0) / HT; j <= min(by + hi, ny - 1) / HT; ++j)
            for (int i = max(bx + lo, 0) / HT; i <= min(bx + hi, nx - 1) / HT; ++i) f[i + tx * j] = 1;
    };
    mark(-1 - YMB, 4 + YMB, near);
    mark(0, 3, touch);
}

// a = b = f on the listed tiles
__global__ void __launch_bounds__(256) k_heat_copy_tiles(const double* __restrict__ f, const int* __restrict__ list, int nx,
                                                         int ny, double* __restrict__ a, double* __restrict__ b)
{
    const int tx = (nx + HT - 1) / HT, x = list[blockIdx.x] % tx * HT + (threadIdx.x & 63);
    if (x >= nx) return;
    for (int r = threadIdx.x >> 6; r < HT; r += 4) {
        const int y = list[blockIdx.x] / tx * HT + r;
        if (y < ny) a[x + (size_t)nx * y] = b[x + (size_t)nx * y] = f[x + (size_t)nx * y];
    }
}

// e = E field - r: sixteen lanes per point, one per tap of its 4 x 4 window
__global__ void __launch_bounds__(256) k_heat_gather(const Term* __restrict__ t, int N, const double* __restrict__ f,
                                                     int nx, int ny, const double* __restrict__ r,
                                                     double* __restrict__ e)
{
    const int k = blockIdx.x * 256 + threadIdx.x, p = k >> 4, l = k & 15;
    if (p >= N) return;   // uniform over the point's lanes
    const Term& tt = t[p];
    const int col = tt.bx + (l & 3), row = tt.by + (l >> 2);
    double v = 0.0;
    if (row >= 0 && row < ny && col >= 0 && col < nx)
        v = tt.coef * (tt.wy[l >> 2] * tt.wx[l & 3]) * f[col + (size_t)nx * row];
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (l == 0) e[p] = r ? v - r[p] : v;
}

// out = base + c R amp on the cells that R touches (base may be out), a wave per row
__global__ void __launch_bounds__(64) k_heat_cells(const int* __restrict__ cell_ptr, const int4* __restrict__ cells,
                                                   const int* __restrict__ cai, const double* __restrict__ cw, int nx,
                                                   const double* __restrict__ amp, const double* base, double c,
                                                   double* out)
{
    const int j = blockIdx.x, c1 = cell_ptr[j + 1];
    for (int ci = cell_ptr[j] + threadIdx.x; ci < c1; ci += 64) {
        const int4 cr = cells[ci];
        double acc = 0.0;
        for (int k = cr.y; k < cr.z; ++k) acc += amp[cai[k]] * cw[k];
        const size_t at = cr.x + (size_t)nx * j;
        out[at] = base[at] + c * acc;
    }
}

// Packing an inverse (row-major, leading dimension ld, a multiple of 32), a
// wave per row: the number of chunks that count, then the chunks.
__device__ __forceinline__ double row_threshold(const double* row, int n, int lane)
{
    double m = 0.0;
    for (int k = lane; k < n; k += 64) m = fmax(m, fabs(row[k]));
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    return m * (1.1102230246251565e-16 / 16.0) / n;
}

__global__ void __launch_bounds__(256) k_pack_count(const double* __restrict__ A, int n, int ld, int* __restrict__ cnt)
{
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= n) return;
    const double* row = A + (size_t)ld * p;
    const double thr = row_threshold(row, n, lane);
    int c = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
        // (written so that a NaN counts)
        const unsigned long long m = __ballot(k0 + lane < n && !(fabs(row[min(k0 + lane, n - 1)]) <= thr));
        c += ((unsigned)m ? 1 : 0) + ((unsigned)(m >> 32) ? 1 : 0);
    }
    if (lane == 0) cnt[p] = c;
}

__global__ void __launch_bounds__(256) k_pack_rows(const double* __restrict__ A, int n, int ld, const int* __restrict__ ptr,
                                                   int* __restrict__ idx, double* __restrict__ val)
{
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= n) return;
    const double* row = A + (size_t)ld * p;
    const double thr = row_threshold(row, n, lane);
    int c = ptr[p];
    for (int k0 = 0; k0 < n; k0 += 64) {
        const bool in = k0 + lane < n;
        const double v = in ? row[k0 + lane] : 0.0;
        const unsigned long long m = __ballot(in && !(fabs(v) <= thr));
        const bool lo = (unsigned)m != 0, hi = (unsigned)(m >> 32) != 0;
        const int at = c + (lane >= 32 && lo ? 1 : 0);
        if (lane < 32 ? lo : hi) {
            val[32 * (size_t)at + (lane & 31)] = v;
            if ((lane & 31) == 0) idx[at] = k0 / 32 + (lane >> 5);
        }
        c += (lo ? 1 : 0) + (hi ? 1 : 0);
    }
}

// y = alpha A x for a packed inverse, a wave per row (two chunks at a time);
// x has room for whole chunks, zero past its end.  Bound by the latency of its
// two dependent loads: N = 5465 at Fo = 0.25, 4.5 us (dense, 239 MB: 55 us).
__global__ void __launch_bounds__(256) k_packed_matvec(const int* __restrict__ ptr, const int* __restrict__ idx,
                                                       const double* __restrict__ val, const double* __restrict__ x,
                                                       double* __restrict__ y, int n, double alpha)
{
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= n) return;
    const int c1 = ptr[p + 1];
    double s = 0.0;
#pragma unroll 4
    for (int c = ptr[p] + (lane >> 5); c < c1; c += 2)
        s = __builtin_fma(val[32 * (size_t)c + (lane & 31)], x[32 * idx[c] + (lane & 31)], s);
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) y[p] = alpha * s;
}

// d = Tb+ - Tb- (scaled by -kappa), r2 = (Tb+ + Tb-)/2
__global__ void k_heat_bc(const double* __restrict__ tp, const double* __restrict__ tm, int n, double kappa,
                          double* __restrict__ dneg, double* __restrict__ r2)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double a = tp[k], b = tm ? tm[k] : 0.0;
    dneg[k] = -kappa * (a - b);
    r2[k] = 0.5 * (a + b);
}

}  // namespace

// e = E field - r (r may be null: e = E field)
static void heat_gather(ilh_plan* pl, const double* field, const double* r, double* e)
{
    k_heat_gather<<<(16 * pl->N + 255) / 256, 256, 0, pl->ctx->stream>>>(
        get_terms(pl, OP_E_PRIMAL), pl->N, field, pl->g.nx(GK_PRIMAL), pl->g.ny(GK_PRIMAL), r, e);
    ILH_HIP(hipGetLastError());
}

// out = H in ... over a list of n tiles, or the whole grid (n < 0); P.M <= YMB
static void tile_pass(ilh_plan* pl, TilePass P, const int* list = nullptr, int n = -1)
{
    P.nx = pl->g.nx(GK_PRIMAL);
    P.ny = pl->g.ny(GK_PRIMAL);
    P.list = n < 0 ? nullptr : list;
    const int ntiles = ((P.nx + HT - 1) / HT) * ((P.ny + HT - 1) / HT);
    const int blocks = n < 0 ? (ntiles + 7) / 8 * 8 : n;
    if (blocks == 0) return;
    hipStream_t st = pl->ctx->stream;
    // the halo is the filter's, to the next even width
    if (P.M <= 8) k_heat_xy<8><<<blocks, HTH, 0, st>>>(P);
    else if (P.M <= 10) k_heat_xy<10><<<blocks, HTH, 0, st>>>(P);
    else if (P.M <= 12) k_heat_xy<12><<<blocks, HTH, 0, st>>>(P);
    else if (P.M <= 14) k_heat_xy<14><<<blocks, HTH, 0, st>>>(P);
    else k_heat_xy<YMB><<<blocks, HTH, 0, st>>>(P);
    ILH_HIP(hipGetLastError());
}

// out = exp(tau kappa L) (a + ca b) + cp add   (b, add may be null; tmp: one
// grid field of scratch; out may be add, not a or b): in one pass for filters
// of at most 16 taps a side, as the shorter one of a step is up to Fo = 1.6, an
// x and a y pass for longer ones.  A step at 2048^2, N = 3000, Fo = 1.25:
// 324 us (its three short passes in two each: 376).
static void heat_apply(ilh_plan* pl, const double* K, int M, const double* a, double ca, const double* b,
                       double* tmp, double* out, double cp = 0.0, const double* add = nullptr)
{
    const int nx = pl->g.nx(GK_PRIMAL), ny = pl->g.ny(GK_PRIMAL);
    hipStream_t st = pl->ctx->stream;
    if (M <= YMB) {
        TilePass P;
        P.in = a;
        P.b = b;
        P.cb = ca;
        P.add = add;
        P.cadd = cp;
        P.K = K;
        P.M = M;
        P.out = out;
        tile_pass(pl, P);
        return;
    }
    if (M <= MX_LDS)
        k_heat_x<<<dim3((nx + XT - 1) / XT, (ny + XR - 1) / XR), XT, 0, st>>>(a, ca, b, nx, ny, K, M, tmp);
    else
        k_heat_x_long<<<dim3((nx + HX - 1) / HX, (ny + HY - 1) / HY), dim3(HX, HY), 0, st>>>(a, ca, b, nx, ny, K, M,
                                                                                          tmp);
    if (M <= MY_LDS)
        k_heat_y<<<dim3((nx + YC - 1) / YC, (ny + YR - 1) / YR), 256, sizeof(double) * (YR + 2 * M) * YC, st>>>(
            tmp, nx, ny, K, M, cp, add, out);
    else
        k_heat_y_long<<<dim3((nx + HX - 1) / HX, (ny + HY - 1) / HY), dim3(HX, HY), 0, st>>>(tmp, nx, ny, K, M, cp,
                                                                                          add, out);
    ILH_HIP(hipGetLastError());
}

// 2-D kernel table K(m)K(n), (M+1)^2, for the Schur assembly
// The stage Schur matrix E H R = M diag(ds / dx^2) with M = E H E^T symmetric
// positive definite (H the heat kernel, or the identity): inverted through the
// Cholesky of M, LU of E H R if that meets a non-positive pivot, and packed.
// F, inv: storage shared by the stages.
static void schur_inverse(ilh_plan* pl, const std::vector<double>& K, bool identity, bool deflate, SymFactor& F, DevBuf& inv,
                          StageInverse& out)
{
    const int N = pl->N;
    hipStream_t st = pl->ctx->stream;
    DevBuf tabd;
    int T = 1;
    if (!identity) {
        T = (int)K.size();
        std::vector<double> tab((size_t)T * T);
        for (int n = 0; n < T; ++n)
            for (int m = 0; m < T; ++m) tab[m + (size_t)T * n] = K[m] * K[n];
        tabd.ensure(sizeof(double) * tab.size());
        ILH_HIP(hipMemcpyAsync(tabd.p, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice, st));
        ILH_HIP(hipStreamSynchronize(st));
    }
    auto build = [&](int opB, double* out) {
        if (identity) assemble(pl, OP_E_PRIMAL, opB, GK_PRIMAL, 1.0, true, out);
        else assemble_table(pl, OP_E_PRIMAL, opB, tabd.as<double>(), T, 1.0, out);
    };
    const int ld = solve_ld(N);
    inv.ensure(sizeof(double) * (size_t)N * ld);
    F.A.ensure(sizeof(double) * (size_t)N * N);
    // E H E^T is positive definite by itself, and without the deflation's
    // dense reflection its inverse keeps the stage matrix's decay: so for
    // filters of at most 16 taps a side (condition numbers of some tens).
    // Longer ones make it all but singular (4e15 at Fo = 50), where deflating
    // the constant mode first keeps an order of magnitude more of the solution.
    // LU takes over from a non-positive pivot, and from one at rounding level of
    // a short filter's matrix: that is points that coincide or are so close that
    // the pivot's sign is chance; LU refuses the former (of 90 geometries with
    // one point twice, the deflated factor as a second attempt took half).
    build(OP_E_PRIMAL, F.A.as<double>());
    if (sym_factor(pl, F, N, inv.as<double>(), deflate)) {
        sym_inverse_rowmajor(pl, F, pl->ds.as<double>(), 1.0 / (pl->g.dx * pl->g.dx), inv.as<double>());
    } else {
        DevBuf S;
        S.ensure(sizeof(double) * (size_t)N * N);
        build(OP_R_PRIMAL, S.as<double>());
        inverse_rowmajor(pl, S.as<double>(), inv.as<double>());
    }
    // pack
    DevBuf cnt;
    cnt.ensure(sizeof(int) * (size_t)N);
    k_pack_count<<<(N + 3) / 4, 256, 0, st>>>(inv.as<double>(), N, ld, cnt.as<int>());
    ILH_HIP(hipGetLastError());
    std::vector<int> ptr(N + 1, 0);
    ILH_HIP(hipMemcpyAsync(ptr.data() + 1, cnt.p, sizeof(int) * (size_t)N, hipMemcpyDeviceToHost, st));
    ILH_HIP(hipStreamSynchronize(st));
    for (int p = 0; p < N; ++p) ptr[p + 1] += ptr[p];
    out.ptr.ensure(sizeof(int) * (size_t)(N + 1));
    out.idx.ensure(sizeof(int) * (size_t)std::max(1, ptr[N]));
    out.val.ensure(sizeof(double) * 32 * (size_t)std::max(1, ptr[N]));
    ILH_HIP(hipMemcpyAsync(out.ptr.p, ptr.data(), sizeof(int) * (size_t)(N + 1), hipMemcpyHostToDevice, st));
    k_pack_rows<<<(N + 3) / 4, 256, 0, st>>>(inv.as<double>(), N, ld, out.ptr.as<int>(), out.idx.as<int>(),
                                            out.val.as<double>());
    ILH_HIP(hipGetLastError());
    ILH_HIP(hipStreamSynchronize(st));   // ptr and cnt are released on return
}

}  // namespace ilh

using namespace ilh;

namespace {
constexpr double A21 = 1.0 / 3.0, A31 = -1.0, A32 = 2.0, B2 = 0.75, B3 = 0.25;
}

extern "C" int ilh_heat_create(ilh_plan* pl, double kappa, double dt, ilh_heat** out)
{
    return guarded_call([&] {
        if (!pl || !out) fail(ILH_ERR_ARG, "null argument");
        if (!(kappa > 0.0) || !(dt > 0.0) || !std::isfinite(kappa * dt)) fail(ILH_ERR_ARG, "kappa and dt must be positive");
        ILH_HIP(hipSetDevice(pl->ctx->device));
        if (pl->N > 0) need_margin(pl, "heat conduction");
        drop_spare(pl);
        const double a13 = kappa * dt / 3.0 / (pl->g.dx * pl->g.dx);
        const std::vector<double> K13 = heat_kernel_1d(a13), K23 = heat_kernel_1d(2.0 * a13);
        if ((int)K23.size() > 256) fail(ILH_ERR_ARG, "time step too large for the integrating-factor filter (a > ~40)");
        ilh_heat* h = new ilh_heat();
        try {
            h->pl = pl;
            h->gen = pl->gen;
            h->kappa = kappa;
            h->dt = dt;
            h->M13 = (int)K13.size() - 1;
            h->M23 = (int)K23.size() - 1;
            hipStream_t st = pl->ctx->stream;
            h->k13.ensure(sizeof(double) * K13.size());
            h->k23.ensure(sizeof(double) * K23.size());
            ILH_HIP(hipMemcpyAsync(h->k13.p, K13.data(), sizeof(double) * K13.size(), hipMemcpyHostToDevice, st));
            ILH_HIP(hipMemcpyAsync(h->k23.p, K23.data(), sizeof(double) * K23.size(), hipMemcpyHostToDevice, st));
            const size_t ng = pl->g.n(GK_PRIMAL);
            for (DevBuf* b : {&h->F, &h->A, &h->Bt, &h->Y, &h->W1, &h->W2}) b->ensure(sizeof(double) * ng);
            const int N = pl->N;
            const int ld = solve_ld(std::max(1, N));
            for (DevBuf* b : {&h->e, &h->sg, &h->r2, &h->r2s}) b->ensure(sizeof(double) * ld);
            fill_zero(st, h->e.as<double>(), ld);   // the packed products read whole chunks
            if (N > 0) {
                SymFactor F;
                DevBuf inv;
                const bool lng = h->M23 > YMB;
                schur_inverse(pl, K13, false, lng, F, inv, h->S13);
                schur_inverse(pl, K23, false, lng, F, inv, h->S23);
                schur_inverse(pl, {1.0}, true, lng, F, inv, h->S0);
                const int nx = pl->g.nx(GK_PRIMAL), ny = pl->g.ny(GK_PRIMAL);
                const size_t nt = (size_t)((nx + HT - 1) / HT) * ((ny + HT - 1) / HT), pad = (nt + 7) / 8 * 8;
                h->near.ensure(2 * pad);
                unsigned char* near = h->near.as<unsigned char>();
                fill_zero(st, (double*)near, 2 * pad / 8);
                k_heat_mark<<<(N + 255) / 256, 256, 0, st>>>(get_terms(pl, OP_E_PRIMAL), N, nx, ny, near,
                                                            near + pad);
                ILH_HIP(hipGetLastError());
                std::vector<unsigned char> f(2 * pad);
                ILH_HIP(hipMemcpyAsync(f.data(), near, 2 * pad, hipMemcpyDeviceToHost, st));
                ILH_HIP(hipStreamSynchronize(st));
                // F and the W_i are nonzero on near tiles only, and set there with the boundary values
                for (DevBuf* w : {&h->W1, &h->W2}) fill_zero(st, w->as<double>(), ng);
                auto list = [&](const unsigned char* on, DevBuf& buf) {
                    std::vector<int> l;
                    for (size_t k = 0; k < nt; ++k)
                        if (on[k]) l.push_back((int)k);
                    buf.ensure(sizeof(int) * std::max<size_t>(1, l.size()));
                    ILH_HIP(hipMemcpyAsync(buf.p, l.data(), sizeof(int) * l.size(), hipMemcpyHostToDevice, st));
                    ILH_HIP(hipStreamSynchronize(st));   // l is released on return
                    return (int)l.size();
                };
                h->n_near = list(f.data(), h->near_list);
                h->n_touch = list(f.data() + pad, h->touch_list);
            }
            ILH_HIP(hipStreamSynchronize(st));
        } catch (...) {
            delete h;
            throw;
        }
        plan_retain(pl);
        *out = h;
    });
}

extern "C" int ilh_heat_set_boundary(ilh_heat* h, const double* tb_plus, const double* tb_minus, int mem)
{
    return guarded_call([&] {
        if (!h) fail(ILH_ERR_ARG, "null heat plan");
        ilh_plan* pl = h->pl;
        if (pl->gen != h->gen) fail(ILH_ERR_STATE, "the plan's geometry changed since ilh_heat_create");
        Io io(pl, mem);
        const int N = pl->N;
        hipStream_t st = pl->ctx->stream;
        if (N > 0) {
            const double* tp = io.in(tb_plus, N, pl->io_a);
            const double* tm = tb_minus ? io.in(tb_minus, N, pl->io_c) : nullptr;
            // r1 = surface_divergence!(-kappa [T]) (heatconduction.jl:97-98), r2 = surface average
            k_heat_bc<<<(N + 255) / 256, 256, 0, st>>>(tp, tm, N, h->kappa, h->e.as<double>(), h->r2.as<double>());
            ILH_HIP(hipGetLastError());
            double* F = h->F.as<double>();
            scatter_op(pl, OP_DS, h->e.as<double>(), F);   // includes the 1/dx of GridScaling
            // a stage's W = F + R sigma differs from F only on R's cells, which every stage rewrites
            if (h->n_near > 0) {
                k_heat_copy_tiles<<<h->n_near, 256, 0, st>>>(F, h->near_list.as<int>(), pl->g.nx(GK_PRIMAL),
                                                            pl->g.ny(GK_PRIMAL), h->W1.as<double>(), h->W2.as<double>());
                ILH_HIP(hipGetLastError());
            }
            if (h->M23 <= YMB && h->n_near > 0) {
                // r2s = r2 - dt a21 E H13 F
                TilePass P;
                P.in = F;
                P.cin = -h->dt * A21;
                P.K = h->k13.as<double>();
                P.M = h->M13;
                P.out = h->Y.as<double>();
                tile_pass(pl, P, h->touch_list.as<int>(), h->n_touch);
                heat_gather(pl, P.out, nullptr, h->r2s.as<double>());
                axpby(st, h->r2s.as<double>(), h->r2.as<double>(), 1.0, 1.0, N);
            }
        } else {
            fill_zero(st, h->F.as<double>(), pl->g.n(GK_PRIMAL));
        }
        h->have_bc = true;
        io.done();
    });
}

extern "C" int ilh_heat_advance(ilh_heat* h, double* T, int nsteps, int mem)
{
    return guarded_call([&] {
        if (!h) fail(ILH_ERR_ARG, "null heat plan");
        if (nsteps < 0) fail(ILH_ERR_ARG, "negative step count");
        ilh_plan* pl = h->pl;
        if (pl->gen != h->gen) fail(ILH_ERR_STATE, "the plan's geometry changed since ilh_heat_create");
        if (!h->have_bc) fail(ILH_ERR_STATE, "ilh_heat_set_boundary must come first");
        Io io(pl, mem);
        const int N = pl->N;
        const size_t ng = pl->g.n(GK_PRIMAL);
        hipStream_t st = pl->ctx->stream;
        double* d_T = io.out(T, ng, pl->io_b);
        if (mem == ILH_MEM_HOST)
            ILH_HIP(hipMemcpyAsync(d_T, T, sizeof(double) * ng, hipMemcpyHostToDevice, st));
        const double dt = h->dt;
        double *F = h->F.as<double>(), *A = h->A.as<double>(), *Bt = h->Bt.as<double>(), *Y = h->Y.as<double>();
        double *W1 = h->W1.as<double>(), *W2 = h->W2.as<double>();
        double *e = h->e.as<double>(), *sg = h->sg.as<double>(), *r2 = h->r2.as<double>();
        const double* K13 = h->k13.as<double>();
        const double* K23 = h->k23.as<double>();
        // sigma = -(1/(dt c)) Sinv (E Yh - r);  W = base + cb R sigma on R's cells
        auto multiplier = [&](const double* Yh, const double* r, const StageInverse& S, double c, const double* base,
                              double cb, double* W) {
            heat_gather(pl, Yh, r, e);
            k_packed_matvec<<<(N + 3) / 4, 256, 0, st>>>(S.ptr.as<int>(), S.idx.as<int>(), S.val.as<double>(), e, sg, N,
                                                         -1.0 / (dt * c));
            const RowBins& b = scatter_bins(pl, OP_R_PRIMAL)[0];
            k_heat_cells<<<b.ny, 64, 0, st>>>(b.cell_ptr, b.cells, b.cai, b.cw, pl->g.nx(GK_PRIMAL), sg, base, cb, W);
            ILH_HIP(hipGetLastError());
        };
        TilePass P13, P23;
        P13.K = K13;
        P13.M = h->M13;
        P23.K = K23;
        P23.M = h->M23;
        P13.near = P23.near = h->near.as<unsigned char>();
        auto pass = [&](TilePass P, const double* in, double* out) {
            P.in = in;
            P.out = out;
            return P;
        };
        const bool tiles = h->M23 <= YMB;
        for (int n = 0; n < nsteps; ++n) {
            if (N == 0) {
                // no bodies (F = 0): T <- H23 H13 T
                if (tiles) {
                    tile_pass(pl, pass(P13, d_T, A));
                    tile_pass(pl, pass(P23, A, d_T));
                } else {
                    heat_apply(pl, K13, h->M13, d_T, 0.0, nullptr, Bt, A);
                    heat_apply(pl, K23, h->M23, A, 0.0, nullptr, Bt, d_T);
                }
                continue;
            }
            if (tiles) {
                tile_pass(pl, pass(P13, d_T, A));                              // G (in A)
                multiplier(A, h->r2s.as<double>(), h->S13, A21, F, 1.0, W1);
                TilePass P = pass(P13, W1, Bt);
                P.cin = dt * A31;
                P.g = A;
                P.add = F;
                P.cadd = dt * A32;
                tile_pass(pl, P, h->near_list.as<int>(), h->n_near);             // A (in Bt)
                tile_pass(pl, pass(P23, Bt, Y), h->touch_list.as<int>(), h->n_touch);
                multiplier(Y, r2, h->S23, A32, F, 1.0, W2);
                P = pass(P23, A, d_T);
                P.b = W2;
                P.cb = dt * B2;
                P.add = F;
                P.cadd = dt * B3;
                tile_pass(pl, P);
            } else {
                // stage 2: Yhat2 = H13 (T + dt a21 F)
                heat_apply(pl, K13, h->M13, d_T, dt * A21, F, Bt, Y);
                multiplier(Y, r2, h->S13, A21, F, 1.0, W1);
                // stage 3: Yhat3 = H23 [H13 (T + dt a31 W1) + dt a32 F]
                heat_apply(pl, K13, h->M13, d_T, dt * A31, W1, Bt, A, dt * A32, F);
                heat_apply(pl, K23, h->M23, A, 0.0, nullptr, Bt, Y);
                multiplier(Y, r2, h->S23, A32, F, 1.0, W2);
                // final: yhat = H23 [H13 T + dt b2 W2] + dt b3 F
                heat_apply(pl, K13, h->M13, d_T, 0.0, nullptr, Bt, A, dt * B2, W2);
                heat_apply(pl, K23, h->M23, A, 0.0, nullptr, Bt, d_T, dt * B3, F);
            }
            multiplier(d_T, r2, h->S0, B3, d_T, dt * B3, d_T);                 // T = yhat + dt b3 R sigma3
        }
        io.back(T, d_T, ng);
        io.done();
    });
}

extern "C" int ilh_heat_destroy(ilh_heat* h)
{
    return guarded_call([&] {
        if (!h) return;
        ilh_plan* pl = h->pl;
        (void)hipSetDevice(pl->ctx->device);
        (void)hipStreamSynchronize(pl->ctx->stream);
        delete h;
        plan_release(pl);
    });
}
