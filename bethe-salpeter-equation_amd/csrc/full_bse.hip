// K12: the full BSE beyond the Tamm-Dancoff approximation (add_coupling_part,
// bse.version13.cpp:2929-3040; eig_gen at 3326), solved by a
// structure-preserving reduction to a Hermitian eigenproblem instead of the
// reference's general (non-Hermitian) eigensolver:
//
//   H = [[A, B], [-conj B, -conj A]] = s3 M,   M = [[A, B], [conj B, conj A]],
//   s3 = diag(1, ..., 1, -1, ..., -1).
//
// For a stable system M is Hermitian positive definite; with M = L L^H
// (Cholesky), W = L^H s3 L is Hermitian and similar to H, so the eigenvalues
// of H (pairs +-E) are those of W, and an eigenvector y of W gives
// x = sqrt(E) L^-H y with x^H s3 x = 1 (Shao, da Jornada, Yang, Deslippe &
// Lin 2016, the method the reference's draft cites at 3371).  The oscillator
// strength of x is rho~^H x = sqrt(E) (L^-1 rho~)^H y, so every exciton's
// strength comes out of the Hermitian pipeline's contraction with
// z = L^-1 rho~, without forming the vectors.
//
// Storage: M (then L), W: tiled lower FP64 storage of order n2 = 2N (the
// layout of the TDA matrix), both halves in the k-major internal order.
// Kernels here: compose M from A and B, the blocked Cholesky (diagonal tile
// factor and inverse on registers, panel and trailing update tile by tile),
// W = L^H s3 L, and the two triangular solves.
#include "mma64.hpp"
#include <algorithm>

// ---------------------------------------------------------------------------
// M from the TDA block A and the coupling block B (both tiled lower FP64 of
// order N; B complex symmetric, its lower triangle stored).  One workgroup per
// lower tile of M; padding rows and columns and the strict upper half of
// diagonal tiles are written as zeros.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_compose_full(int64_t N, const double2* __restrict__ A,
                                                      const double2* __restrict__ Bm, double2* __restrict__ M)
{
    const int64_t n2 = 2 * N;
    const int nt2 = tile_count(n2), ntA = tile_count(N);
    int ti, tj;
    tri_tile(blockIdx.x, ti, tj);
    double2* t = M + tile_pos(ti, tj, nt2) * (BSE_TILE * BSE_TILE);
    for (int e = threadIdx.x; e < BSE_TILE * BSE_TILE; e += blockDim.x) {
        const int64_t r = (int64_t)ti * 64 + (e & 63), c = (int64_t)tj * 64 + (e >> 6);
        double2 x = cmk(0, 0);
        if (r < n2 && c < n2 && r >= c) {
            if (r < N) {
                x = A[tix(r, c, ntA)];
            } else if (c < N) {
                const int64_t rr = r - N;
                x = cconj(rr >= c ? Bm[tix(rr, c, ntA)] : Bm[tix(c, rr, ntA)]);
            } else {
                x = cconj(A[tix(r - N, c - N, ntA)]);
            }
            if (r == c) x.y = 0.0;
        }
        t[e] = x;
    }
}

// ---------------------------------------------------------------------------
// Cholesky step J, part 1: factor the diagonal tile (J, J) and invert the
// factor.  L_JJ goes back to the tile (zeros above the diagonal), its inverse
// to Linv[J] (64 x 64, column-major).  Padding rows beyond n2 get a unit pivot
// so that the factor of the last tile stays regular; they are written back as
// zeros.  A pivot <= 0 means M is not positive definite: err[0] receives the
// (1-based) row.
//
// One workgroup is all there is, so the bound is the chain of 64 steps.  The
// tile lives in registers (thread: row i = lane, 8 columns of its wave) and
// step j is one rank-one elimination of the rows below j, of the matrix on
// the columns beyond j and of the inverse of the unit factor on the columns
// before it; the pivot column passes through LDS, one barrier a step (the
// columns, published unscaled, stay as L D^1/2), the inverse's part of the
// pivot row is lane j of every wave.  200 us with three barriers a step on an LDS tile and a serial
// substitution per column for the inverse, 65 us this way.
// ---------------------------------------------------------------------------
__device__ inline double lane_value(double x, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}

__global__ __launch_bounds__(512) void k_potrf_tile(int n2, int J, double2* __restrict__ M,
                                                    double2* __restrict__ Linv, int* __restrict__ err)
{
    __shared__ double2 sL[64][65];      // sL[c][r]: column c as published
    __shared__ double rs[64];
    const int nt2 = tile_count(n2);
    double2* t = M + tile_pos(J, J, nt2) * (BSE_TILE * BSE_TILE);
    const int i = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int r0 = J * 64;
    for (int e = threadIdx.x; e < 64 * 64; e += 512) sL[e >> 6][e & 63] = t[e];
    __syncthreads();
    double2 a[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int c = 8 * g + q;
        const double2 lo = sL[c][i], up = sL[i][c];
        a[q] = csel(i >= c, lo, cconj(up));
        const bool unit = i == c && r0 + i >= n2;
        a[q] = csel(unit, cmk(1.0, 0.0), a[q]);
    }
    __syncthreads();
    int bad = 0;
    // the outer loop is not unrolled: straight-line code runs once and would
    // wait for the instruction cache at every line
#pragma unroll 1
    for (int jb = 0; jb < 8; ++jb) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int j = 8 * jb + u;
            if (g == jb) sL[j][i] = a[u];
            // row j: the inverse's entries before the pivot; beyond it the
            // column's conjugate (from the upper triangle, with the real part as
            // the pivot, its rounding differences from the lower one would grow
            // fourfold a step)
            double2 pr[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) pr[q] = cmk(lane_value(a[q].x, j), lane_value(a[q].y, j));
            __syncthreads();
            double d = sL[j][j].x;
            const double2 col = sL[j][i];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const double2 x = sL[j][8 * g + q];
                pr[q] = csel(8 * g + q > j, cconj(x), pr[q]);
            }
            if (!(d > 0.0)) {
                if (!bad) bad = r0 + j + 1;
                d = 1.0;
            }
            // (1 / d of a subnormal pivot would overflow: both sides scaled up)
            const double us = d < 1e-290 ? 0x1p600 : 1.0;
            const double2 m = cscale(cscale(col, us), rcp_nr(d * us));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int c = 8 * g + q;
                const double2 z = csel(c == j, cmk(-m.x, -m.y), csub(a[q], cmul(m, pr[q])));
                a[q] = csel(i > j, z, csel(i == j && c == j, cmk(1.0, 0.0), a[q]));
            }
        }
    }
    if (threadIdx.x < 64) {
        const double d = sL[i][i].x;
        rs[i] = d > 0.0 ? 1.0 / sqrt(d) : 1.0;
    }
    __syncthreads();
    double2* li = Linv + (int64_t)J * 64 * 64;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int c = 8 * g + q;
        const bool in = i >= c && r0 + i < n2;
        const double2 l = i == c ? cmk(1.0 / rs[c], 0.0) : cscale(sL[c][i], rs[c]);
        t[i + 64 * c] = csel(in, l, cmk(0, 0));
        li[i + 64 * c] = csel(in, cscale(a[q], rs[i]), cmk(0, 0));
    }
    if (threadIdx.x == 0 && bad && err[0] == 0) err[0] = bad;
}

// ---------------------------------------------------------------------------
// Cholesky step J, part 2: the panel below the diagonal tile, L_IJ = A_IJ
// L_JJ^-H for I > J (trail = 0: one workgroup per tile), then the trailing
// update A_IK -= L_IJ L_KJ^H for J < K <= I (trail = 1: one workgroup per lower
// tile).  Both are X(r, c) = sum_k A(r, k) conj(B(c, k)) over the 64 columns of
// two tiles, on matrix cores with the operands straight from L2 (a wave forms
// the transpose of its 32 x 32 part: 16 lanes hold 16 consecutive rows).
// 2592 rows: 60 us a panel on the vector units and two rank-64 launches of
// 35 us each on a copy of the panel before, two launches of 17 us on average now.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_chol_tiles(int n2, int J, int trail, double2* __restrict__ M,
                                                    const double2* __restrict__ Linv)
{
    const int nt2 = tile_count(n2);
    int I = J + 1 + (int)blockIdx.x, K = J;
    if (trail) {
        tri_tile(blockIdx.x, I, K);
        I += J + 1;
        K += J + 1;
    }
    constexpr int64_t TE = BSE_TILE * BSE_TILE;
    const double2* A = M + tile_pos(I, J, nt2) * TE;
    const double2* B = trail ? M + tile_pos(K, J, nt2) * TE : Linv + (int64_t)J * TE;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int c0 = 32 * (w & 1), r0 = 32 * (w >> 1);
    btg_d4 cr[2][2], ci[2][2];
    btg_zero<2, 2>(cr, ci);
    double2 a[BTG_KB][2], b[BTG_KB][2];
    // K step s + u: column 4 (s + u) + lq of both tiles
    auto load = [&](int s, double2 (&x)[BTG_KB][2], double2 (&y)[BTG_KB][2]) {
#pragma unroll
        for (int u = 0; u < BTG_KB; ++u) {
            const int k = 4 * (s + u) + lq;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                x[u][q] = cconj(B[c0 + 16 * q + li + 64 * k]);
                y[u][q] = A[r0 + 16 * q + li + 64 * k];
            }
        }
    };
    load(0, a, b);
#pragma unroll
    for (int s = 0; s < 16; s += BTG_KB) {
        double2 an[BTG_KB][2], bn[BTG_KB][2];
        if (s + BTG_KB < 16) load(s + BTG_KB, an, bn);
#pragma unroll
        for (int u = 0; u < BTG_KB; ++u) btg_cmma<2, 2>(cr, ci, a[u], b[u]);
        if (s + BTG_KB < 16) {
#pragma unroll
            for (int u = 0; u < BTG_KB; ++u)
#pragma unroll
                for (int q = 0; q < 2; ++q) { a[u][q] = an[u][q]; b[u][q] = bn[u][q]; }
        }
    }
    __syncthreads();                      // trail = 0 replaces what the other waves read
    double2* t = M + tile_pos(I, K, nt2) * TE;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
        for (int tj = 0; tj < 2; ++tj)
#pragma unroll
            for (int reg = 0; reg < 4; ++reg) {
                double2* x = t + (r0 + 16 * tj + li) + 64 * (c0 + 16 * ti + mfma16_row_f64(lane, reg));
                const double2 p = cmk(cr[ti][tj][reg], ci[ti][tj][reg]);
                *x = trail ? csub(*x, p) : p;
            }
}

// ---------------------------------------------------------------------------
// W = L^H s3 L, lower tiles: W_IJ = sum_{K >= I} L_KI^H diag(s_K) L_KJ with
// s = +1 on rows < N, -1 on rows N .. n2 - 1 (padding rows of L are zero).
// One workgroup per tile of W on matrix cores, as above (the wave forms the
// conjugate transpose of its part); the rows from N on are summed first and
// the sums negated.  2592 rows: 925 us on the vector units from LDS, 815
// us this way.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_lsl(int64_t N, const double2* __restrict__ L, double2* __restrict__ Wt)
{
    const int64_t n2 = 2 * N;
    const int nt2 = tile_count(n2);
    int ti, tj;
    tri_tile(blockIdx.x, ti, tj);
    constexpr int64_t TE = BSE_TILE * BSE_TILE;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int c0 = 32 * (w & 1), r0 = 32 * (w >> 1);
    btg_d4 cr[2][2], ci[2][2];
    btg_zero<2, 2>(cr, ci);
    const bool on[2] = {true, true};
    auto tiles = [&](int K, int rlo, int rhi) {
        const double2* pa[2];
        const double2* pb[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            pa[q] = L + tile_pos(K, tj, nt2) * TE + 64 * (c0 + 16 * q + li);
            pb[q] = L + tile_pos(K, ti, nt2) * TE + 64 * (r0 + 16 * q + li);
        }
        btg_rows(cr, ci, pa, on, pb, on, rlo, rhi, lq);
    };
    const int KN = (int)(N >> 6), rN = (int)(N & 63);   // first row with s = -1
    for (int K = nt2 - 1; K >= max(ti, KN); --K) tiles(K, K == KN ? rN : 0, 64);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            cr[a][b] = -cr[a][b];
            ci[a][b] = -ci[a][b];
        }
    for (int K = ti; K <= min(KN, nt2 - 1); ++K) tiles(K, 0, K == KN ? rN : 64);
    double2* wt = Wt + tile_pos(ti, tj, nt2) * TE;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int reg = 0; reg < 4; ++reg) {
                const int lc = c0 + 16 * a + mfma16_row_f64(lane, reg), lr = r0 + 16 * b + li;
                const int64_t gr = (int64_t)ti * 64 + lr, gc = (int64_t)tj * 64 + lc;
                double2 x = cmk(cr[a][b][reg], -ci[a][b][reg]);
                if (gr >= n2 || gc >= n2 || gr < gc) x = cmk(0, 0);
                if (gr == gc) x.y = 0.0;
                wt[lr + lc * 64] = x;
            }
}

// ---------------------------------------------------------------------------
// z = L^-1 b, forward substitution by tile rows: launch J forms z_J = Linv_JJ b_J
// (every workgroup for itself; the first one stores it) and workgroup I takes
// L_IJ z_J from b_I, I > J.  b is overwritten.  2592 rows: 1390 us with one
// workgroup walking all of L, 180 us this way.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_lower_step(int n2, int J, const double2* __restrict__ L,
                                                    const double2* __restrict__ Linv, double2* __restrict__ b,
                                                    double2* __restrict__ z)
{
    __shared__ double2 part[4][64];
    __shared__ double2 zv[64];
    const int nt2 = tile_count(n2), I = J + (int)blockIdx.x;
    const int r = threadIdx.x & 63, q = threadIdx.x >> 6;
    // 64 x 64 product: quarter q takes 16 columns
    auto product = [&](const double2* t, const double2* x) {
        double2 a[16], s = cmk(0, 0);
#pragma unroll
        for (int c = 0; c < 16; ++c) a[c] = t[r + 64 * (16 * q + c)];
#pragma unroll
        for (int c = 0; c < 16; ++c) cfma(s, a[c], x[16 * q + c]);
        part[q][r] = s;
        __syncthreads();
        return cadd(cadd(part[0][r], part[1][r]), cadd(part[2][r], part[3][r]));
    };
    const double2 x = product(Linv + (int64_t)J * 64 * 64, b + (int64_t)J * 64);
    if (q == 0) {
        zv[r] = x;
        if (I == J) z[(int64_t)J * 64 + r] = x;
    }
    __syncthreads();
    if (I == J) return;
    const double2 y = product(L + tile_pos(I, J, nt2) * (BSE_TILE * BSE_TILE), zv);
    if (q == 0) b[(int64_t)I * 64 + r] = csub(b[(int64_t)I * 64 + r], y);
}

// ---------------------------------------------------------------------------
// X = scale_v * L^-H Y for nv vectors: X starts as the scaled Y (rows beyond n2
// zero), then tile rows J from the bottom, x_J <- Linv_JJ^H x_J and, for every
// I < J, x_I -= L_JI^H x_J.  Both are products over the 64 rows of tile row J
// on matrix cores, one workgroup per 64 x 64 block of the result, operands
// straight from L2 (each wave forms the transposed conjugate of its 32 x 32
// part, so that 16 lanes hold 16 consecutive rows of X).  2592 rows and 1296
// vectors: 12 ms with one workgroup per vector reading all of L, 2.2 ms
// this way, where the 81 dependent launches are the bound; more vectors or rows
// fill them.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_upper_init(int n2, int nv, const double2* __restrict__ Y, int64_t ldy,
                                                    double2* __restrict__ X, int64_t ldx,
                                                    const double* __restrict__ scale)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= (int64_t)tile_count(n2) * 64) return;
    for (int v = blockIdx.y; v < nv; v += gridDim.y)
        X[r + v * ldx] = r < n2 ? cscale(Y[r + v * ldy], scale ? scale[v] : 1.0) : cmk(0, 0);
}

// upd = 1: tile row I = blockIdx.y of X loses L_JI^H x_J; upd = 0: x_J is
// replaced by Linv_JJ^H x_J.
__global__ __launch_bounds__(256) void k_upper_step(int n2, int nv, int J, int upd, const double2* __restrict__ L,
                                                    const double2* __restrict__ Linv, double2* __restrict__ X,
                                                    int64_t ldx)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int c0 = blockIdx.x * 64 + 32 * (w & 1), r0 = 32 * (w >> 1);
    const int I = upd ? (int)blockIdx.y : J;
    const double2* t = upd ? L + tile_pos(J, I, tile_count(n2)) * (BSE_TILE * BSE_TILE)
                           : Linv + (int64_t)J * 64 * 64;
    const double2* pa[2];
    const double2* pb[2];
    bool va[2], vb[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int c = c0 + 16 * q + li;
        va[q] = c < nv;
        vb[q] = true;
        pa[q] = X + (int64_t)J * 64 + (int64_t)min(c, nv - 1) * ldx;
        pb[q] = t + (int64_t)(r0 + 16 * q + li) * 64;
    }
    btg_d4 cr[2][2], ci[2][2];
    btg_zero<2, 2>(cr, ci);
    btg_rows(cr, ci, pa, va, pb, vb, 0, 64, lq);
    __syncthreads();                      // upd = 0 replaces what the other waves read
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
        for (int tj = 0; tj < 2; ++tj)
#pragma unroll
            for (int reg = 0; reg < 4; ++reg) {
                const int c = c0 + 16 * ti + mfma16_row_f64(lane, reg), r = r0 + 16 * tj + li;
                if (c >= nv) continue;
                double2* x = X + (int64_t)I * 64 + r + (int64_t)c * ldx;
                const double2 p = cmk(cr[ti][tj][reg], -ci[ti][tj][reg]);
                *x = upd ? csub(*x, p) : p;
            }
}

// rho~ = (rho; -conj(rho)) in the internal order of both halves, zero-padded
// to ntot entries (the anti-resonant pair densities rho_vc = -conj(rho_cv) of
// the point-orbital dipole limit).
__global__ __launch_bounds__(256) void k_full_rho(int64_t N, const double2* __restrict__ rho,
                                                  double2* __restrict__ out, int64_t ntot)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= ntot) return;
    double2 x = cmk(0, 0);
    if (i < N) x = rho[i];
    else if (i < 2 * N) x = cscale(cconj(rho[i - N]), -1.0);
    out[i] = x;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
extern "C" hipError_t bse_launch_full_rho(hipStream_t st, int64_t N, const double2* rho, double2* out,
                                          int64_t ntot)
{
    hipLaunchKernelGGL(k_full_rho, dim3((unsigned)ceil_div64(ntot, 256)), dim3(256), 0, st, N, rho, out, ntot);
    return hipGetLastError();
}

extern "C" hipError_t bse_launch_compose_full(hipStream_t st, int64_t N, const double2* A, const double2* Bm,
                                              double2* M)
{
    const int64_t nt2 = tile_count(2 * N);
    hipLaunchKernelGGL(k_compose_full, dim3((unsigned)(nt2 * (nt2 + 1) / 2)), dim3(256), 0, st, N, A, Bm, M);
    return hipGetLastError();
}

extern "C" hipError_t bse_launch_potrf_tile(hipStream_t st, int n2, int J, double2* M, double2* Linv, int* err)
{
    hipLaunchKernelGGL(k_potrf_tile, dim3(1), dim3(512), 0, st, n2, J, M, Linv, err);
    return hipGetLastError();
}

// Panel J of the factor and the trailing update behind it.
extern "C" hipError_t bse_launch_chol_panel(hipStream_t st, int n2, int J, double2* M, const double2* Linv)
{
    const int64_t r = tile_count(n2) - J - 1;
    if (r <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_chol_tiles, dim3((unsigned)r), dim3(256), 0, st, n2, J, 0, M, Linv);
    hipLaunchKernelGGL(k_chol_tiles, dim3((unsigned)(r * (r + 1) / 2)), dim3(256), 0, st, n2, J, 1, M, Linv);
    return hipGetLastError();
}

extern "C" hipError_t bse_launch_lsl(hipStream_t st, int64_t N, const double2* L, double2* Wt)
{
    const int64_t nt2 = tile_count(2 * N);
    hipLaunchKernelGGL(k_lsl, dim3((unsigned)(nt2 * (nt2 + 1) / 2)), dim3(256), 0, st, N, L, Wt);
    return hipGetLastError();
}

// z = L^-1 b for whole tiles of rows; b is overwritten.
extern "C" hipError_t bse_launch_lower_solve(hipStream_t st, int n2, const double2* L, const double2* Linv,
                                             double2* b, double2* z)
{
    const int nt2 = tile_count(n2);
    for (int J = 0; J < nt2; ++J)
        hipLaunchKernelGGL(k_lower_step, dim3((unsigned)(nt2 - J)), dim3(256), 0, st, n2, J, L, Linv, b, z);
    return hipGetLastError();
}

extern "C" hipError_t bse_launch_upper_solve(hipStream_t st, int n2, int nv, const double2* L,
                                             const double2* Linv, const double2* Y, int64_t ldy, double2* X,
                                             int64_t ldx, const double* scale)
{
    if (nv <= 0) return hipSuccess;
    if (ldx < (int64_t)tile_count(n2) * 64) return hipErrorInvalidValue;
    const int nt2 = tile_count(n2);
    const unsigned cb = (unsigned)ceil_div64(nv, 64);
    hipLaunchKernelGGL(k_upper_init, dim3((unsigned)ceil_div64((int64_t)nt2 * 64, 256), (unsigned)std::min(nv, 4096)),
                       dim3(256), 0, st, n2, nv, Y, ldy, X, ldx, scale);
    for (int J = nt2 - 1; J >= 0; --J) {
        hipLaunchKernelGGL(k_upper_step, dim3(cb, 1), dim3(256), 0, st, n2, nv, J, 0, L, Linv, X, ldx);
        if (J > 0)
            hipLaunchKernelGGL(k_upper_step, dim3(cb, (unsigned)J), dim3(256), 0, st, n2, nv, J, 1, L, Linv, X, ldx);
    }
    return hipGetLastError();
}
