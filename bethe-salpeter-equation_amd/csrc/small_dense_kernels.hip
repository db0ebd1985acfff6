// Small dense FP64 linear algebra for the Rayleigh-Ritz refinement (K8):
// everything lives in one workgroup's LDS (n <= 64).
//
// * Hermitian eigensolver: cyclic Jacobi in the round-robin order (n/2 disjoint
//   rotations per step, n-1 steps per sweep), each rotation the complex 2x2
//   Jacobi rotation of Golub & Van Loan sec. 8.5, applied as a block J^H A J.
// * Rayleigh-Ritz with SVQB basis stabilisation (Stathopoulos & Wu 2002): for
//   a basis S (not orthonormal) with G = S^H S and Hs = S^H H S, eig G =
//   U diag(s) U^H, P = U diag(s^-1/2) (dropping s < tol s_max), eig of
//   P^H Hs P = Y diag(l) Y^H, coefficients C = P Y of the lowest k Ritz pairs.
#include "jacobi.hpp"

#define SD_MAX 40

// Jacobi on the LDS matrix A (ld SD_LD), eigenvectors into V.  n <= SD_MAX; rows and
// columns from n up to the next even number are set to zero (such a pair does
// not rotate).  On exit the diagonal of A holds the eigenvalues (unsorted).
// A step rotates n/2 disjoint pairs: thread (P, Q) of the first waves forms
// both pairs' rotations itself, reads the 2 x 2 block of A in the rows of pair
// P and columns of pair Q and writes J_P^H B J_Q into the other copy of A, so a
// step takes one barrier.  The other waves rotate V by the rotations of the
// step before, which the threads (P, P) left in LDS: they form none themselves,
// and the first waves have one SIMD each to themselves but for their few
// products.  Bound by the latency of a step (LDS reads, two reciprocal square
// roots, LDS writes, a barrier).  The Rayleigh-Ritz of order 32 took 1.29 ms
// with two barriers, square roots and divisions per step and one task per
// (pair, row), 0.76 ms with V's threads forming their rotations too, 0.53 ms now.
#define SD_LD (SD_MAX + 1)
#define SD_PAIRS (SD_MAX / 2)
#define SD_JACOBI_THREADS 1024
static_assert(SD_PAIRS * SD_PAIRS + 63 < SD_JACOBI_THREADS, "threads left for V");
__device__ void sd_jacobi(int n, double2 (*A)[SD_LD], double2 (*V)[SD_LD])
{
    __shared__ double2 A2[SD_MAX][SD_LD];
    __shared__ JacobiRot rot[2][SD_PAIRS];
    __shared__ double sh[32];
    const int tid = threadIdx.x, nt = blockDim.x;
    const int m = (n + 1) & ~1, h = m / 2;
    for (int e = tid; e < SD_MAX * SD_MAX; e += nt) {
        const int i = e / SD_MAX, j = e % SD_MAX;
        V[i][j] = cmk(i == j ? 1.0 : 0.0, 0.0);
        if ((i >= n || j >= n) && i < m && j < m) A[i][j] = cmk(0, 0);
    }
    __syncthreads();
    double fro = 0.0;
    for (int e = tid; e < n * n; e += nt) fro += cabs2(A[e / n][e % n]);
    fro = block_sum(fro, sh);
    // pair j of step r: {m - 1, r} (j = 0) or {(r + j), (r - j)} mod (m - 1)
    auto pair = [m](int j, int r, int& p, int& q) {
        int u = (j == 0) ? m - 1 : r + j, v = r - j;
        if (j > 0 && u >= m - 1) u -= m - 1;
        if (v < 0) v += m - 1;
        p = min(u, v);
        q = max(u, v);
    };
    const int va = (h * h + 63) & ~63;               // first thread of V's waves
    const bool act = tid < h * h;
    int last = -1, cur = 0;                          // step whose rotations V still waits for
    auto rotate_v = [&](int r, const JacobiRot* js) {
        for (int t = tid - va; t < h * n; t += nt - va) {
            int p, q;
            const int j = t / n, i = t % n;
            pair(j, r, p, q);
            const JacobiRot rt = js[j];
            const double2 v0 = V[i][p], v1 = V[i][q];
            V[i][p] = csub(cscale(v0, rt.c), cmulc(rt.s, v1));
            V[i][q] = cadd(cmul(rt.s, v0), cscale(v1, rt.c));
        }
    };
    const int P = act ? tid / h : 0, Q = act ? tid % h : 0;
    double2 (*X)[SD_LD] = A;
    double2 (*Y)[SD_LD] = A2;
    for (int sweep = 0; sweep < 30; ++sweep) {
        double off = 0.0;
        for (int e = tid; e < n * n; e += nt) {
            const int r = e / n, j = e % n;
            if (r != j) off += cabs2(X[r][j]);
        }
        off = block_sum(off, sh);
        if (off <= 1e-30 * fro) break;
        for (int r = 0; r < m - 1; ++r) {
            if (act) {
                int p1, q1, p2, q2;
                pair(P, r, p1, q1);
                pair(Q, r, p2, q2);
                const JacobiRot rp = jacobi_rot(X[p1][p1].x, X[q1][q1].x, X[p1][q1]);
                const JacobiRot rq = jacobi_rot(X[p2][p2].x, X[q2][q2].x, X[p2][q2]);
                const double2 a00 = X[p1][p2], a01 = X[p1][q2], a10 = X[q1][p2], a11 = X[q1][q2];
                const double2 b00 = csub(cscale(a00, rq.c), cmulc(rq.s, a01)), b01 = cadd(cmul(rq.s, a00), cscale(a01, rq.c));
                const double2 b10 = csub(cscale(a10, rq.c), cmulc(rq.s, a11)), b11 = cadd(cmul(rq.s, a10), cscale(a11, rq.c));
                double2 c00 = csub(cscale(b00, rp.c), cmul(rp.s, b10)), c01 = csub(cscale(b01, rp.c), cmul(rp.s, b11));
                double2 c10 = cadd(cmulc(rp.s, b00), cscale(b10, rp.c)), c11 = cadd(cmulc(rp.s, b01), cscale(b11, rp.c));
                if (P == Q) {
                    rot[cur][P] = rp;
                    c00 = cmk(a00.x - rp.dl, 0.0);
                    c11 = cmk(a11.x + rp.dl, 0.0);
                    c01 = c10 = cmk(0, 0);
                }
                Y[p1][p2] = c00;
                Y[p1][q2] = c01;
                Y[q1][p2] = c10;
                Y[q1][q2] = c11;
            }
            if (tid >= va && last >= 0) rotate_v(last, rot[cur ^ 1]);
            last = r;
            cur ^= 1;
            __syncthreads();
            double2 (*t)[SD_LD] = X;
            X = Y;
            Y = t;
        }
    }
    if (tid >= va && last >= 0) rotate_v(last, rot[cur ^ 1]);
    __syncthreads();
    if (X != A) {
        for (int e = tid; e < n * n; e += nt) A[e / n][e % n] = X[e / n][e % n];
        __syncthreads();
    }
}

// Sort the Jacobi result ascending: writes eigenvalues to w[0..n) and the
// permutation to perm[0..n) (shared).
__device__ void sd_sort(int n, double2 (*A)[SD_LD], double* w, int* perm)
{
    __shared__ double tmp[SD_MAX];
    if (threadIdx.x == 0) {
        for (int i = 0; i < n; ++i) { perm[i] = i; w[i] = A[i][i].x; }
        for (int i = 1; i < n; ++i) {
            const int pi = perm[i];
            const double x = w[pi];
            int j = i - 1;
            while (j >= 0 && w[perm[j]] > x) { perm[j + 1] = perm[j]; --j; }
            perm[j + 1] = pi;
        }
        for (int i = 0; i < n; ++i) tmp[i] = w[perm[i]];
        for (int i = 0; i < n; ++i) w[i] = tmp[i];
    }
    __syncthreads();
}

// Rayleigh-Ritz with SVQB: inputs G, Hs (m x m, ld m, device), outputs the
// lowest k Ritz values (evals) and the m x k coefficient matrix C (ld m).
// Returns the rank kept in info[0].
__global__ __launch_bounds__(SD_JACOBI_THREADS) void k_small_rr(int m, int k, const double2* __restrict__ G,
                                                 const double2* __restrict__ Hs, double tol,
                                                 double* __restrict__ evals,
                                                 double2* __restrict__ C, int* __restrict__ info)
{
    __shared__ double2 A[SD_MAX][SD_LD];
    __shared__ double2 V[SD_MAX][SD_LD];
    __shared__ double2 P[SD_MAX][SD_LD];
    __shared__ double w[SD_MAX];
    __shared__ int perm[SD_MAX];
    __shared__ int rank;
    const int tid = threadIdx.x, nt = blockDim.x;
    // 1. eig of G
    for (int e = tid; e < m * m; e += nt) A[e % m][e / m] = G[e];
    __syncthreads();
    sd_jacobi(m, A, V);
    sd_sort(m, A, w, perm);
    // 2. P = U diag(s^-1/2) over the kept (largest) eigenvalues, in descending order
    if (tid == 0) {
        const double smax = w[m - 1];
        int r = 0;
        for (int i = m - 1; i >= 0; --i)
            if (w[i] > tol * smax) ++r;
        rank = r;
    }
    __syncthreads();
    const int r = rank;
    for (int e = tid; e < m * r; e += nt) {
        const int i = e % m, j = e / m;            // column j of P <- eigenvector perm[m-1-j]
        const int src = perm[m - 1 - j];
        P[i][j] = cscale(V[i][src], 1.0 / sqrt(w[m - 1 - j]));
    }
    __syncthreads();
    // 3. Hr = P^H Hs P  (r x r) into A
    for (int e = tid; e < m * r; e += nt) {          // V <- Hs P  (m x r)
        const int i = e % m, j = e / m;
        double2 s = cmk(0, 0);
        for (int l = 0; l < m; ++l) cfma(s, Hs[i + l * m], P[l][j]);
        V[i][j] = s;
    }
    __syncthreads();
    for (int e = tid; e < r * r; e += nt) {
        const int i = e % r, j = e / r;
        double2 s = cmk(0, 0);
        for (int l = 0; l < m; ++l) cfmac(s, P[l][i], V[l][j]);
        A[i][j] = s;
    }
    __syncthreads();
    for (int e = tid; e < r * r; e += nt) {         // exact Hermitian symmetrisation
        const int i = e % r, j = e / r;
        if (i < j) {
            const double2 a = A[i][j], b = A[j][i];
            const double2 h = cmk(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
            A[i][j] = h;
            A[j][i] = cconj(h);
        } else if (i == j) {
            A[i][i].y = 0.0;
        }
    }
    __syncthreads();
    // 4. eig of Hr, lowest k
    sd_jacobi(r, A, V);
    sd_sort(r, A, w, perm);
    const int kk = k < r ? k : r;
    for (int e = tid; e < m * kk; e += nt) {         // C = P Y(:, lowest)
        const int i = e % m, j = e / m;
        const int src = perm[j];
        double2 s = cmk(0, 0);
        for (int l = 0; l < r; ++l) cfma(s, P[i][l], V[l][src]);
        C[i + j * m] = s;
    }
    for (int j = tid; j < kk; j += nt) evals[j] = w[j];
    if (tid == 0) info[0] = r;
}

extern "C" hipError_t bse_launch_small_rr(hipStream_t st, int m, int k, const double2* G,
                                          const double2* Hs, double tol, double* evals,
                                          double2* C, int* info)
{
    if (m > SD_MAX || k > m) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_small_rr, dim3(1), dim3(SD_JACOBI_THREADS), 0, st, m, k, G, Hs, tol, evals, C, info);
    return hipGetLastError();
}

// R = Y - X diag(lam) with lam_j = Re(x_j^H y_j) / (x_j^H x_j), then scale each
// residual column to unit norm (columns with zero residual stay zero).  One
// workgroup per column.  rnorm_j = ||y_j - lam_j x_j|| / ||x_j||; rq (may be
// null) receives lam_j.
__global__ __launch_bounds__(256) void k_residual(int64_t N, const double2* __restrict__ X,
                                                 const double2* __restrict__ Y, int64_t ld,
                                                 double2* __restrict__ R, double* __restrict__ rnorm,
                                                 double* __restrict__ rq)
{
    __shared__ double sh[32];
    const int j = blockIdx.x;
    const double2* x = X + (int64_t)j * ld;
    const double2* y = Y + (int64_t)j * ld;
    double2* r = R + (int64_t)j * ld;
    double xy = 0.0, xx = 0.0;
    for (int64_t i = threadIdx.x; i < N; i += blockDim.x) {
        xy += x[i].x * y[i].x + x[i].y * y[i].y;
        xx += cabs2(x[i]);
    }
    xy = block_sum(xy, sh);
    xx = block_sum(xx, sh);
    const double lam = xy / xx;
    double rr = 0.0;
    for (int64_t i = threadIdx.x; i < N; i += blockDim.x) {
        const double2 v = csub(y[i], cscale(x[i], lam));
        r[i] = v;
        rr += cabs2(v);
    }
    rr = block_sum(rr, sh);
    const double inv = (rr > 0.0) ? 1.0 / sqrt(rr) : 0.0;
    for (int64_t i = threadIdx.x; i < N; i += blockDim.x) r[i] = cscale(r[i], inv);
    if (threadIdx.x == 0) {
        rnorm[j] = sqrt(rr / xx);
        if (rq) rq[j] = lam;
    }
}

extern "C" hipError_t bse_launch_residual(hipStream_t st, int64_t N, int k, const double2* X,
                                          const double2* Y, int64_t ld, double2* R, double* rnorm,
                                          double* rq)
{
    hipLaunchKernelGGL(k_residual, dim3(k), dim3(256), 0, st, N, X, Y, ld, R, rnorm, rq);
    return hipGetLastError();
}

// out[j] = Re(x_j^H y_j) for k columns (one workgroup per column).
__global__ __launch_bounds__(256) void k_coldot(int64_t N, const double2* __restrict__ X,
                                               const double2* __restrict__ Y, int64_t ld,
                                               double* __restrict__ out)
{
    __shared__ double sh[32];
    const int j = blockIdx.x;
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < N; i += blockDim.x) {
        const double2 a = X[i + (int64_t)j * ld], b = Y[i + (int64_t)j * ld];
        s += a.x * b.x + a.y * b.y;
    }
    s = block_sum(s, sh);
    if (threadIdx.x == 0) out[j] = s;
}

extern "C" hipError_t bse_launch_coldot(hipStream_t st, int64_t N, int k, const double2* X,
                                        const double2* Y, int64_t ld, double* out)
{
    hipLaunchKernelGGL(k_coldot, dim3(k), dim3(256), 0, st, N, X, Y, ld, out);
    return hipGetLastError();
}
