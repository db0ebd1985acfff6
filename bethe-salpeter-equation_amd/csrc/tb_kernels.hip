// K1 + K2: per-k tight-binding Hamiltonian and its FP64 Hermitian eigenpairs.
//
// Replaces Hamiltonian_TB::FFT (bse.version13.cpp:647-705) and
// pull_ks_states / pull_ks_states_subset (706-821): H_lm(k) = sum_R H_lm(R)
// e^{i k.R} (Cartesian R, no orbital centre in the phase), eigenpairs sorted
// ascending with unit columns, then the band window: valence slots v = 0..nv-1
// are bands n_occ-1-v at k - q (top down, 812-813), conduction slots are bands
// n_occ+c at k (bottom up, + scissor, 815-816).
//
// One matrix per (k, half): half 0 diagonalises H(k) for the conduction
// states, half 1 diagonalises H(k - q) for the valence states (a half without
// slots is not formed).  The eig is a complex Jacobi method in FP64
// (norb <= 16) in the round-robin order, whose rounds rotate disjoint pairs of
// rows and columns at once; it is accurate to working precision and has no
// branches that depend on LAPACK-style deflation.  Each eigenvector's
// largest-modulus component is made real and positive so outputs are
// deterministic (every downstream quantity is gauge invariant).
//
// Mapping: MP x MP lanes per matrix, MP = 1, 2, 4 or 8 >= norb / 2 (the order
// is padded with a zero row and column), 64 / MP^2 matrices per wave, A and V in
// LDS (12, 10, 9 and 8.5 KB per wave).  Lane (P, Q) applies a round's rotations to
// the 2 x 2 block of A in the rows of pair P and the columns of pair Q, and
// that of pair Q to rows P and P + MP of V.  A round is bound by its latency
// (LDS reads, two reciprocal square roots, LDS writes), so the lanes share
// one matrix rather than taking one each: 257 matrices of order 8 took
// 1.27 ms (of order 16: 11 ms) with one thread per matrix and its arrays in
// scratch memory, 0.047 ms (0.16 ms) now.
#include "jacobi.hpp"

#define TB_MAXORB BSE_MAXORB
#define TB_WAVES 4             // waves per workgroup
#define TB_SWEEPS 40

// Hand-over through LDS between the lanes of one wave.
__device__ inline void tb_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
}

template <int MP> struct TbShape {
    static constexpr int N = 2 * MP, L = MP * MP, G = 64 / L, LD = N + 1;
    static constexpr int EL = N * LD;                      // elements of one matrix in LDS
};

// Derivative mode: dhr != nullptr adds a first-order perturbation dH(k)
// (same Fourier form) and returns d eps and dc (parallel transport gauge).
template <int MP>
__global__ __launch_bounds__(64 * TB_WAVES) void k_tb_states(
    int nk, int norb, int nr, const double* __restrict__ rcart,
    const double2* __restrict__ hr, const double* __restrict__ kpts,
    double qx, double qy, double qz, int n_occ, int nv, int nc, double scissor,
    const double2* __restrict__ dhr,   // optional nr x norb x norb perturbation
    double* __restrict__ eps_out,      // nk x (nv+nc)
    double2* __restrict__ coef_out,    // nk x (nv+nc) x norb
    double* __restrict__ deps_out,     // optional nk x (nv+nc)
    double2* __restrict__ dcoef_out,   // optional nk x (nv+nc) x norb
    int nhalf)                         // halves formed: 2, or the one that has slots
{
    using S = TbShape<MP>;
    __shared__ double2 sA[TB_WAVES][S::G][S::EL];
    __shared__ double2 sV[TB_WAVES][S::G][S::EL];
    __shared__ double2 sT[TB_WAVES][64 * (MP == 1 ? 2 : 1)];   // phases; w of the derivative
    __shared__ double2 sP[TB_WAVES][64 * (MP == 1 ? 2 : 1)];   // projections
    __shared__ double sE[TB_WAVES][S::G][S::N];
    __shared__ int sO[TB_WAVES][S::G][S::N];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane / S::L, l = lane % S::L;            // matrix of the wave, lane of the matrix
    const int P = l / MP, Q = l % MP;
    const int64_t t = ((int64_t)blockIdx.x * TB_WAVES + wave) * S::G + g;
    const bool live = t < (int64_t)nk * nhalf;
    const int k = live ? (int)(nhalf == 2 ? t >> 1 : t) : 0;
    const int half = nhalf == 2 ? (int)(t & 1) : (nc > 0 ? 0 : 1);
    const int n = norb;
    double kx = kpts[3 * k], ky = kpts[3 * k + 1], kz = kpts[3 * k + 2];
    if (half) { kx -= qx; ky -= qy; kz -= qz; }
    double2* A = sA[wave][g];
    double2* V = sV[wave][g];
    double2* ph = &sT[wave][lane - l];
    double* ev = sE[wave][g];
    int* ord = sO[wave][g];
    auto at = [](int r, int c) { return r * S::LD + c; };

    // H(k) of one Fourier table into M: lane (P, Q) forms its 2 x 2 block, the
    // phases L lattice vectors at a time, one per lane
    auto fourier = [&](const double2* __restrict__ tab, double2* M) {
        double2 acc[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = cmk(0, 0);
        for (int r0 = 0; r0 < nr; r0 += S::L) {
            const int r = min(r0 + l, nr - 1);
            const double p = kx * rcart[3 * r] + ky * rcart[3 * r + 1] + kz * rcart[3 * r + 2];
            double s, c;
            sincos(p, &s, &c);
            tb_sync();
            ph[l] = cmk(c, s);
            tb_sync();
            const int cnt = min(S::L, nr - r0);
            for (int j = 0; j < cnt; ++j) {
                const double2 e = ph[j];
                const double2* h = tab + (size_t)(r0 + j) * n * n;
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        if (2 * P + x < n && 2 * Q + y < n) cfma(acc[x][y], h[(2 * P + x) * n + 2 * Q + y], e);
            }
        }
        tb_sync();
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) M[at(2 * P + x, 2 * Q + y)] = acc[x][y];
        tb_sync();
    };
    fourier(hr, A);
    // Exact Hermiticity of the input (the average of the two triangles), V = I.
    double fro = 0.0;
    {
        double2 sym[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int r = 2 * P + x, c = 2 * Q + y;
                const double2 a = A[at(r, c)], b = A[at(c, r)];
                sym[x][y] = cmk(0.5 * (a.x + b.x), (r == c) ? 0.0 : 0.5 * (a.y - b.y));
                fro += cabs2(sym[x][y]);
            }
        tb_sync();
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int r = 2 * P + x, c = 2 * Q + y;
                A[at(r, c)] = sym[x][y];
                V[at(r, c)] = cmk(r == c ? 1.0 : 0.0, 0.0);
            }
        tb_sync();
    }
#pragma unroll
    for (int o = 1; o < S::L; o <<= 1) fro += __shfl_xor(fro, o, 64);
    // Sweeps of N - 1 rounds; pair j of round r is {N - 1, r} (j = 0) or
    // {(r + j) mod (N - 1), (r - j) mod (N - 1)}.  A wave stops when all its
    // matrices have converged.
    for (int sweep = 0; sweep < TB_SWEEPS; ++sweep) {
        double off = 0.0;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int r = 2 * P + x, c = 2 * Q + y;
                if (r < c) off += cabs2(A[at(r, c)]);
            }
#pragma unroll
        for (int o = 1; o < S::L; o <<= 1) off += __shfl_xor(off, o, 64);
        if (__all(off <= 1e-34 * fro)) break;
#pragma unroll 1
        for (int r = 0; r < S::N - 1; ++r) {
            auto pair = [&](int j, int& p, int& q) {
                const int m = S::N - 1;
                int u = (j == 0) ? m : r + j, v = r - j;
                if (j > 0 && u >= m) u -= m;
                if (v < 0) v += m;
                p = min(u, v);
                q = max(u, v);
            };
            int p1, q1, p2, q2;
            pair(P, p1, q1);
            pair(Q, p2, q2);
            const JacobiRot rp = jacobi_rot(A[at(p1, p1)].x, A[at(q1, q1)].x, A[at(p1, q1)]);
            const JacobiRot rq = jacobi_rot(A[at(p2, p2)].x, A[at(q2, q2)].x, A[at(p2, q2)]);
            const double2 a00 = A[at(p1, p2)], a01 = A[at(p1, q2)], a10 = A[at(q1, p2)], a11 = A[at(q1, q2)];
            const double2 v00 = V[at(P, p2)], v01 = V[at(P, q2)], v10 = V[at(P + MP, p2)], v11 = V[at(P + MP, q2)];
            // columns of pair Q, then rows of pair P (J^H from the left)
            const double2 b00 = csub(cscale(a00, rq.c), cmulc(rq.s, a01)), b01 = cadd(cmul(rq.s, a00), cscale(a01, rq.c));
            const double2 b10 = csub(cscale(a10, rq.c), cmulc(rq.s, a11)), b11 = cadd(cmul(rq.s, a10), cscale(a11, rq.c));
            double2 c00 = csub(cscale(b00, rp.c), cmul(rp.s, b10)), c01 = csub(cscale(b01, rp.c), cmul(rp.s, b11));
            double2 c10 = cadd(cmulc(rp.s, b00), cscale(b10, rp.c)), c11 = cadd(cmulc(rp.s, b01), cscale(b11, rp.c));
            if (P == Q) {
                c00 = cmk(a00.x - rp.dl, 0.0);
                c11 = cmk(a11.x + rp.dl, 0.0);
                c01 = c10 = cmk(0, 0);
            }
            tb_sync();
            A[at(p1, p2)] = c00;
            A[at(p1, q2)] = c01;
            A[at(q1, p2)] = c10;
            A[at(q1, q2)] = c11;
            V[at(P, p2)] = csub(cscale(v00, rq.c), cmulc(rq.s, v01));
            V[at(P, q2)] = cadd(cmul(rq.s, v00), cscale(v01, rq.c));
            V[at(P + MP, p2)] = csub(cscale(v10, rq.c), cmulc(rq.s, v11));
            V[at(P + MP, q2)] = cadd(cmul(rq.s, v10), cscale(v11, rq.c));
            tb_sync();
        }
    }
    // ascending order (stable, NaN last, so that ord is a permutation whatever the
    // values); the padding row is not an eigenvalue
    for (int i = l; i < n; i += S::L) {
        const double x = A[at(i, i)].x;
        int rank = 0;
        for (int j = 0; j < n; ++j) {
            const double y = A[at(j, j)].x;
            const bool xn = x != x, yn = y != y;
            if (y < x || (xn && !yn) || ((y == x || (xn && yn)) && j < i)) ++rank;
        }
        ev[i] = x;
        ord[rank] = i;
    }
    tb_sync();
    const int ns = nv + nc;
    // The needed bands, normalised, gauge fixed: one slot per lane.
    const int b_lo = half ? 0 : nv, b_hi = half ? nv : ns;
    for (int slot = b_lo + l; slot < b_hi; slot += S::L) {
        const int band = half ? (n_occ - 1 - slot) : (n_occ + (slot - nv));
        const int col = ord[band];
        double nrm = 0.0, best = -1.0;
        int ib = 0;
        for (int i = 0; i < n; ++i) {
            const double a2 = cabs2(V[at(i, col)]);
            nrm += a2;
            if (a2 > best) { best = a2; ib = i; }
        }
        const double2 piv = V[at(ib, col)];
        const double pa = sqrt(cabs2(piv));
        const double inv = 1.0 / sqrt(nrm);
        const double2 gf = cmk(piv.x / pa * inv, -piv.y / pa * inv);  // conj(piv)/|piv|/||v||
        if (live) {
            double2* out = coef_out + ((size_t)k * ns + slot) * n;
            for (int i = 0; i < n; ++i) out[i] = cmul(V[at(i, col)], gf);
            eps_out[(size_t)k * ns + slot] = ev[col] + (half ? 0.0 : scissor);
        }
    }
    if (dhr == nullptr) return;
    // dH(k) (in place of A), then per slot w = dH c_n, the projections
    // <m|dH|n>/(e_n - e_m) and dc_n = sum_{m != n} c_m proj_m
    tb_sync();
    fourier(dhr, A);
    double2* w = &sT[wave][MP == 1 ? 2 * lane : lane - l];
    double2* pj = &sP[wave][MP == 1 ? 2 * lane : lane - l];
    // (at most the wave's largest slot count, so every lane takes every round)
    for (int sl = 0; sl < max(nv, nc); ++sl) {
        const bool on = sl < b_hi - b_lo;
        const int slot = b_lo + (on ? sl : 0);
        const int band = half ? (n_occ - 1 - slot) : (n_occ + (slot - nv));
        const int col = on ? ord[band] : 0;
        double nrm = 0.0, best = -1.0;
        int ib = 0;
        for (int i = 0; i < n; ++i) {
            const double a2 = cabs2(V[at(i, col)]);
            nrm += a2;
            if (a2 > best) { best = a2; ib = i; }
        }
        const double2 piv = V[at(ib, col)];
        const double pa = sqrt(cabs2(piv));
        const double inv = 1.0 / sqrt(nrm);
        const double2 gf = cmk(piv.x / pa * inv, -piv.y / pa * inv);
        for (int i = l; i < n; i += S::L) {
            double2 acc = cmk(0, 0);
            for (int m = 0; m < n; ++m) cfma(acc, A[at(i, m)], cmul(V[at(m, col)], gf));
            w[i] = acc;
        }
        tb_sync();
        for (int m = l; m < n; m += S::L) {
            const double gap = ev[col] - ev[m];
            double2 proj = cmk(0, 0);                     // <m|dH|n>
            for (int i = 0; i < n; ++i) cfmac(proj, V[at(i, m)], w[i]);
            if (m == col) {
                // with the gauge-fixed c_n: <n|dH|n>
                const double2 d = cmulc(gf, proj);
                if (live && on) deps_out[(size_t)k * ns + slot] = d.x;
                proj = cmk(0, 0);
            } else {
                const bool deg = gap == 0.0;
                proj = cscale(proj, deg ? 0.0 : 1.0 / (deg ? 1.0 : gap));
            }
            pj[m] = proj;
        }
        tb_sync();
        for (int i = l; i < n; i += S::L) {
            double2 dc = cmk(0, 0);
            for (int mb = 0; mb < n; ++mb) {
                const int cm = ord[mb];
                cfma(dc, V[at(i, cm)], pj[cm]);
            }
            if (live && on) dcoef_out[((size_t)k * ns + slot) * n + i] = dc;
        }
        tb_sync();
    }
}

extern "C" hipError_t bse_launch_tb_states(
    hipStream_t st, int nk, int norb, int nr, const double* rcart, const double2* hr,
    const double* kpts, const double* q, int n_occ, int nv, int nc, double scissor,
    const double2* dhr, double* eps, double2* coef, double* deps, double2* dcoef)
{
    if (norb < 1 || norb > TB_MAXORB) return hipErrorInvalidValue;
    const int nhalf = (nv > 0 && nc > 0) ? 2 : 1;
    auto go = [&](auto kernel, int per_wave) {
        const int64_t blocks = ceil_div64((int64_t)nk * nhalf, (int64_t)TB_WAVES * per_wave);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(64 * TB_WAVES), 0, st, nk, norb, nr, rcart, hr, kpts,
                           q[0], q[1], q[2], n_occ, nv, nc, scissor, dhr, eps, coef, deps, dcoef, nhalf);
    };
    // the smallest padded order that holds norb
    if (norb <= 2) go(k_tb_states<1>, TbShape<1>::G);
    else if (norb <= 4) go(k_tb_states<2>, TbShape<2>::G);
    else if (norb <= 8) go(k_tb_states<4>, TbShape<4>::G);
    else go(k_tb_states<8>, TbShape<8>::G);
    return hipGetLastError();
}
