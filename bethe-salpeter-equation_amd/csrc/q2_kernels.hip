// K7, two-stage form with many vectors: Z <- Q2 Z, where Q2 is the product of
// the bulge chase's reflectors (chase_kernels.hip), H_{s,k} acting on rows
// s + 1 + 32 k .. s + 32 + 32 k.  Later sweeps are applied first; within a
// sweep the reflectors commute.
//
// Thirty-two consecutive sweeps S (s = 32 S + j) at one k form a block on the 63
// rows from 32 q + 1, q = S + k.  Blocks of one S run with increasing q; block
// (S, q) follows block (S + 1, q + 1), which overlaps it, and nothing else.
//
// The reflectors are applied as they are, z -= tau v (v^H z): the compact form of
// a block would put a 63 x 32 parallelogram through the matrix cores, twice the
// multiplications at the same FP64 rate as the vector units'.  A workgroup owns
// a strip of 16 columns, so strips need no synchronisation.  Four lanes share a
// column: lane part h holds rows 4 t + h (t = 0 .. 15) of a 64-row window in
// registers, and a reflector's rows are 8 registers, 9 when its first row does
// not start a group of four (v is zero outside its 32 rows).  v comes from LDS,
// one address per part.  Two reflectors at a time: both dots are taken of the
// same z and the second is corrected by v_0^H v_1, so that the parts' partial
// dots meet by lane exchanges once per pair.  Sixteen reflectors are unrolled
// (register indices must be known); then the window turns by their four
// registers, so the same code serves the next sixteen.  All 32 unrolled waited
// for the instruction cache (70 KB of code; 192 ms instead of 150 at n = 8096).
//
// The four waves of a workgroup run four consecutive S of the same strip, each
// one block behind the one before: chunk q (rows 32 q + 1 ..) of Z goes from wave
// to wave through LDS and to memory only after the fourth, so Z is read and
// written once per 128 sweeps.  Wave 0 takes the next four S as soon as it is
// free; a pass p (S = C - 1 - 4 p - w) starts q2_start(p) block steps after the
// first, so that wave 3 is done with the chunk that wave 0 reads again.
//
// Bound by instruction issue of the vector units: 56 % of a block's instructions
// are its FP64 multiply-adds (8 n^3 flops for n columns).  n = 8096, all columns:
// 150 ms (28 TFLOP/s), 179 ms with each dot's parts summed on their own and the
// window turned every eight reflectors; n = 3600: 20 ms, one wave a SIMD.
#include "bse_common.hpp"

#define Q2_W 4                    // waves of a workgroup = sweep groups in flight
#define Q2_NC 16                  // columns of a strip
#define Q2_H 4                    // lanes of a column
#define Q2_T (32 / Q2_H)          // registers of a chunk
#define Q2_LDV (32 + 2 * (Q2_H - 1))

__device__ inline int q2_start(int p) { return 2 * p * (p - 1) + 5 * p; }   // sum of 4 i + 5, i < p

// Exchange of lane rows of 32 (16) between two registers: x keeps its even rows
// and takes y's, y the odd ones of both.
__device__ __forceinline__ void q2_swap32(double& x, double& y) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false, false);
    x = __hiloint2double((int)hi[0], (int)lo[0]);
    y = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ void q2_swap16(double& x, double& y) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(x), __double2loint(y), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(x), __double2hiint(y), false, false);
    x = __hiloint2double((int)hi[0], (int)lo[0]);
    y = __hiloint2double((int)hi[1], (int)lo[1]);
}
// Sums of two complex numbers over the four parts of the wave, in every lane: the
// four real sums are folded until each part holds one, then handed back.
__device__ __forceinline__ void q2_parts(double2& a, double2& b) {
    q2_swap32(a.x, b.x);
    q2_swap32(a.y, b.y);
    double x = a.x + b.x, y = a.y + b.y;        // parts 0, 1: a; parts 2, 3: b
    q2_swap16(x, y);
    double re = x + y, im = re;                 // a.x, a.y, b.x, b.y
    q2_swap16(re, im);
    a.x = b.x = re;
    a.y = b.y = im;
    q2_swap32(a.x, b.x);
    q2_swap32(a.y, b.y);
}

// Rows of reflector J in registers T0 .. T0 + NT - 1 of the window.
template <int J> struct Q2Rows {
    static constexpr int T0 = J / Q2_H, NT = Q2_T + (J % Q2_H ? 1 : 0);
};
template <int J>
__device__ __forceinline__ void q2_load(const double2* sv, double2 (&v)[Q2_T + 1]) {
#pragma unroll
    for (int t = 0; t < Q2Rows<J>::NT; ++t) v[t] = sv[Q2_H - 1 + Q2_H * (Q2Rows<J>::T0 + t) - J];
}
template <int J>
__device__ __forceinline__ double2 q2_dot(const double2 (&z)[2 * Q2_T], const double2 (&v)[Q2_T + 1]) {
    double r0 = 0.0, r1 = 0.0, i0 = 0.0, i1 = 0.0;
#pragma unroll
    for (int t = 0; t < Q2Rows<J>::NT; ++t) {
        const double2 x = z[Q2Rows<J>::T0 + t];
        r0 = fma(v[t].x, x.x, r0);
        i0 = fma(v[t].x, x.y, i0);
        r1 = fma(v[t].y, x.y, r1);
        i1 = fma(-v[t].y, x.x, i1);
    }
    return cmk(r0 + r1, i0 + i1);
}
template <int J>
__device__ __forceinline__ void q2_sub(double2 (&z)[2 * Q2_T], const double2 (&v)[Q2_T + 1], double2 f) {
#pragma unroll
    for (int t = 0; t < Q2Rows<J>::NT; ++t) {
        double2& x = z[Q2Rows<J>::T0 + t];
        x.x = fma(-f.x, v[t].x, fma(f.y, v[t].y, x.x));
        x.y = fma(-f.x, v[t].y, fma(-f.y, v[t].x, x.y));
    }
}
// Reflectors J (odd) and then J - 1 of the window's last sixteen; sv, tau and g of
// the half block.
template <int J>
__device__ __forceinline__ void q2_pairs(double2 (&z)[2 * Q2_T], const double2* sv, const double2* tau,
                                         const double2* g) {
    double2 v1[Q2_T + 1], v0[Q2_T + 1];
    q2_load<J>(sv + (J & 15) * Q2_LDV, v1);
    q2_load<J - 1>(sv + ((J - 1) & 15) * Q2_LDV, v0);
    const double2 t1 = tau[J & 15], t0 = tau[(J - 1) & 15], gg = g[(J & 15) >> 1];
    double2 d1 = q2_dot<J>(z, v1), d0 = q2_dot<J - 1>(z, v0);
    q2_parts(d1, d0);
    const double2 f1 = cmul(t1, d1), f0 = cmul(t0, csub(d0, cmul(gg, f1)));
    q2_sub<J>(z, v1, f1);
    q2_sub<J - 1>(z, v0, f0);
    // one pair's operands at a time: more would cost the second workgroup of a CU
    __builtin_amdgcn_sched_barrier(0);
    if constexpr ((J & 15) > 1) q2_pairs<J - 2>(z, sv, tau, g);
}

// Grid: strips of columns.  C = ceil((n - 1) / 32) groups of sweeps = chunks of rows.
__global__ __launch_bounds__(64 * Q2_W, 2) void k_q2_apply(int n, int C, const double2* __restrict__ V2,
                                                           double2* __restrict__ Z, int64_t ldz, int ncols)
{
    __shared__ double2 sV[Q2_W][16 * Q2_LDV];       // half a block's reflectors
    __shared__ double2 sTau[Q2_W][16], sG[Q2_W][8];
    __shared__ double2 ring[Q2_W - 1][32 * Q2_NC];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int h = lane >> 4, c = lane & 15;
    const int col = blockIdx.x * Q2_NC + c;
    const bool on = col < ncols;
    double2* zc = Z + (int64_t)min(col, ncols - 1) * ldz + 1 + h;     // row 0 of chunk 0, this part
    double2* sv = sV[w];
    auto lds_order = [] {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
        __builtin_amdgcn_wave_barrier();
    };
    // rows 32 q + 1 + 4 t + h, t < 8
    auto load = [&](int q, double2 (&x)[Q2_T]) {
#pragma unroll
        for (int t = 0; t < Q2_T; ++t) {
            const int r = 32 * q + 1 + Q2_H * t + h;
            const double2 a = zc[min(32 * q + Q2_H * t, n - 2 - h)];
            x[t] = cmk(r < n ? a.x : 0.0, r < n ? a.y : 0.0);
        }
    };
    double2 vn[8];
    // reflectors 16 half .. of block (S, k): two per 64 lanes
    auto fetch = [&](int S, int k, int half) {
        const double2* b = V2 + bse_q2_block(C, S, k) + 512 * half;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool valid = 32 * S + 16 * half + 2 * u + (lane >> 5) <= n - 2 - 32 * k;
            const double2 a = b[64 * u + lane];
            vn[u] = cmk(valid ? a.x : 0.0, valid ? a.y : 0.0);
        }
    };
    // ... into LDS, with tau and the products v_j^H v_{j+1}, j even, of the pairs
    auto stage = [&](int S, int k, int half) {
        lds_order();
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int j = 2 * u + (lane >> 5), e = lane & 31;
            const bool valid = 32 * S + 16 * half + j <= n - 2 - 32 * k;
            if (e == 0) sTau[w][j] = vn[u];
            sv[j * Q2_LDV + Q2_H - 1 + e] = cmk(e == 0 ? (valid ? 1.0 : 0.0) : vn[u].x, e == 0 ? 0.0 : vn[u].y);
        }
        lds_order();
        const int pr = lane >> 3, part = lane & 7;
        double2 g = cmk(0, 0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // entry e of v_{j+1} meets entry e + 1 of v_j (zero beyond the last)
            const int e = 8 * t + part;
            cfmac(g, sv[2 * pr * Q2_LDV + Q2_H + e], sv[(2 * pr + 1) * Q2_LDV + Q2_H - 1 + e]);
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            g.x += __shfl_xor(g.x, o, 64);
            g.y += __shfl_xor(g.y, o, 64);
        }
        if (part == 0) sG[w][pr] = g;
        lds_order();
    };
    // entries outside a reflector's rows
    for (int e = lane; e < 16 * Q2_LDV; e += 64) sv[e] = cmk(0, 0);
    const int npass = (C + Q2_W - 1) / Q2_W;
    int total = 0;
    for (int p = 0; p < npass; ++p)
        for (int u = 0; u < Q2_W; ++u) {
            const int S = C - 1 - Q2_W * p - u;
            if (S >= 0) total = max(total, q2_start(p) + u + C - S);
        }
    // z: chunk q in registers 0 .. 7 and chunk q + 1 in 8 .. 15
    double2 z[2 * Q2_T], nxt[Q2_T];
#pragma unroll
    for (int t = 0; t < Q2_T; ++t) z[t] = z[Q2_T + t] = nxt[t] = cmk(0, 0);
    int p = 0, i = 0;
    int S = C - 1 - w;
    bool live = S >= 0;
    if (live) fetch(S, 0, 1);
    for (int T = 0; T < total; ++T) {
        const bool act = live && T >= q2_start(p) + w;        // uniform over the wave
        const int q = S + i;
        if (act) {
            if (i == 0) {
                double2 lo[Q2_T];
                load(q, lo);
                if (w == 0 && q + 1 < C) load(q + 1, nxt);
#pragma unroll
                for (int t = 0; t < Q2_T; ++t) z[t] = lo[t];
            }
#pragma unroll
            for (int t = 0; t < Q2_T; ++t) {
                if (q + 1 >= C) z[Q2_T + t] = cmk(0, 0);
                else if (w == 0) z[Q2_T + t] = nxt[t];
                else z[Q2_T + t] = ring[w - 1][64 * t + lane];
            }
        }
        __syncthreads();
        if (act) {
            // operands of what comes next are in flight behind the arithmetic
            const bool lastq = q + 1 >= C;
            if (w == 0 && q + 2 < C) load(q + 2, nxt);
#pragma unroll 1
            for (int half = 1; half >= 0; --half) {
                stage(S, i, half);
                if (half) fetch(S, i, 0);
                else if (!lastq) fetch(S, i + 1, 1);
                else if (S >= Q2_W) fetch(S - Q2_W, 0, 1);
                q2_pairs<31>(z, sv + h, sTau[w], sG[w]);
#pragma unroll
                for (int t = 0; t < Q2_T / 2; ++t) {
                    const double2 a = z[12 + t];
                    z[12 + t] = z[8 + t];
                    z[8 + t] = z[4 + t];
                    z[4 + t] = z[t];
                    z[t] = a;
                }
            }
            // half a turn: the finished chunk q is in 8 .. 15, chunk q + 1 in 0 .. 7
            const bool out = w == Q2_W - 1 || S == 0;
#pragma unroll
            for (int t = 0; t < Q2_T; ++t) {
                if (!out) ring[w][64 * t + lane] = z[Q2_T + t];
                else if (on && 32 * q + 1 + Q2_H * t + h < n) zc[32 * q + Q2_H * t] = z[Q2_T + t];
            }
            if (!lastq) {
                ++i;
            } else {
                ++p;
                i = 0;
                S -= Q2_W;
                live = S >= 0;
            }
        }
        __syncthreads();
    }
}

// Complex elements of the reflector store.
extern "C" int64_t bse_q2_workspace(int n)
{
    const int C = n > 1 ? (int)ceil_div64(n - 1, 32) : 0;
    return bse_q2_block(C, 0, C);
}

// Z (n x ncols, ld ldz) <- Q2 Z.
extern "C" hipError_t bse_apply_q2(hipStream_t st, int n, const double2* V2, double2* Z, int64_t ldz, int ncols)
{
    if (n < 2 || ncols <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_q2_apply, dim3((unsigned)ceil_div64(ncols, Q2_NC)), dim3(64 * Q2_W), 0, st, n,
                       (int)ceil_div64(n - 1, 32), V2, Z, ldz, ncols);
    return hipGetLastError();
}
