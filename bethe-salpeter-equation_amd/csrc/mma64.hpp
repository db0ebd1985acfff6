// Complex FP64 products of 16 x 16 tiles on matrix cores, operands straight
// from global memory: shared by the grouped back-transform and the full-BSE
// triangular solve.
#pragma once
#include "bse_common.hpp"

typedef double btg_d4 __attribute__((ext_vector_type(4)));
#ifndef BTG_KB
#define BTG_KB 4                  // K steps per prefetched block
#endif

__device__ __forceinline__ btg_d4 btg_mfma(double a, double b, btg_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// c += a b for MT x NT complex 16 x 16 tiles (one K step of 4); a[i] is the
// lane's A element of row tile i, b[j] its B element of column tile j.
template <int MT, int NT>
__device__ __forceinline__ void btg_cmma(btg_d4 (&cr)[MT][NT], btg_d4 (&ci)[MT][NT], const double2 (&a)[MT],
                                         const double2 (&b)[NT]) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) cr[i][j] = btg_mfma(a[i].x, b[j].x, cr[i][j]);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) ci[i][j] = btg_mfma(a[i].x, b[j].y, ci[i][j]);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) cr[i][j] = btg_mfma(-a[i].y, b[j].y, cr[i][j]);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) ci[i][j] = btg_mfma(a[i].y, b[j].x, ci[i][j]);
}

template <int MT, int NT>
__device__ __forceinline__ void btg_zero(btg_d4 (&cr)[MT][NT], btg_d4 (&ci)[MT][NT]) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            cr[i][j] = btg_d4{0.0, 0.0, 0.0, 0.0};
            ci[i][j] = btg_d4{0.0, 0.0, 0.0, 0.0};
        }
}

// Reduction over rows r in [rlo, rhi) of conj(A[r][a]) B[r][b] for one wave's
// 32 x 32 output (2 x 2 tiles).  The
// lane's operand pointers pa[i], pb[j] address row 0 of its column (valid
// flags va, vb).  Inside a block of 4 BTG_KB rows, K step t of lane quad lq
// reads row rb + lq BTG_KB + t, so a lane reads BTG_KB consecutive rows.
__device__ __forceinline__ void btg_rows(btg_d4 (&cr)[2][2], btg_d4 (&ci)[2][2], const double2* const (&pa)[2],
                                         const bool (&va)[2], const double2* const (&pb)[2], const bool (&vb)[2],
                                         int rlo, int rhi, int lq) {
    double2 a[BTG_KB][2], b[BTG_KB][2];
    auto load = [&](int rb, double2 (&A)[BTG_KB][2], double2 (&B)[BTG_KB][2]) {
#pragma unroll
        for (int t = 0; t < BTG_KB; ++t) {
            const int r = rb + lq * BTG_KB + t;
            const bool in = r < rhi;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const double2 v = (in && va[i]) ? pa[i][r] : cmk(0, 0);
                A[t][i] = cmk(v.x, -v.y);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) B[t][j] = (in && vb[j]) ? pb[j][r] : cmk(0, 0);
        }
    };
    if (rlo >= rhi) return;
    load(rlo, a, b);
    for (int rb = rlo; rb < rhi; rb += 4 * BTG_KB) {
        double2 an[BTG_KB][2], bn[BTG_KB][2];
        const bool more = rb + 4 * BTG_KB < rhi;
        if (more) load(rb + 4 * BTG_KB, an, bn);
#pragma unroll
        for (int t = 0; t < BTG_KB; ++t) btg_cmma<2, 2>(cr, ci, a[t], b[t]);
        if (more) {
#pragma unroll
            for (int t = 0; t < BTG_KB; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i) { a[t][i] = an[t][i]; b[t][i] = bn[t][i]; }
        }
    }
}
