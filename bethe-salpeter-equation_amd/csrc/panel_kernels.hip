// K5, one-stage form: one panel of up to 32 columns of the Householder
// reduction (hetrd_kernels.hip) in a single launch, for trailing blocks whose
// column step is bound by latency.
//
// The three dependent launches of a column step (column update, Hermitian
// product, reduction of its partials) cost 27 us a column however small the
// trailing block is.  Here the workgroups stay and hand data on through
// tagged messages (resident.hpp), two per column:
//   owners -> tiles   the updated column x, 64 rows per owner;
//   tiles -> owners   partial products of A22 x.
// Workgroup b < nbk owns the 64 rows of tile row b: it keeps their rows of V
// and W in LDS, reduces the partials of its rows, forms their v, w and at
// once the next column.  What a step needs of all rows is arranged so that
// no third exchange is needed:
//   - ||x||^2, x^H a(:, s0) and W^H x, V^H x are published by the owners with x and
//     summed by every owner, x^H A x likewise by the tile workgroups;
//   - y^H v, which w = y - (tau/2)(y^H v) v needs, is the quadratic form
//       conj(tau) (v^H A v - 2 Re (W^H v)^H (V^H v)),  v = e_1 + sc x,
//       v^H A v = |sc|^2 x^H A x + 2 Re(conj(sc) x^H A e_1) + a(s0, s0);
//   - the next column is s0 itself, and its update needs row s0 of V and W:
//     published one step earlier up to the newest column, where V(s0) = 1 and
//     every owner sums W(s0) itself from the partials of that one row.
// x^H A x is of third order in the matrix, so x is that column in units of the
// matrix (times 2^-e, 2^e <= max |a| < 2^(e+1), an exact scaling): without them a matrix
// of size 1e-129 had x^H A x = 0 and one of 1e120 an infinite one.  d and beta take
// the 2^e back; everything else is formed from v = e_1 + sc x, which has none.
//
// Tiles: NT 64 x 64 tiles of the lower triangle per workgroup, 8 columns of each
// per wave, kept in registers for the whole panel (the panel does not change
// A); with four, the last one is read again for each column (it would not
// fit beside the rest).  Row sums stay in the lanes and are added over the
// waves in LDS, column sums go through lane exchanges.
//
// What an owner needs arrives at two times: the sums over x (norm, dots, rows
// of V and W) soon after x, the partial products a tile product and a message
// later.  So it polls the former first and forms the reflector and the panel
// corrections from them while the latter are on their way.
//
// Reuse of the message areas.  Each has two copies by the column's parity, so a
// workgroup's words for column c + 2 replace those for column c, which every
// reader must have read by then.  A workgroup posts words for column c + 2
// only once it holds a word of x(c + 2), and the owner that posted this word had
// finished column c + 1, in which it waited for the sums over x(c + 1) of every
// owner, posted by each behind its last read of column c; and it waited for
// x^H A x of column c + 1 from every workgroup, posted behind their last read of
// x(c).  So every workgroup has to wait for some row of x in every column, row
// s0 included (pn_awaits): the last row of an order 64 k + 1 is s0 itself in the
// last column, and all there is to wait for in tile (k, k).  An owner needs no
// such row: it has finished column c + 1 itself.  Tile row 0 can be behind s0,
// but its tile (0, 0) is workgroup 0's, an owner; every other one reaches s0 or
// beyond (bse_panel_unawaited counts what does not, on the host).
//
// Every sum runs in a fixed order.  FP64 throughout; T is the storage type.
//
// Measured (FP64 storage), us per column: 6.7 with 3 tile rows, 7.9 with 22 (one
// tile per workgroup), 12.7, 17 and 21.6 with two, three and four tiles,
// against 27 (orders up to 3600) for the three launches.  Whole reductions:
// N = 144 3.0 to 1.3 ms, 2304 57 to 27 ms, 2592 65 to 33 ms, 3600 99 to 66 ms.  A
// column is bound by the latency of two messages and of about 700 dependent
// instructions of one wave.
#include "resident.hpp"
#include <cfloat>

#define PN_WAVES 8
#define PN_THREADS (64 * PN_WAVES)
#define PN_B 32                // panel width
#define PN_ROWMSG (2 * PN_B * 2)
#define PN_MAXTILES 4          // tiles of a workgroup (beyond, the column step streams the trailing block)

struct PanelArgs {
    int n, j0, nbp;            // order, first column, columns of this panel
    int tc0, nbk, ntl;         // first tile row, tile rows, tiles
    const void* A;             // tiled lower storage
    double2* Vp;               // (n - j0) x 32 reflectors
    double2* Wp;               // (n - j0) x 32
    double2* alpha2;           // 32, zeroed here (W is complete)
    double2* G;                // 64 x 64 Gram block of the panel
    double* d;
    double* e;
    double2* tau;
    bse_i4v* msg;
    unsigned* meet;
    int* err;
    const double* big;         // the matrix's largest |Re a|, |Im a| before the first panel
};

// Message areas, in 16-byte words (two copies each, by the column's parity).
struct PanelMsg {
    int x, s, dot, q, row, p;                  // offsets
    int xs, ss, ds, qs, rs, ps;                // sizes of one copy
    int64_t total;
};
__host__ __device__ inline PanelMsg panel_msg(int nbk, int grid) {
    PanelMsg L;
    L.xs = nbk * 64 * 2;                           // x
    L.ss = nbk * 4;                                // (||x||^2, -), x^H a(:, s0)
    L.ds = nbk * PN_B * 2 * 2;                     // W^H x, V^H x
    L.qs = (grid + 1) & ~1;                        // x^H A x per workgroup
    L.rs = PN_ROWMSG;                              // a row of W, V
    L.ps = nbk * (nbk + 1) * 64 * 2;               // partial products
    L.x = 0;
    L.s = L.x + 2 * L.xs;
    L.dot = L.s + 2 * L.ss;
    L.q = L.dot + 2 * L.ds;
    L.row = L.q + 2 * L.qs;
    L.p = L.row + 2 * L.rs;
    L.total = (int64_t)L.p + 2 * (int64_t)L.ps;
    return L;
}

// Whether a tile waits for row g of x in the column with x below row s0: its rows
// below s0 and, for the reuse rule above, s0 itself (which takes no part).
__host__ __device__ inline bool pn_awaits(int g, int s0, int n) { return g >= s0 && g < n; }

// R complex values, value u at word off[u] (off < 0: not wanted, zero), all
// polled together.  False when the wait was given up.
template <int R>
__device__ __attribute__((always_inline)) inline bool pn_poll(__amdgpu_buffer_rsrc_t r, const int (&off)[R], int tag,
                                                              double2 (&v)[R], int* err)
{
    unsigned spins = 0;
    for (;;) {
        asm volatile("" ::: "memory");
        bse_i4v a[R], b[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int o = off[u] >= 0 ? off[u] * 16 : 0;
            a[u] = __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, RS_COHERENT);
            b[u] = __builtin_amdgcn_raw_buffer_load_b128(r, o + 16, 0, RS_COHERENT);
        }
        bool ok = true;
#pragma unroll
        for (int u = 0; u < R; ++u) ok = ok && (off[u] < 0 || (rs_here(a[u], tag) && rs_here(b[u], tag)));
        if (__all(ok)) {
#pragma unroll
            for (int u = 0; u < R; ++u)
                v[u] = cmk(off[u] >= 0 ? rs_value(a[u]) : 0.0, off[u] >= 0 ? rs_value(b[u]) : 0.0);
            return true;
        }
        if (rs_give_up(spins, err)) return false;
    }
}
__device__ inline void pn_post(__amdgpu_buffer_rsrc_t r, int off, double2 v, int tag) {
    __builtin_amdgcn_raw_buffer_store_b128(rs_word(v.x, tag), r, off * 16, 0, RS_COHERENT);
    __builtin_amdgcn_raw_buffer_store_b128(rs_word(v.y, tag), r, off * 16 + 16, 0, RS_COHERENT);
}
__device__ inline void pn_post1(__amdgpu_buffer_rsrc_t r, int off, double v, int tag) {
    __builtin_amdgcn_raw_buffer_store_b128(rs_word(v, tag), r, off * 16, 0, RS_COHERENT);
}

// Lane exchanges: a becomes the half-wave (row-of-16 pair) sum of a in the
// lanes that keep it, of b in the others.
__device__ inline double pn_swap32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double pn_swap16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double2 pn_swap32(double2 a, double2 b) { return cmk(pn_swap32(a.x, b.x), pn_swap32(a.y, b.y)); }
__device__ inline double2 pn_swap16(double2 a, double2 b) { return cmk(pn_swap16(a.x, b.x), pn_swap16(a.y, b.y)); }
template <int CTRL> __device__ inline double2 pn_dpp(double2 v) {
    return cmk(dpp_mov_d<CTRL, 0xF>(v.x), dpp_mov_d<CTRL, 0xF>(v.y));
}
__device__ inline double2 pn_sel(bool c, double2 a, double2 b) { return cmk(c ? a.x : b.x, c ? a.y : b.y); }
// Sums over the wave of 8 values per lane, given as p[k] = swap32 of values k
// and k + 4: that of value pn_col8(lane), in the eight lanes that share it.
__device__ inline int pn_col8(int lane) { return 4 * (lane >> 5) + 2 * ((lane >> 4) & 1) + ((lane >> 3) & 1); }
__device__ inline double2 pn_sum8(const double2 (&p)[4], int lane) {
    const double2 a = pn_swap16(p[0], p[2]), b = pn_swap16(p[1], p[3]);
    const bool b3 = (lane >> 3) & 1;
    double2 v = cadd(pn_sel(b3, b, a), pn_dpp<0x128>(pn_sel(b3, a, b)));   // row_ror:8
    v = cadd(v, pn_dpp<0x141>(v));
    v = cadd(v, pn_dpp<0xB1>(v));
    return cadd(v, pn_dpp<0x4E>(v));
}

template <typename T, int NT>
__global__ __launch_bounds__(PN_THREADS) void k_trd_panel(PanelArgs a)
{
    constexpr int CQ = 64 / PN_WAVES;                // columns of a wave
    constexpr int NR = NT < 4 ? NT : 3;              // tiles kept in registers
    constexpr int PL = 4, PD = 3;                    // values polled at once: late, early
    constexpr int LW = PN_WAVES - 2;                 // waves that poll the partials of an owner's rows
    __shared__ double2 sV[PN_B][64], sW[PN_B][64];
    __shared__ double2 sAcc[PN_WAVES][64], sXp[PN_WAVES][64];
    __shared__ double2 sXr[NT][64], sXc[NT][64], sX[64];
    __shared__ double2 sRS[NT][PN_WAVES][64], sCS[NT][64];
    __shared__ double2 sDot[2][PN_B], sRow[2][PN_B];   // [0]: with W, [1]: with V
    __shared__ double sS[2][3], sC[5], sB[4], sQ, sQw[PN_WAVES];
    __shared__ int go;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wg = blockIdx.x;
    const int n = a.n, j0 = a.j0, nt = tile_count(n), m = n - j0, G = gridDim.x;
    const int R0 = 64 * a.tc0;
    const T* A = (const T*)a.A;
    const PanelMsg L = panel_msg(a.nbk, G);
    const __amdgpu_buffer_rsrc_t rm = bse_rsrc(a.msg, (int)(L.total * 16));
    // units of x: 2^ex (1 for a zero matrix or one that is not finite)
    const double big = *a.big;
    const int ex = (big > 0.0 && big <= DBL_MAX) ? max(-1000, min(1000, ilogb(big))) : 0;
    const double up = ldexp(1.0, -ex), down = ldexp(1.0, ex);
    const bool owner = wg < a.nbk;
    const int grow = R0 + 64 * wg + lane;              // an owner's row of this lane
    int I[NT], J[NT];                                  // tiles wg, wg + G, ..; I < 0: none
#pragma unroll
    for (int r = 0; r < NT; ++r) {
        I[r] = J[r] = -1;
        if (wg + r * G < a.ntl) tri_tile(wg + r * G, I[r], J[r]);
    }
    T el[NR][CQ], es[CQ];
    auto load = [&](int r, T (&e)[CQ]) {
        const bool ok = I[r] >= 0;
        const T* p = A + (ok ? tile_pos(a.tc0 + I[r], a.tc0 + J[r], nt) : 0) * (BSE_TILE * BSE_TILE) + w * CQ * 64 + lane;
#pragma unroll
        for (int q = 0; q < CQ; ++q) {
            const T x = p[q * 64];
            e[q].x = ok ? x.x : 0;
            e[q].y = ok ? x.y : 0;
        }
    };
#pragma unroll
    for (int r = 0; r < NR; ++r) load(r, el[r]);
    if (tid == 0) go = (__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0 &&
                        rs_meet(a.meet, gridDim.x, a.err)) ? 1 : 0;
    __syncthreads();
    if (!go) return;
    // row grow of the stored column c (rows >= c; the diagonal is real)
    auto acol = [&](int c) -> double2 {
        double2 z = cmk(0, 0);
        if (grow >= c && grow < n) z = cplx<T>::load(A + tix(grow, c, nt));
        if (grow == c) z.y = 0.0;
        return z;
    };
    auto diag = [&](int c) { return cplx<T>::load(A + tix(min(c, n - 1), min(c, n - 1), nt)).x; };
    // an owner's sums for column c: ||.||^2 of x below s0 = c + 1 and x^H a(:, s0) (one wave)
    auto post_sums = [&](int c, double2 x, double2 as0) {
        const bool below = grow > c + 1 && grow < n;
        const double nr = wave_sum_dpp(below ? cabs2(x) : 0.0);
        const double2 px = cmulc(x, as0);
        const double p0 = wave_sum_dpp(below ? px.x : 0.0), p1 = wave_sum_dpp(below ? px.y : 0.0);
        const double v = lane == 0 ? nr : (lane == 2 ? p0 : (lane == 3 ? p1 : 0.0));
        if (lane < 4) pn_post1(rm, L.s + (c & 1) * L.ss + wg * 4 + lane, v, c + 1);
    };
    // wave 0 of an owner holds its rows of x, of column s0 and of the one after
    // (also in wave 1), and a(s0, s0), each loaded a column ahead
    double2 xown = cmk(0, 0), as0 = cmk(0, 0), as1 = cmk(0, 0);
    double a11 = 0.0, a11n = 0.0;
    if (owner && w < 2) {
        xown = cscale(acol(j0), up);
        as0 = acol(j0 + 1);
        if (w == 0) {
            a11 = diag(j0 + 1);
            if (grow >= j0 && grow < n) pn_post(rm, L.x + (j0 & 1) * L.xs + (wg * 64 + lane) * 2, xown, j0 + 1);
        } else {
            post_sums(j0, xown, as0);
        }
    }
    if (wg == 0 && tid < PN_B) a.alpha2[tid] = cmk(0, 0);
    for (int i = 0; i < a.nbp; ++i) {
        const int c = j0 + i, s0 = c + 1, tag = c + 1, par = c & 1;
        const bool more = i + 1 < a.nbp;
        if (owner && w < 2 && more) {
            as1 = acol(s0 + 1);
            if (w == 0) a11n = diag(s0 + 1);
        }
        // ---------------- tiles
        if (NT > NR) load(NT - 1, es);
        if (w < 2 * NT) {
            const int r = w >> 1;
            int tb = -1;
#pragma unroll
            for (int k = 0; k < NT; ++k) tb = (r == k) ? ((w & 1) ? J[k] : I[k]) : tb;
            const int g = R0 + 64 * tb + lane;
            const int off[1] = {(tb >= 0 && pn_awaits(g, s0, n)) ? L.x + par * L.xs + (tb * 64 + lane) * 2 : -1};
            double2 v[1];
            if (!pn_poll<1>(rm, off, tag, v, a.err)) return;
            const double2 x = pn_sel(g == s0, cmk(0, 0), v[0]);
            if (w & 1) sXc[r][lane] = x;
            else sXr[r][lane] = x;
        }
        __syncthreads();
        double ql = 0.0;
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            const double2 xr = sXr[r][lane];
            auto elem = [&](int q) {
                const T x = r < NR ? el[r < NR ? r : 0][q] : es[q];
                return cmk((double)x.x, (double)x.y);
            };
            double2 acc = cmk(0, 0), p[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                cfma(acc, elem(q), sXc[r][w * CQ + q]);
                cfma(acc, elem(q + 4), sXc[r][w * CQ + q + 4]);
                p[q] = pn_swap32(cmulc(elem(q), xr), cmulc(elem(q + 4), xr));
            }
            // (the eight lanes that share a sum write the same value)
            sCS[r][w * CQ + pn_col8(lane)] = pn_sum8(p, lane);
            if (I[r] == J[r]) {
                // a diagonal tile's diagonal is in both sums: take it off once
                double dg = 0.0;
#pragma unroll
                for (int q = 0; q < CQ; ++q) dg = (w * CQ + q == lane) ? elem(q).x : dg;
                acc = csub(acc, cscale(xr, dg));
                ql += dg * cabs2(xr);
            }
            ql += 2.0 * (xr.x * acc.x + xr.y * acc.y);     // x_I^H (A x_J) and its conjugate
            sRS[r][w][lane] = acc;
        }
        ql = wave_sum_dpp(ql);
        if (lane == 0) sQw[w] = ql;
        __syncthreads();
        if (w < 2 * NT) {
            const int r = w >> 1;
            const bool col = w & 1;
            int ti = -1, tj = -1;
#pragma unroll
            for (int k = 0; k < NT; ++k) { ti = (r == k) ? I[k] : ti; tj = (r == k) ? J[k] : tj; }
            if (ti >= 0) {
                double2 v = cmk(0, 0);
                if (!col) {
#pragma unroll
                    for (int k = 0; k < PN_WAVES; ++k) v = cadd(v, sRS[r][k][lane]);
                } else {
                    v = sCS[r][lane];
                }
                // tile row K: slots J = 0 .. K of its tiles, then K + 1 + (I - K) of its tile column
                const int K = col ? tj : ti, slot = col ? tj + 1 + (ti - tj) : tj;
                pn_post(rm, L.p + par * L.ps + ((K * (a.nbk + 1) + slot) * 64 + lane) * 2, v, tag);
            }
        }
        if (w == PN_WAVES - 1 && lane == 0) {
            double q = 0.0;
#pragma unroll
            for (int k = 0; k < PN_WAVES; ++k) q += sQw[k];
            pn_post1(rm, L.q + par * L.qs + wg, q, tag);
            // (the words are read in pairs)
            if (wg == G - 1 && (G & 1)) pn_post1(rm, L.q + par * L.qs + G, 0.0, tag);
        }
        if (!owner) continue;
        // ---------------- owners, early: the sums over x, alpha and d, row s0 of W and V
        {
            // dots: eight lanes per sum, tile rows kk, kk + 8, ..
            const int kk = tid & 7, l = tid >> 4, which = (tid >> 3) & 1;
            auto dot_off = [&](int b) {
                return (l < i && b < a.nbk) ? L.dot + par * L.ds + ((b * 2 + which) * PN_B + l) * 2 : -1;
            };
            int off[PD + 2];
            double2 v[PD + 2];
#pragma unroll
            for (int u = 0; u < PD; ++u) off[u] = dot_off(kk + 8 * u);
            off[PD] = off[PD + 1] = -1;
            if (w == 7) {
                // (at most 64 tile rows)
                if (lane < a.nbk) {
                    off[PD] = L.s + par * L.ss + lane * 4;
                    off[PD + 1] = off[PD] + 2;
                }
            } else if (w == 6) {
                if (lane < 2) off[PD] = L.x + par * L.xs + ((lane == 0 ? s0 : c) - R0) * 2;
            } else if (w == 5) {
                if ((lane & 31) < i) off[PD] = L.row + par * L.rs + lane * 2;
            }
            if (!pn_poll<PD + 2>(rm, off, tag, v, a.err)) return;
            double2 sum = cmk(0, 0);
#pragma unroll
            for (int u = 0; u < PD; ++u) sum = cadd(sum, v[u]);
            if (w == 7) {
                const double x0 = wave_sum_dpp(v[PD].x), p0 = wave_sum_dpp(v[PD + 1].x), p1 = wave_sum_dpp(v[PD + 1].y);
                if (lane == 0) { sS[0][0] = x0; sS[0][1] = p0; sS[0][2] = p1; }
            } else if (w == 6) {
                if (lane == 0) { sC[2] = v[PD].x; sC[3] = v[PD].y; }
                if (lane == 1) sC[4] = v[PD].x;
            } else if (w == 5) {
                sRow[lane >> 5][lane & 31] = v[PD];
            }
            for (int b0 = 8 * PD; b0 < a.nbk; b0 += 8 * PD) {
                int od[PD];
                double2 vd[PD];
#pragma unroll
                for (int u = 0; u < PD; ++u) od[u] = dot_off(b0 + kk + 8 * u);
                if (!pn_poll<PD>(rm, od, tag, vd, a.err)) return;
#pragma unroll
                for (int u = 0; u < PD; ++u) sum = cadd(sum, vd[u]);
            }
            sum = cadd(sum, pn_dpp<0x141>(sum));
            sum = cadd(sum, pn_dpp<0xB1>(sum));
            sum = cadd(sum, pn_dpp<0x4E>(sum));
            if (kk == 0) sDot[which][l] = sum;
        }
        __syncthreads();
        // ---------------- with dW = W^H x, dV = V^H x, w0 and v0 the rows s0 of W, V:
        // t1 = conj(w0) + sc dW, t2 = conj(v0) + sc dV, so V t1 + W t2 = xp + sc D with
        //   xp = V conj(w0) + W conj(v0)   (also the next column's update),
        //   D  = V dW + W dV;
        // the sums over l go to waves 1 .. 7, wave 0 forms the reflector
        double beta = 0.0, al2 = 0.0;
        double2 tau = cmk(0, 0), sc = cmk(0, 0);
        if (w == 0) {
            const double2 alpha = cmk(sC[2], sC[3]);
            const double xn2 = sS[0][0];
            beta = alpha.x;
            if (!(xn2 == 0.0 && alpha.y == 0.0)) {
                const double nr = sqrt(alpha.x * alpha.x + alpha.y * alpha.y + xn2);
                beta = (alpha.x >= 0.0) ? -nr : nr;
                tau = cmk((beta - alpha.x) / beta, -alpha.y / beta);
                sc = crecip_safe(cmk(alpha.x - beta, alpha.y), nr);
            }
        } else {
            double2 xp = cmk(0, 0), D = cmk(0, 0);
#pragma unroll
            for (int u = 0; u < (PN_B + PN_WAVES - 2) / (PN_WAVES - 1); ++u) {
                const int l = w - 1 + (PN_WAVES - 1) * u;
                if (l < i) {
                    const double2 V = sV[l][lane], W = sW[l][lane];
                    cfma(xp, V, cconj(sRow[0][l]));
                    cfma(xp, W, cconj(sRow[1][l]));
                    cfma(D, V, sDot[0][l]);
                    cfma(D, W, sDot[1][l]);
                }
            }
            sAcc[w][lane] = D;
            sXp[w][lane] = xp;
            if (w == 1) {
                // sums over l: B = v0 dW + w0 dV, Re w0 conj(v0), Re conj(dW) dV
                double2 B = cmk(0, 0);
                double c0 = 0.0, ee = 0.0;
                if (lane < i) {
                    const double2 w0 = sRow[0][lane], v0 = sRow[1][lane], dw = sDot[0][lane], dv = sDot[1][lane];
                    B = cadd(cmul(v0, dw), cmul(w0, dv));
                    c0 = w0.x * v0.x + w0.y * v0.y;
                    ee = dw.x * dv.x + dw.y * dv.y;
                }
                const double b0 = wave_sum_dpp(B.x), b1 = wave_sum_dpp(B.y);
                c0 = wave_sum_dpp(c0);
                ee = wave_sum_dpp(ee);
                if (lane == 0) { sB[0] = b0; sB[1] = b1; sB[2] = c0; sB[3] = ee; }
            }
        }
        __syncthreads();
        double2 D = cmk(0, 0), xs = cmk(0, 0);
        if (w == 0) {
#pragma unroll
            for (int k = 1; k < PN_WAVES; ++k) {
                D = cadd(D, sAcc[k][lane]);
                xs = cadd(xs, sXp[k][lane]);
            }
        }
        // ---------------- owners, late: the partial products of their rows, of row s0, x^H A x
        {
            const bool ok = grow >= s0 && grow < n;
            double2 acc = cmk(0, 0);
            for (int sb = 0; sb < a.nbk + 1; sb += LW * PL) {
                int off[PL];
                double2 v[PL];
#pragma unroll
                for (int u = 0; u < PL; ++u) {
                    const int s = sb + w + LW * u;
                    off[u] = (w < LW && ok && s < a.nbk + 1) ? L.p + par * L.ps + ((wg * (a.nbk + 1) + s) * 64 + lane) * 2 : -1;
                }
                if (sb == 0 && w == LW && lane < a.nbk + 1)
                    off[0] = L.p + par * L.ps + ((((s0 >> 6) - a.tc0) * (a.nbk + 1) + lane) * 64 + (s0 & 63)) * 2;
                if (sb == 0 && w == LW + 1) {
#pragma unroll
                    for (int u = 0; u < PL; ++u)
                        if (2 * (lane + 64 * u) < G) off[u] = L.q + par * L.qs + 2 * (lane + 64 * u);
                }
                if (!pn_poll<PL>(rm, off, tag, v, a.err)) return;
#pragma unroll
                for (int u = 0; u < PL; ++u) acc = cadd(acc, v[u]);
            }
            if (w < LW) {
                sRS[0][w][lane] = acc;
            } else {
                const double y0 = wave_sum_dpp(acc.x), y1 = wave_sum_dpp(acc.y);
                if (lane == 0) {
                    if (w == LW) { sC[0] = y0; sC[1] = y1; }
                    else sQ = y0 + y1;
                }
            }
        }
        __syncthreads();
        if (w == 0) {
            double2 y = cmk(0, 0);
#pragma unroll
            for (int k = 0; k < LW; ++k) y = cadd(y, sRS[0][k][lane]);
            y = cmul(tau, csub(cadd(cmul(sc, csub(y, D)), as0), xs));
            const double2 scB = cmul(sc, cmk(sB[0], sB[1]));
            const double s2 = cabs2(sc);
            const double vav = s2 * sQ + 2.0 * (sc.x * sS[0][1] + sc.y * sS[0][2]) + a11;
            const double tt = sB[2] + scB.x + s2 * sB[3];          // Re (W^H v)^H (V^H v)
            al2 = -0.5 * cabs2(tau) * (vav - 2.0 * tt);
            const double2 c0 = cmk(2.0 * sB[2] + scB.x, scB.y);    // row s0 of V t1 + W t2
            const double2 ys0 = cmul(tau, csub(cadd(cmul(sc, cmk(sC[0], sC[1])), cmk(a11, 0.0)), c0));
            const double2 ws0 = cmk(ys0.x + al2, ys0.y);
            const bool in = grow >= s0 && grow < n;
            double2 v = pn_sel(grow == s0, cmk(1.0, 0.0), cmul(sc, xown));
            v = pn_sel(in, v, cmk(0, 0));
            const double2 wv = pn_sel(in, cadd(y, cscale(v, al2)), cmk(0, 0));
            if (more) {
                double2 x = csub(csub(as0, xs), cadd(cmul(v, cconj(ws0)), wv));
                if (grow == s0) x.y = 0.0;
                x = cscale(x, up);
                xown = x;
                if (in) pn_post(rm, L.x + (par ^ 1) * L.xs + (wg * 64 + lane) * 2, x, tag + 1);
                sX[lane] = pn_sel(in && grow > s0 + 1, x, cmk(0, 0));
            }
            sV[i][lane] = v;
            sW[i][lane] = wv;
            if (grow >= j0 && grow < n) {
                a.Vp[(grow - j0) + (int64_t)i * m] = v;
                a.Wp[(grow - j0) + (int64_t)i * m] = wv;
            }
            if (wg == 0) {
                if (lane == 0) {
                    a.d[c] = sC[4] * down;
                    a.e[c] = beta * down;
                    a.tau[c] = tau;
                }
                if (lane < i) a.G[lane + (int64_t)i * 64] = cadd(cconj(sRow[1][lane]), cmul(sc, sDot[1][lane]));
            }
        }
        if (!more) break;
        __syncthreads();
        // ---------------- for the next column: W^H x, V^H x of these rows (wave w:
        // l = w, w + 8, ...), its sums, and row s0 + 1 of W, V
        {
            // value 2 u + which of the eight: l = w + 8 u, W (0) or V (1)
            const double2 x = sX[lane];
            double2 p[4];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int l = w + PN_WAVES * u, l2 = l + 2 * PN_WAVES;
                const double2 zero = cmk(0, 0);
                const double2 w0 = l <= i ? cmulc(sW[l][lane], x) : zero, v0 = l <= i ? cmulc(sV[l][lane], x) : zero;
                const double2 w1 = l2 <= i ? cmulc(sW[l2][lane], x) : zero, v1 = l2 <= i ? cmulc(sV[l2][lane], x) : zero;
                p[2 * u] = pn_swap32(w0, w1);
                p[2 * u + 1] = pn_swap32(v0, v1);
            }
            const double2 sum = pn_sum8(p, lane);
            const int q = pn_col8(lane), l = w + PN_WAVES * (q >> 1), which = q & 1;
            if ((lane & 7) == 0 && l <= i)
                pn_post(rm, L.dot + (par ^ 1) * L.ds + ((wg * 2 + which) * PN_B + l) * 2, sum, tag + 1);
            if (w == 1) post_sums(s0, x, as1);
            if (w == 2 && ((s0 + 1) >> 6) - a.tc0 == wg) {
                const int lr = lane & 31, wh = lane >> 5;
                const double2 v = wh ? sV[lr][(s0 + 1) & 63] : sW[lr][(s0 + 1) & 63];
                if (lr <= i) pn_post(rm, L.row + (par ^ 1) * L.rs + lane * 2, v, tag + 1);
            }
        }
        as0 = as1;
        a11 = a11n;
    }
}

// dst = src (vec 16-byte vectors of the tiled storage, whose padding is zero) and
// the largest component's size into *big (zeroed before), NaNs left out.
template <typename V>
__global__ __launch_bounds__(256) void k_copy_max(int64_t vec, const V* __restrict__ src, V* __restrict__ dst,
                                                  unsigned long long* __restrict__ big)
{
    __shared__ double sm[4];
    double m = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < vec; i += (int64_t)gridDim.x * 256) {
        const V x = src[i];
        dst[i] = x;
        m = fmax(m, fmax(fabs((double)x.x), fabs((double)x.y)));
        if constexpr (sizeof(x.x) == 4) m = fmax(m, fmax(fabs((double)x.z), fabs((double)x.w)));
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3]));
        // sizes of doubles order as their bits do
        if (m > 0.0) atomicMax(big, (unsigned long long)__double_as_longlong(m));
    }
}

extern "C" hipError_t bse_launch_copy_max(hipStream_t st, int fp32, int n, const void* src, void* dst, double* big)
{
    const int64_t vec = tiled_elems(n) / (fp32 ? 2 : 1);
    const dim3 g((unsigned)std::min<int64_t>(ceil_div64(vec, 256), 2048));
    if (fp32)
        hipLaunchKernelGGL(k_copy_max<float4>, g, dim3(256), 0, st, vec, (const float4*)src, (float4*)dst,
                           (unsigned long long*)big);
    else
        hipLaunchKernelGGL(k_copy_max<double2>, g, dim3(256), 0, st, vec, (const double2*)src, (double2*)dst,
                           (unsigned long long*)big);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Host side.  A panel is taken here when its tiles number at most four per
// workgroup and its tile rows (the owners) at most 63: a wave polls a row's
// partials, and the sums of all owners, one per lane.
// ---------------------------------------------------------------------------
struct PanelPlan {
    bool ok;
    int per, grid, tc0, nbk, ntl;
    int64_t words;
};
static PanelPlan panel_plan(int n, int j0, int nwg)
{
    PanelPlan p{};
    if (j0 + 1 >= n || nwg < 1) return p;
    p.tc0 = (j0 + 1) >> 6;
    p.nbk = tile_count(n) - p.tc0;
    const int64_t ntl = (int64_t)p.nbk * (p.nbk + 1) / 2;
    nwg = std::min(nwg, 512);                       // (x^H A x words: four pairs a lane)
    if (p.nbk > 63 || ntl > (int64_t)PN_MAXTILES * nwg) return p;
    p.ntl = (int)ntl;
    p.per = (int)ceil_div64(ntl, nwg);
    p.grid = (int)std::max<int64_t>(ceil_div64(ntl, p.per), p.nbk);
    if (p.grid > nwg) return p;
    p.words = panel_msg(p.nbk, p.grid).total;
    p.ok = p.words * 16 < ((int64_t)1 << 31);
    return p;
}

// Workgroups of the panel kernel the device holds at once (0: none).
extern "C" int bse_panel_workgroups(int device, int fp32)
{
    const void* k[4];
    if (fp32) {
        k[0] = (const void*)k_trd_panel<float2, 1>; k[1] = (const void*)k_trd_panel<float2, 2>;
        k[2] = (const void*)k_trd_panel<float2, 3>; k[3] = (const void*)k_trd_panel<float2, 4>;
    } else {
        k[0] = (const void*)k_trd_panel<double2, 1>; k[1] = (const void*)k_trd_panel<double2, 2>;
        k[2] = (const void*)k_trd_panel<double2, 3>; k[3] = (const void*)k_trd_panel<double2, 4>;
    }
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    for (const void* f : k) {
        int per = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, PN_THREADS, 0) != hipSuccess || per < 1) return 0;
    }
    return ncu;
}

// First panel (column of it) that the panel kernel takes, n when none does.
extern "C" int bse_panel_first(int n, int nwg)
{
    for (int j0 = 0; j0 < n - 1; j0 += PN_B)
        if (panel_plan(n, j0, nwg).ok) return j0;
    return n;
}

// Workgroups without tile rows of their own (no owners) that would wait for no
// row of x in some column, over all panels: none, or the reuse rule is broken.
extern "C" int64_t bse_panel_unawaited(int n, int nwg)
{
    int64_t bad = 0;
    for (int j0 = bse_panel_first(n, nwg); j0 < n - 1; j0 += PN_B) {
        const PanelPlan p = panel_plan(n, j0, nwg);
        if (!p.ok) return -1;
        for (int wg = p.nbk; wg < p.grid; ++wg)
            for (int s0 = j0 + 1; s0 <= std::min(j0 + PN_B, n - 1); ++s0) {
                bool waits = false;
                for (int t = wg; t < p.ntl && !waits; t += p.grid) {
                    int I, J;
                    tri_tile(t, I, J);
                    for (int r = 0; r < 64 && !waits; ++r)
                        waits = pn_awaits(64 * (p.tc0 + I) + r, s0, n) || pn_awaits(64 * (p.tc0 + J) + r, s0, n);
                }
                bad += waits ? 0 : 1;
            }
    }
    return bad;
}

// 16-byte elements of the messages and of the panels' meeting counters.
extern "C" int64_t bse_panel_workspace(int n, int nwg)
{
    const int first = bse_panel_first(n, nwg);
    int64_t words = 0;
    for (int j0 = first; j0 < n - 1; j0 += PN_B) words = std::max(words, panel_plan(n, j0, nwg).words);
    return words > 0 ? words + ceil_div64(n, PN_B) / 4 + 2 : 0;
}

// The panel at j0 (a multiple of 32, >= bse_panel_first).  ws: zeroed before
// the first panel of a reduction; err: zeroed, set as in resident.hpp; big: from
// bse_launch_copy_max; refuse: the last panel is refused (rs_refuse).
extern "C" hipError_t bse_launch_panel(hipStream_t st, int device, int fp32, int n, int j0, int nwg, const void* A,
                                       double2* Vp, double2* Wp, double2* alpha2, double2* G, double* d, double* e,
                                       double2* tau, double2* ws, int64_t ws_el, int* err, const double* big,
                                       int refuse)
{
    const PanelPlan p = panel_plan(n, j0, nwg);
    const int64_t cnt = ceil_div64(n, PN_B) / 4 + 2;
    if (!p.ok || p.words + cnt > ws_el) return hipErrorInvalidValue;
    unsigned* meet = reinterpret_cast<unsigned*>(ws + (ws_el - cnt)) + j0 / PN_B;
    if (refuse && j0 + PN_B >= n - 1) {
        const hipError_t rc = rs_refuse(st, meet);
        if (rc != hipSuccess) return rc;
    }
    const PanelArgs args{n, j0, std::min(PN_B, n - 1 - j0), p.tc0, p.nbk, p.ntl, A, Vp, Wp, alpha2, G,
                         d, e, tau, reinterpret_cast<bse_i4v*>(ws), meet, err, big};
    return resident_launch(device, st, [&]() -> hipError_t {
        const dim3 g((unsigned)p.grid), t(PN_THREADS);
#define PN_GO(TT, NT) hipLaunchKernelGGL((k_trd_panel<TT, NT>), g, t, 0, st, args)
#define PN_PICK(TT)                                                                                     \
    switch (p.per) {                                                                                    \
    case 1: PN_GO(TT, 1); break;                                                                        \
    case 2: PN_GO(TT, 2); break;                                                                        \
    case 3: PN_GO(TT, 3); break;                                                                        \
    default: PN_GO(TT, 4); break;                                                                       \
    }
        if (fp32) { PN_PICK(float2) } else { PN_PICK(double2) }
#undef PN_PICK
#undef PN_GO
        return hipGetLastError();
    });
}
