// lsmp_adv_tile.hip -- the CRWENO5 line solve of an advection pass
// (level_set_rk3_solver.f90:1-221: crweno_flux_split :347-414, the WENO-JS
// boundary faces :288-345, the RK stage :16-88) for many lines of 34..513
// cells, or lines of 514..1025 cells, through LDS tiles.
//
// A workgroup of TW waves takes TL lines with neighbouring indices (for y and
// z lines, neighbouring in memory): 4 waves and 8 lines for lines of up to 513
// cells, 8 waves and 4 lines (one system per wave, 16 rows per lane) for lines
// of 514..1025 cells, which come in fewer lines per pass.
// (1) Every thread loads cells of the TL lines, coalesced -- along the line
// for x lines, across the lines for y and z lines -- and stores their split
// fluxes g and f in two LDS tiles, one row of slots per line, f in reversed
// cell order; then 4 TL threads form the WENO-JS boundary faces of the TL
// lines' two systems.  Reversing a line
// mirrors the stencil and exchanges A and C, which is what an f row does to a
// g row, so the f system of a line is the g system of its reversed f fluxes,
// with the reversed orientation's sign on the flux differences.  (2) Each
// wave solves 2 TL / TW of the TL lines' 2 TL systems (g, and f reversed, both
// with the g rows), with SL lanes per system: lane s eliminates its
// K = ceil((n-1)/SL) rows with the two neighbouring interface values as
// parameters, X_i = p_i + q_i L + r_i R; the interface rows form a tridiagonal
// system across the SL lanes, solved by parallel cyclic reduction; then each lane
// back-substitutes its rows, reading its stencils from the tiles.  The flux
// differences of the g and f systems go back into the tiles, over the line's own
// fluxes, which only its wave reads.
// (3) Every thread forms the RHS or the RK stage of cells of the TL lines and
// stores them, coalesced as in (1).  Nothing goes to scratch memory: the HBM
// traffic is the pass's own fields.  In MODE 2 the in-place update of phi is
// safe: the stencils run along the lines, and a workgroup reads and writes
// only its own lines.
//
// Bound by issue and LDS together (256^3 FP64: 57% and 39% of the time), so a
// system is as narrow as four rows a lane allow: both of a line in one wave up
// to 129 cells (128^3 advection 443 -> 352 us, FP32 265 -> 233), a wave per system up
// to 257, where half the lanes with eight rows take 144 VGPRs instead of 104
// (256^3 2256 against 2305, FP32 1290 against 1366).
//
// Same rows as the reference's (an f row is the g row of the mirrored stencil
// with A and C exchanged); the solve differs from one Thomas sweep only in
// rounding.
#include <hip/hip_runtime.h>

#include "lsmp_device.h"
#include "lsmp_internal.h"

namespace lsmp {

namespace {

// LDS slot of cell q (0-based) of a line: a pad slot after every 8 cells, so
// that the lanes of a system, K cells apart, spread over the banks
LSMP_DEV int tpos(int q) { return q + (q >> 3); }

}  // namespace

// slots per tile row for lines of n cells (odd: the y and z loads write TL
// rows at once)
static int adv_tile_row_slots(int n)
{
    const int rs = n + ((n - 1) >> 3) + 1;
    return rs | 1;
}

// TW waves per workgroup, TL lines per workgroup: 2 TL / TW systems per wave
template <typename T, int MODE, int STAGE, int KR, int SL, bool TUBE, int TL, int TW>
__global__ __launch_bounds__(TW * 64) void k_adv_tile(T *phi, const T *__restrict__ vel, T *R, T *L1, T *L2,
                                                       int nlines, int n, int lw, long ostride, long istride,
                                                       long estride, T dd, T dt, const int *__restrict__ lines,
                                                       TubeMask tm, int rs)
{
    static_assert((2 * TL) % TW == 0 && (TL & (TL - 1)) == 0, "whole systems per wave, TL a power of two");
    extern __shared__ __align__(16) unsigned char adv_lds[];
    T *tg = reinterpret_cast<T *>(adv_lds);   // TL rows of rs slots: g fluxes, then g flux differences
    T *tf = tg + TL * rs;                     // the same for f, cells in reversed order
    __shared__ size_t sbase[TL];
    __shared__ int2 stube[TL];   // i, j of a z line (the tube's lines are along z in the stage pass)
    // boundary faces: [line][0] g face 0, [1] g face n, [2] f face n, [3] f face 0
    // (the f system's start and end in its reversed order)
    __shared__ T sbc[TL][4];
    const int L0 = xcd_block() * TL;
    const int tid = threadIdx.x;
    if (tid < TL) {
        // lines past the end shadow the last one and store nothing
        const int Lc = min(L0 + tid, nlines - 1);
        const int bl = lines ? lines[Lc] : Lc;
        sbase[tid] = (size_t)(bl / lw) * (size_t)ostride + (size_t)(bl % lw) * (size_t)istride;
        if (MODE == 2 && TUBE) stube[tid] = make_int2(bl % lw, bl / lw);
    }
    __syncthreads();
    const int ne = TL * n;
    const bool along = estride == 1;   // x lines: cells of a line are contiguous
    // cell e of the tile: line l, cell q (the product with 1 / n is exact enough
    // for the at most 8 x 1,025 cells)
    const float inv_n = 1.0f / (float)n;
    auto cell_of = [&](int e, int &l, int &q) {
        if (along) {
            l = (int)(((float)e + 0.5f) * inv_n);
            q = e - l * n;
        } else {
            q = e / TL;
            l = e - q * TL;
        }
    };
    // (1) split fluxes of the TL lines into the tiles, the loads of U cells in flight
    constexpr int U = 4, NT = TW * 64;
    for (int e0 = tid; e0 < ne; e0 += U * NT) {
        T pv[U], uv[U];
        int at[U], rt[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            int l, q;
            cell_of(min(e0 + i * NT, ne - 1), l, q);
            const size_t a = sbase[l] + (size_t)q * (size_t)estride;
            pv[i] = phi[a];
            uv[i] = vel[a];
            at[i] = l * rs + tpos(q);
            rt[i] = l * rs + tpos(n - 1 - q);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {   // past the end: the last cell once more
            T g, f;
            flux_split(pv[i], uv[i], g, f);
            tg[at[i]] = g;
            tf[rt[i]] = f;
        }
    }
    __syncthreads();
    if (tid < 4 * TL) {
        // WENO-JS closures (crweno_flux_split :383-384, 409-410) on the clamped
        // cells in natural order: g on cells -2..2 or n-2..n+2, f on -1..3 or
        // n-1..n+3 (1-based)
        const int l = tid >> 2, w = tid & 3;
        const bool fs = w >= 2, right = (w == 1) || (w == 2);
        T v[5];
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            const int q = clampi((right ? n - 2 : -2) + (fs ? 1 : 0) + t - 1, 0, n - 1);
            v[t] = fs ? tf[l * rs + tpos(n - 1 - q)] : tg[l * rs + tpos(q)];
        }
        sbc[l][w] = fs ? wenojs_f(v[0], v[1], v[2], v[3], v[4]) : wenojs_g(v[0], v[1], v[2], v[3], v[4]);
    }
    __syncthreads();

    // (2) one system at a time per wave, or both of a line (SL = 32)
    const int wave = tid >> 6, lane = tid & 63;
    const int s = lane & (SL - 1);
    const int N = n - 1, K = (N + SL - 1) / SL;
    const int lo = s * K + 1;
    const bool active = lo <= N;
    const bool last = (s + 1) * K >= N;
    const int hi = last ? N : (s + 1) * K - 1;
    const int nrow = active ? hi - lo + 1 : 0;
    const bool irow = active && !last;
    const bool next_last = (s + 2) * K >= N;
    for (int job = wave; job < TL * (SL / 32); job += TW) {
        const int l = SL == 32 ? job : job >> 1;
        const bool isf = SL == 32 ? lane >= 32 : job & 1;
        const T sdd = isf ? -(T(1) / dd) : T(1) / dd;
        T *tile = (isf ? tf : tg) + l * rs;
        auto flux = [&](int c) { return tile[tpos(clampi(c - 1, 0, n - 1))]; };   // cell c = 1..n, clamped
        // fl[t] = flux at cell lo - 2 + t: the stencils of rows lo .. lo + KR
        T fl[KR + 6];
#pragma unroll
        for (int t = 0; t < KR + 6; ++t) fl[t] = flux(lo - 2 + t);
        auto coeffs = [&](int j, T &A, T &B, T &C, T &S) {   // row lo + j
            crweno_row<T, TUBE>(fl[j], fl[j + 1], fl[j + 2], fl[j + 3], fl[j + 4], A, B, C, S);
        };
        // boundary faces at the system's start and end
        const T bc0 = sbc[l][isf ? 2 : 0], bcN = sbc[l][isf ? 3 : 1];
        // local sweep: X_i = d'_i + e'_i L - c'_i X_{i+1}; the row after the
        // last (j == nrow) is the interface row of a lane that has one
        T cp[KR], dp[KR], ep[KR];
        T A = T(0), B = T(1), C = T(0), S = T(0);   // interface row
#pragma unroll
        for (int j = 0; j < KR; ++j) {
            if (j < nrow || (irow && j == nrow)) {
                T a_, b_, c_, s_;
                coeffs(j, a_, b_, c_, s_);
                if (j == nrow) {
                    A = a_;
                    B = b_;
                    C = c_;
                    S = s_;
                } else if (j == 0) {
                    const T r = rcp_pos(b_);
                    cp[j] = c_ * r;
                    dp[j] = s_ * r;
                    ep[j] = -a_ * r;
                } else {
                    const T r = rcp_pos(b_ - a_ * cp[j - 1]);
                    cp[j] = c_ * r;
                    dp[j] = (s_ - a_ * dp[j - 1]) * r;
                    ep[j] = -a_ * ep[j - 1] * r;
                }
            }
        }
        // (p, q, r) of the last row and of the first
        T ph = T(0), qh = T(1), rh = T(0), pl = T(0), ql = T(0), rl = T(1);
#pragma unroll
        for (int j = KR - 1; j >= 0; --j) {
            if (j < nrow) {
                if (j == nrow - 1) {
                    pl = dp[j];
                    ql = ep[j];
                    rl = -cp[j];
                    ph = pl;
                    qh = ql;
                    rh = rl;
                } else {
                    pl = dp[j] - cp[j] * pl;
                    ql = ep[j] - cp[j] * ql;
                    rl = -cp[j] * rl;
                }
            }
        }
        // interface row (s+1)K: X_hi of this lane and X_lo of the next enter it
        T ra = T(0), rb = T(1), rc = T(0), rd = T(0);
        const T npl = __shfl(pl, (lane + 1) & 63, 64), nql = __shfl(ql, (lane + 1) & 63, 64);
        const T nrl = __shfl(rl, (lane + 1) & 63, 64), nbcN = bcN;
        if (irow) {
            ra = A * qh;
            rb = B + A * rh + C * nql;
            rc = C * nrl;
            rd = S - A * ph - C * npl;
            if (s == 0) {
                rd = rd - ra * bc0;
                ra = T(0);
            }
            if (next_last) {
                rd = rd - rc * nbcN;
                rc = T(0);
            }
        }
        const T Xb = adv_exact<T, TUBE>() ? pcr_solve_full<SL, false>(ra, rb, rc, rd) : pcr_solve<SL>(ra, rb, rc, rd);
        const T Xprev = __shfl(Xb, (lane - 1) & 63, 64);
        const T Lv = s == 0 ? bc0 : Xprev;
        const T Rv = last ? bcN : Xb;

        // back-substitution: the flux differences of cells lo .. hi + 1 of this
        // system go over the line's fluxes (every lane of the wave has read its
        // stencils above)
        T x = Rv;
#pragma unroll
        for (int j = KR - 1; j >= 0; --j) {
            if (j < nrow) {
                const T xn = dp[j] + ep[j] * Lv - cp[j] * x;
                tile[tpos(lo + j)] = (xn - x) * sdd;   // cell lo + j + 1
                x = xn;
            }
        }
        if (active) tile[tpos(lo - 1)] = (Lv - x) * sdd;   // cell lo
    }
    __syncthreads();

    // (3) the RHS or the RK stage of every cell of the TL lines
    constexpr int U3 = 4;
    for (int e0 = tid; e0 < ne; e0 += U3 * NT) {
        T t1[U3], t2[U3], Rv[U3], Pv[U3], l1[U3], l2[U3];
        size_t at[U3];
        bool on[U3];
#pragma unroll
        for (int i = 0; i < U3; ++i) {
            int l, q;
            cell_of(min(e0 + i * NT, ne - 1), l, q);
            const size_t a = sbase[l] + (size_t)q * (size_t)estride;
            at[i] = a;
            on[i] = e0 + i * NT < ne && L0 + l < nlines;
            if (MODE == 2 && TUBE) on[i] = on[i] && tm.in(stube[l].x, stube[l].y, q);
            if (MODE != 0) Rv[i] = R[a];
            if (MODE == 2) {
                Pv[i] = phi[a];
                if (STAGE > 1) l1[i] = L1[a];
                if (STAGE > 2) l2[i] = L2[a];
            }
            t1[i] = tg[l * rs + tpos(q)];
            t2[i] = tf[l * rs + tpos(n - 1 - q)];
        }
#pragma unroll
        for (int i = 0; i < U3; ++i) {
            if (!on[i]) continue;
            const size_t a = at[i];
            if (MODE == 0) {
                R[a] = t1[i] + t2[i];
                continue;
            }
            const T r = (Rv[i] + t1[i]) + t2[i];
            if (MODE == 1) {
                R[a] = r;
            } else if (STAGE == 1) {
                L1[a] = r;
                phi[a] = Pv[i] + r * dt;
            } else if (STAGE == 2) {
                L2[a] = r;
                phi[a] = Pv[i] + fma(T(-3), l1[i], r) / T(4) * dt;
            } else {
                phi[a] = Pv[i] + (-l1[i] - l2[i] + T(8) * r) / T(12) * dt;
            }
        }
    }
}

template <typename T>
void launch_adv_tile(hipStream_t st, int mode, int stage, T *phi, const T *vel, T *R, T *L1, T *L2, int nlines, int n,
                     int lw, long ostride, long istride, long estride, T dd, T dt, const int *lines,
                     const TubeMask &tm)
{
    const int rs = adv_tile_row_slots(n);
    const bool tube = lines != nullptr;   // the narrow band's lines: the stage pass has the mask tm, FP32 adv_exact
    const bool h4 = n <= 32 * 4 + 1 && !(tube && sizeof(T) == 4);   // half a wave per system and four rows a lane suffice
    const bool k4 = n <= 64 * 4 + 1;   // else a wave per system and four, or eight (up to 513 cells)
    // lines of 514..1025 cells: sixteen rows per lane, four lines per workgroup
    const bool k16 = n > 64 * 8 + 1;
    const int tl = k16 ? 4 : 8;
    const size_t lds = 2 * (size_t)tl * rs * sizeof(T);
    const dim3 g((unsigned)((nlines + tl - 1) / tl)), b(k16 ? 8 * 64 : 4 * 64);
    // tiles of lines longer than 257 cells take more than 64 KiB of LDS (FP64)
#define LSMP_TILEK(M, S, KR, SL, TB, TLV, TWV)                                                                 \
    do {                                                                                                       \
        if (lds > 65536)                                                                                       \
            (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_adv_tile<T, M, S, KR, SL, TB, TLV, TWV>), \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                   \
        hipLaunchKernelGGL((k_adv_tile<T, M, S, KR, SL, TB, TLV, TWV>), g, b, lds, st, phi, vel, R, L1, L2,    \
                           nlines, n, lw, ostride, istride, estride, dd, dt, lines, tm, rs);                   \
    } while (0)
#define LSMP_TILET(M, S, TB)                                                                                   \
    do {                                                                                                       \
        if (k16) LSMP_TILEK(M, S, 16, 64, (TB && M != 2), 4, 8);   /* (its stage pass has no mask) */            \
        else if (h4) LSMP_TILEK(M, S, 4, 32, TB, 8, 4);                                                        \
        else if (k4) LSMP_TILEK(M, S, 4, 64, TB, 8, 4);                                                        \
        else LSMP_TILEK(M, S, 8, 64, TB, 8, 4);                                                                \
    } while (0)
#define LSMP_TILE(M, S)                                                                                        \
    do {                                                                                                       \
        if constexpr (M == 2 || adv_exact<T, true>()) {                                                        \
            if (tube) LSMP_TILET(M, S, true);                                                                  \
            else LSMP_TILET(M, S, false);                                                                      \
        } else {                                                                                               \
            LSMP_TILET(M, S, false);                                                                           \
        }                                                                                                      \
    } while (0)
    if (mode == 0) LSMP_TILE(0, 0);
    else if (mode == 1) LSMP_TILE(1, 1);
    else if (stage == 1) LSMP_TILE(2, 1);
    else if (stage == 2) LSMP_TILE(2, 2);
    else LSMP_TILE(2, 3);
#undef LSMP_TILE
#undef LSMP_TILET
#undef LSMP_TILEK
}

#define LSMP_INST_TILE(T)                                                                                      \
    template void launch_adv_tile<T>(hipStream_t, int, int, T *, const T *, T *, T *, T *, int, int, int, long, \
                                     long, long, T, T, const int *, const TubeMask &);
LSMP_INST_TILE(double)
LSMP_INST_TILE(float)
#undef LSMP_INST_TILE

}  // namespace lsmp
