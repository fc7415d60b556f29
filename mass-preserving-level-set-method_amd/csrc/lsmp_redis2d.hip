// lsmp_redis2d.hip -- the 2D reinitialisation stage (level_set_rk3_redis.f90:176-264
// with the gradient :266-369 and lambda :371-454 in their Disk/ and Vortex2D/
// forms: |grad| without z, lambda box 3x3 with centre weight 17,
// Disk/...redis.f90:357-361, 434-438; ls_funs ns_solver/others.f90:1-45).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lsmp_device.h"
#include "lsmp_internal.h"

namespace lsmp {

namespace {

// cells a wave finishes of its 64 columns: a WENO-HJ face takes its lanes l - 2
// to l + 3, the slopes of a cell two faces, lambda the cells beside it
constexpr int r2_margin(int btn) { return btn ? 4 : 3; }
constexpr int r2_cols(int btn) { return 64 - 2 * r2_margin(btn); }
constexpr int R2_WAVES = 8;   // waves of a workgroup, at most

}  // namespace

// A wave takes 64 columns and R rows and marches down them in registers: the
// column's second differences and the face below carry over from row to row, and
// the neighbours along x come by lane shifts, so the faces go nowhere through
// LDS.  The waves of a workgroup take successive rows; lambda's 3x3 box also needs
// the rows next to a wave's, whose sums over three columns go through LDS (the
// workgroup's first and last row are only there for that).  All loads are issued
// before the look at the stop flag.
//
// Tiles of 32 x 16 cells with phi, every face and s2, s3 in LDS and three
// barriers took 17.4 us per pseudo-step at 200^2, 25.8 at 613x389 and 64.0 (FP32
// 48.6) at 1,024^2, most of it indices, LDS traffic and waits; with each wave
// also computing the rows beside its own (no LDS at all) 13.9, 23.0 and 45.0
// (33.1); this form 13.1, 21.9 and 42.9 (32.8).  What is left at 200^2 is the
// launches (3.5-4 us each), at 1,024^2 the traffic of fields that no L2 keeps
// from one kernel to the next (2.6 TB/s).
template <typename T, int STAGE, int BTN, int R>
__global__ __launch_bounds__(64 * R2_WAVES) void k_redis2d(const T *__restrict__ phi, T *__restrict__ phi_out,
                                                           const T *__restrict__ phi0, const T *__restrict__ S0,
                                                           RedisArgs ra, unsigned long long *ctl, RedisStep step)
{
    extern __shared__ __align__(16) unsigned char r2_lds[];
    // per wave: the sums of s2 and s3 of its first and its last row
    T(*const box)[2][2][64] = reinterpret_cast<T(*)[2][2][64]>(r2_lds);
    constexpr int MARGIN = r2_margin(BTN);
    const int nx = ra.nx, ny = ra.ny;
    const T kx = (T)(2.0 * ra.inv12dx), ky = (T)(2.0 * ra.inv12dy);
    const T inv_w = (T)ra.inv_ls_wid, rdt = (T)ra.rdt;
    const int lane = threadIdx.x & 63, waves = (int)(blockDim.x >> 6);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // column strips fastest, in one grid dimension (no bound on nx or ny)
    const unsigned strips = (unsigned)(nx + r2_cols(BTN) - 1) / (unsigned)r2_cols(BTN);
    const int i = (int)(blockIdx.x % strips) * r2_cols(BTN) - MARGIN + lane;
    const int top = (int)(blockIdx.x / strips) * (waves * R - 2 * BTN) - BTN;   // the workgroup's rows
    const int ja = top + wave * R;                                   // the wave's
    const int jo0 = BTN ? std::max(top + 1, 0) : top, jo1 = std::min(top + waves * R - BTN, ny);   // rows to finish
    const bool own = lane >= MARGIN && lane < 64 - MARGIN && i < nx;
    const unsigned ic = (unsigned)clampi(i, 0, nx - 1);
    T pv[R + 6], sv[R], qv[R];
    // row ja - 3 + k of phi (ghosts: the boundary row)
#pragma unroll
    for (int k = 0; k < R + 6; ++k) pv[k] = (phi + (size_t)clampi(ja - 3 + k, 0, ny - 1) * nx)[ic];
#pragma unroll
    for (int k = 0; k < R; ++k) sv[k] = (S0 + (size_t)clampi(ja + k, 0, ny - 1) * nx)[ic];
    if (STAGE > 1)
#pragma unroll
        for (int k = 0; k < R; ++k) qv[k] = (phi0 + (size_t)clampi(ja + k, 0, ny - 1) * nx)[ic];
    // the pseudo-time loop has stopped
    if (STAGE == 1 ? redis_begin_step(ctl, step, blockIdx.x == 0) : ctl[1] != 0) return;
    double lerr = 0.0;
    T a[R], b[R], g[R], c2[R], c3[R], d[R];   // sums of s2 and s3, |grad|, s2, s3, delta
    bool any[R];                              // the row has a band cell
    // s(m-1), s(m), s(m+1) and the face m-1/2 for the first row m = ja
    T za = pv[1] - T(2) * pv[2] + pv[3], zb = pv[2] - T(2) * pv[3] + pv[4], zc = pv[3] - T(2) * pv[4] + pv[5];
    T zhb = hj_h(zb), ze = zc - T(2) * zb + za, zq;
    {
        const T z = pv[0] - T(2) * pv[1] + pv[2];   // s(m-2)
        T unused;
        weno_hj_face(z, za, zb, zc, hj_h(za), zhb, ze, zb - T(2) * za + z, unused, zq);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        a[r] = b[r] = g[r] = c2[r] = c3[r] = d[r] = T(0);
        any[r] = false;
        const int j = ja + r;
        if (j >= ny) continue;   // (row -1, which nothing uses, only carries the faces on)
        const T c = pv[r + 3], s0 = sv[r];
        // y: face j + 1/2
        const T zd = pv[r + 4] - T(2) * pv[r + 5] + pv[r + 6];
        const T zhc = hj_h(zc), zen = zd - T(2) * zc + zb;
        T zp, zqn;
        weno_hj_face(za, zb, zc, zd, zhb, zhc, zen, ze, zp, zqn);
        const T by = hj_base(c, pv[r + 4], zb, zc);
        const T yp = by + zp, ym = (by + ze) - zq;
        za = zb; zb = zc; zc = zd; zhb = zhc; ze = zen; zq = zqn;
        // x: face i + 1/2
        const T cp = from_right(c), s = from_left(c) - T(2) * c + cp;
        const T sm = from_left(s), sp = from_right(s), spp = from_right(sp);
        const T e2 = sp - T(2) * s + sm;
        T xP, xQ;
        weno_hj_face(sm, s, sp, spp, hj_h(s), hj_h(sp), spp - T(2) * sp + s, e2, xP, xQ);
        const T bx = hj_base(c, cp, s, sp);
        g[r] = godunov_sig(bx + xP, (bx + e2) - from_left(xQ), yp, ym, s0, kx, ky);
        if (BTN) {
            const bool band = in_band_x(c * inv_w);
            any[r] = __ballot(band) != 0;
            if (any[r]) {
                d[r] = band ? band_delta(c, inv_w) : T(0);
                const T s2 = d[r] * s0 * (g[r] - T(1)), s3 = g[r] * d[r] * d[r];
                const T l2 = from_left(s2), r2 = from_right(s2), l3 = from_left(s3), r3 = from_right(s3);
                a[r] = ((i <= 0 ? s2 : l2) + s2) + (i >= nx - 1 ? s2 : r2);   // ghosts: the boundary cell's
                b[r] = ((i <= 0 ? s3 : l3) + s3) + (i >= nx - 1 ? s3 : r3);
                c2[r] = s2;
                c3[r] = s3;
            }
        }
    }
    if (BTN) {
        box[wave][0][0][lane] = a[0];
        box[wave][0][1][lane] = b[0];
        if (R > 1) {
            box[wave][1][0][lane] = a[R - 1];
            box[wave][1][1][lane] = b[R - 1];
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = ja + r;
        if (j < jo0 || j >= jo1) continue;
        const T c = pv[r + 3], s0 = sv[r], p0 = STAGE > 1 ? qv[r] : c;
        T lam = T(0);
        if (BTN && any[r]) {
            T a1 = a[r], b1 = b[r], a3 = a[r], b3 = b[r];   // rows j - 1 and j + 1 (ghosts: the boundary row's)
            if (j > 0) {
                a1 = r > 0 ? a[r > 0 ? r - 1 : 0] : box[wave - 1][R > 1][0][lane];
                b1 = r > 0 ? b[r > 0 ? r - 1 : 0] : box[wave - 1][R > 1][1][lane];
            }
            if (j < ny - 1) {
                a3 = r < R - 1 ? a[r < R - 1 ? r + 1 : 0] : box[wave + 1][0][0][lane];
                b3 = r < R - 1 ? b[r < R - 1 ? r + 1 : 0] : box[wave + 1][0][1][lane];
            }
            const T la = T(17) * c2[r] + ((a1 + a[r]) + a3), lb = T(17) * c3[r] + ((b1 + b[r]) + b3);
            if (fabs(lb) > T(1.0e-12)) lam = la / lb * d[r];
        }
        const T pn = rk_stage<T, STAGE>(c, p0, (s0 - lam) * g[r] - s0, rdt);
        if (own) {
            (phi_out + (size_t)j * nx)[ic] = pn;
            if (STAGE == 3) lerr = fmax(lerr, (double)fabs(pn - p0));
        }
    }
    if (STAGE == 3) {
        const double m = block_max(lerr);
        if (threadIdx.x == 0 && m > 0.0) atomic_max_nonneg(ctl_slot(ctl, step, blockIdx.x), m);
    }
}

template <typename T>
void launch_redis2d(hipStream_t st, int stage, int btn, const T *phi, T *phi_out, const T *phi0, const T *S0,
                    const RedisArgs &ra, unsigned long long *ctl, RedisStep step)
{
    // Small grids want waves, larger ones less work at the seams (two faces and
    // two rows of a workgroup).  us per pseudo-step of waves x rows 4x1, 8x1, 8x2:
    // 100x60 11.9, 14.4, 16.3; 200^2 13.7, 13.5, 16.3; 256^2 15.9, 14.5, 16.7;
    // 512^2 28.9, 24.7, 24.0; 1,024^2 69.5, 53.1, 43.3.  Without lambda 4x1, 4x2:
    // 200^2 11.1, 12.0; 512^2 20.3, 18.6; 1,024^2 42.2, 36.0.
    const size_t n = (size_t)ra.nx * ra.ny;
    const int rows = n <= ((size_t)1 << 17) ? 1 : 2, waves = btn && n > ((size_t)1 << 14) ? 8 : 4;
    const int per = waves * rows - 2 * btn;   // rows a workgroup finishes
    const unsigned g = (unsigned)((ra.nx + r2_cols(btn) - 1) / r2_cols(btn)) * (unsigned)((ra.ny + per - 1) / per);
    const size_t lds = btn ? (size_t)waves * 256 * sizeof(T) : 0;
#define LSMP_R2(S, B)                                                                                              \
    {                                                                                                              \
        if (rows == 1)                                                                                             \
            hipLaunchKernelGGL((k_redis2d<T, S, B, 1>), dim3(g), dim3(64 * waves), lds, st, phi, phi_out, phi0, S0, ra,  \
                               ctl, step);                                                                         \
        else                                                                                                       \
            hipLaunchKernelGGL((k_redis2d<T, S, B, 2>), dim3(g), dim3(64 * waves), lds, st, phi, phi_out, phi0, S0, ra,  \
                               ctl, step);                                                                         \
    }
    if (btn) { if (stage == 1) LSMP_R2(1, 1) else if (stage == 2) LSMP_R2(2, 1) else LSMP_R2(3, 1) }
    else { if (stage == 1) LSMP_R2(1, 0) else if (stage == 2) LSMP_R2(2, 0) else LSMP_R2(3, 0) }
#undef LSMP_R2
}

template void launch_redis2d<double>(hipStream_t, int, int, const double *, double *, const double *, const double *,
                                     const RedisArgs &, unsigned long long *, RedisStep);
template void launch_redis2d<float>(hipStream_t, int, int, const float *, float *, const float *, const float *,
                                    const RedisArgs &, unsigned long long *, RedisStep);

}  // namespace lsmp
