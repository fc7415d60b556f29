// lsmp_redis_box.hip -- the 3D reinitialisation stage with lambda in the same
// launch (level_set_rk3_redis.f90:176-264 with the gradient :266-369, lambda
// :371-454 and ls_funs ns_solver/others.f90:1-45), for grids so small that the
// launches of the two-kernel stage cost more than the work that is done twice here.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lsmp_device.h"
#include "lsmp_internal.h"

namespace lsmp {

namespace {

// cells a wave finishes of its 64 columns: a WENO-HJ face takes its lanes l - 2
// to l + 3, the slopes of a cell two faces, lambda the cells beside it
constexpr int BOX_MARGIN = 4, BOX_COLS = 64 - 2 * BOX_MARGIN;

}  // namespace

// The waves of a workgroup take W successive rows of 64 columns and march through
// kc planes and the one before and after.  Along x the neighbours and faces come
// by lane shifts, along z they carry over in registers, the two faces of a cell
// along y are formed for it alone (the rows beside it are loaded).  lambda's box
// sums: three columns by lane shifts, three rows through LDS, three planes
// carried over; a plane is finished when the next one's sums are there.  A wave
// is bound by issue (0.5 us a plane in FP64) once the launch and the first loads
// are over (3.5 us); the band's list, its second launch and the stores and loads
// of |grad|, s2 and s3 between them are gone.
template <typename T, int STAGE, int W>
__global__ __launch_bounds__(64 * W) void k_redis3d_box(const T *__restrict__ phi, T *__restrict__ phi_out,
                                                        const T *__restrict__ phi0, const T *__restrict__ S0,
                                                        RedisArgs ra, unsigned long long *ctl, RedisStep step, int kc)
{
    __shared__ T box[2][W][2][64];   // by plane parity: the sums of s2 and s3 over three columns of each row
    const int nx = ra.nx, ny = ra.ny, nz = ra.nz;
    const T kx = (T)(2.0 * ra.inv12dx), ky = (T)(2.0 * ra.inv12dy), kz = (T)(2.0 * ra.inv12dz);
    const T inv_w = (T)ra.inv_ls_wid, rdt = (T)ra.rdt;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = (int)blockIdx.x * BOX_COLS - BOX_MARGIN + lane;
    const int j = (int)blockIdx.y * (W - 2) - 1 + wave;   // the first and the last wave's rows are the box's only
    const int jc = clampi(j, 0, ny - 1);
    const bool own = lane >= BOX_MARGIN && lane < 64 - BOX_MARGIN && i < nx && wave > 0 && wave < W - 1 && j < ny;
    const int k0 = (int)blockIdx.z * kc, k1 = std::min(k0 + kc, nz);   // planes to finish
    const int ps = std::max(k0 - 1, 0), pe = std::min(k1, nz - 1);     // planes to march, pe included
    const size_t plane = (size_t)nx * ny;
    const unsigned ic = (unsigned)clampi(i, 0, nx - 1);
    // row offsets of rows j - 3 .. j + 3 (ghosts: the boundary row)
    unsigned row[7];
#pragma unroll
    for (int r = 0; r < 7; ++r) row[r] = (unsigned)clampi(jc - 3 + r, 0, ny - 1) * (unsigned)nx + ic;
    auto zplane = [&](int k) { return (size_t)clampi(k, 0, nz - 1) * plane; };
    T zv[6];   // this row of planes ps - 3 .. ps + 2
#pragma unroll
    for (int r = 0; r < 6; ++r) zv[r] = (phi + zplane(ps - 3 + r))[row[3]];
    // of the plane at hand: the rows beside this one, the row three planes on, S0, phi0
    T yn[6], zn, sn, qn = T(0);
    auto fetch = [&](int p) {
        const T *const f = phi + (size_t)p * plane;
#pragma unroll
        for (int r = 0; r < 6; ++r) yn[r] = f[row[r < 3 ? r : r + 1]];
        zn = (phi + zplane(p + 3))[row[3]];
        sn = (S0 + (size_t)p * plane)[row[3]];
        if (STAGE > 1) qn = (phi0 + (size_t)p * plane)[row[3]];
    };
    fetch(ps);
    // the pseudo-time loop has stopped
    if (STAGE == 1 ? redis_begin_step(ctl, step, (blockIdx.x | blockIdx.y | blockIdx.z) == 0) : ctl[1] != 0) return;
    double lerr = 0.0;
    // s(p-1), s(p), s(p+1) along z and the face p-1/2 for the first plane p = ps
    T za = zv[1] - T(2) * zv[2] + zv[3], zb = zv[2] - T(2) * zv[3] + zv[4], zc = zv[3] - T(2) * zv[4] + zv[5];
    T zhb = hj_h(zb), ze = zc - T(2) * zb + za, zq;
    {
        const T z = zv[0] - T(2) * zv[1] + zv[2];
        T unused;
        weno_hj_face(z, za, zb, zc, hj_h(za), zhb, ze, zb - T(2) * za + z, unused, zq);
    }
    T w0 = zv[3], w1 = zv[4], w2 = zv[5];   // phi of planes p, p + 1, p + 2
    T a1 = T(0), b1 = T(0), a2 = T(0), b2 = T(0);   // sums over 3x3 cells of planes p - 2 and p - 1
    T pc = T(0), p0 = T(0), s01 = T(0), g1 = T(0), d1 = T(0), c2 = T(0), c3 = T(0);   // of plane p - 1
    bool any1 = false;                              // it has a band cell in this row
    auto finish = [&](int k, T a3, T b3) {   // plane k, with the sums of the plane after it
        T lam = T(0);
        if (any1) {
            const T la = T(51) * c2 + ((a1 + a2) + a3), lb = T(51) * c3 + ((b1 + b2) + b3);
            if (fabs(lb) > T(1.0e-12)) lam = la / lb * d1;
        }
        const T pn = rk_stage<T, STAGE>(pc, p0, (s01 - lam) * g1 - s01, rdt);
        if (own) {
            (phi_out + (size_t)k * plane)[row[3]] = pn;
            if (STAGE == 3) lerr = fmax(lerr, (double)fabs(pn - p0));
        }
    };
    for (int p = ps; p <= pe; ++p) {
        const T y0 = yn[0], y1 = yn[1], y2 = yn[2], y4 = yn[3], y5 = yn[4], y6 = yn[5], w3 = zn, s0 = sn, q0 = qn;
        if (p < pe) fetch(p + 1);
        const T c = w0;
        // z: face p + 1/2
        const T zd = w1 - T(2) * w2 + w3, zhc = hj_h(zc), zen = zd - T(2) * zc + zb;
        T zP, zqn;
        weno_hj_face(za, zb, zc, zd, zhb, zhc, zen, ze, zP, zqn);
        const T bz = hj_base(c, w1, zb, zc);
        const T zp = bz + zP, zm = (bz + ze) - zq;
        za = zb; zb = zc; zc = zd; zhb = zhc; ze = zen; zq = zqn;
        w0 = w1; w1 = w2; w2 = w3;
        // x: face i + 1/2
        const T cp = from_right(c), s = from_left(c) - T(2) * c + cp;
        const T sm = from_left(s), sp = from_right(s), spp = from_right(sp);
        const T e2 = sp - T(2) * s + sm;
        T xP, xQ, yp, ym;
        weno_hj_face(sm, s, sp, spp, hj_h(s), hj_h(sp), spp - T(2) * sp + s, e2, xP, xQ);
        const T bx = hj_base(c, cp, s, sp);
        // y: both faces
        weno_hj_cell(y0, y1, y2, c, y4, y5, y6, yp, ym);
        const T g = godunov_sig(bx + xP, (bx + e2) - from_left(xQ), yp, ym, zp, zm, s0, kx, ky, kz);
        const bool band = in_band_x(c * inv_w), any = __ballot(band) != 0;
        T del = T(0), s2 = T(0), s3 = T(0), a = T(0), b = T(0);
        if (any) {
            del = band ? band_delta(c, inv_w) : T(0);
            s2 = del * s0 * (g - T(1));
            s3 = g * del * del;
            const T l2 = from_left(s2), r2 = from_right(s2), l3 = from_left(s3), r3 = from_right(s3);
            a = ((i <= 0 ? s2 : l2) + s2) + (i >= nx - 1 ? s2 : r2);   // ghosts: the boundary cell's
            b = ((i <= 0 ? s3 : l3) + s3) + (i >= nx - 1 ? s3 : r3);
        }
        T(*const bp)[2][64] = box[p & 1];
        bp[wave][0][lane] = a;
        bp[wave][1][lane] = b;
        __syncthreads();   // (a plane's sums are overwritten two planes on, past the next barrier)
        const int up = j > 0 && wave > 0 ? wave - 1 : wave, dn = j < ny - 1 && wave < W - 1 ? wave + 1 : wave;
        const T a3 = (bp[up][0][lane] + a) + bp[dn][0][lane], b3 = (bp[up][1][lane] + b) + bp[dn][1][lane];
        if (p == 0) {   // plane -1 is the first one's ghost
            a2 = a3;
            b2 = b3;
        }
        if (p - 1 >= k0) finish(p - 1, a3, b3);
        a1 = a2; a2 = a3;
        b1 = b2; b2 = b3;
        pc = c; p0 = q0; s01 = s0; g1 = g; d1 = del; c2 = s2; c3 = s3;
        if (STAGE == 1) p0 = c;
        any1 = any;
    }
    if (pe < k1) finish(pe, a2, b2);   // the last plane's ghost
    if (STAGE == 3) {
        const double m = block_max(lerr);
        if (threadIdx.x == 0 && m > 0.0)
            atomic_max_nonneg(ctl_slot(ctl, step, (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x), m);
    }
}

// Waves a workgroup and planes a march for a grid that this stage suits: as many
// workgroups as the CUs take at once, else none (waves 0).  us per pseudo-step
// FP64 (FP32) against the two-kernel stage: 16^3 18.5 (16.1) against 33.5 (27.4),
// 32^3 22.9 (19.4), 34.2 (27.7); 48^3 30.3 (23.0), 38.0 (32.4); 56^3 37.2 (27.5),
// 40.2 (32.6); 110x40x40 36.5 (27.3), 39.9 (31.3); past the limits 64^3 58.9
// (42.3), 42.3 (35.7); 96^3 96.5 (58.9), 59.0 (46.4).
static void box_shape(int nx, int ny, int nz, int &waves, int &kc)
{
    const long strips = (nx + BOX_COLS - 1) / BOX_COLS;
    auto groups = [&](int w, int k) { return strips * ((ny + w - 3) / (w - 2)) * ((nz + k - 1) / k); };
    waves = 4;
    kc = 1;
    if (groups(4, 1) <= 256) return;
    kc = 2;
    if (groups(4, 2) <= 512) return;
    waves = 8;
    if (groups(8, 2) <= 256) return;
    kc = 3;
    if (groups(8, 3) <= 256) return;
    waves = 0;
}

bool redis3d_box_suits(int nx, int ny, int nz)
{
    int w, kc;
    box_shape(nx, ny, nz, w, kc);
    return w != 0;
}

template <typename T>
void launch_redis3d_box(hipStream_t st, int stage, const T *phi, T *phi_out, const T *phi0, const T *S0,
                        const RedisArgs &ra, unsigned long long *ctl, RedisStep step)
{
    int w, kc;
    box_shape(ra.nx, ra.ny, ra.nz, w, kc);
    const dim3 g((unsigned)((ra.nx + BOX_COLS - 1) / BOX_COLS), (unsigned)((ra.ny + w - 3) / (w - 2)),
                 (unsigned)((ra.nz + kc - 1) / kc));
#define LSMP_BOX(S, W) \
    hipLaunchKernelGGL((k_redis3d_box<T, S, W>), g, dim3(64 * W), 0, st, phi, phi_out, phi0, S0, ra, ctl, step, kc)
    if (w == 4) { if (stage == 1) LSMP_BOX(1, 4); else if (stage == 2) LSMP_BOX(2, 4); else LSMP_BOX(3, 4); }
    else { if (stage == 1) LSMP_BOX(1, 8); else if (stage == 2) LSMP_BOX(2, 8); else LSMP_BOX(3, 8); }
#undef LSMP_BOX
}

template void launch_redis3d_box<double>(hipStream_t, int, const double *, double *, const double *, const double *,
                                         const RedisArgs &, unsigned long long *, RedisStep);
template void launch_redis3d_box<float>(hipStream_t, int, const float *, float *, const float *, const float *,
                                        const RedisArgs &, unsigned long long *, RedisStep);

}  // namespace lsmp
