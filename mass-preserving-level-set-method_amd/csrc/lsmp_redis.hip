// lsmp_redis.hip -- the 3D reinitialisation stage (level_set_rk3_redis.f90:176-264
// with the gradient :266-369, lambda :371-454 and ls_funs ns_solver/others.f90:1-45),
// as two kernels per RK stage.
//
// k_redis3d updates every cell of the domain with lambda = 0.  That is the
// final value wherever delta = 0 (lambda is multiplied by delta), i.e. outside
// the band |phi| < ls_wid.  For the cells inside it, it also stores |grad|,
// s2 = delta S0 (|grad| - 1) and s3 = |grad| delta^2 in side fields and lists the cell: first in the workgroup's list in LDS,
// which the workgroup appends to the device list with one atomic at its end.
// k_redis3d_band then takes the listed cells, four lanes per cell over the
// whole device, and forms lambda from the sums of s2 and s3 over the band cells
// of the 3x3x3 box around each (centre weight 51) and the cell's final value
// with the same expression.  Off the band s2
// and s3 are zero, so the box sums take band cells only.
//
// k_redis3d: a workgroup of R3X*R3Y threads owns an interior tile in (i, j),
// one cell per thread, and marches over kc planes in k.  Each thread keeps
// its column phi(k..k+3) in registers; the current plane, with a 4-cell
// halo for the x and y stencils, goes to LDS.  The weighted third differences
// of D+ at m (P) and of D- at m+1 (Q) are built from the same four second
// differences s(m-1..m+2) (weno_hj_face), so each direction evaluates one
// face m+1/2 per cell.  z: each plane evaluates face p+1/2 and carries its Q,
// the second and fourth differences and h(s) to the next plane.  x and y:
// each thread evaluates the faces i+1/2 and j+1/2 of its cell and hands the Q
// terms to its neighbours through LDS; one wave (a different one from tile to
// tile) also evaluates the tile's first faces i0-1/2 and j0-1/2.  Two barriers
// per plane: the plane is in LDS, the Q terms are.
//
// Bound by FP64 issue: 205 VALU instructions per plane and thread, 158 of them
// FP64, are 100 us of the 143 us a 256^3 stage takes (2.05 ns per FP64
// instruction and SIMD measured alone; reading S0 as two bits a cell, a
// quarter of the traffic, changes nothing).  256^3, per pseudo-step of three
// stages and band passes, FP64 (FP32):
//   534 us (302)  indicators as expanded quadratic forms, a central part beside
//                 the face terms
//   506 us (271)  the forms of weno_hj_face
//   494 us (269)  no plane waits for its own loads or the last plane's stores
//                 (one wait a plane, before its stores)
//   480 us (250)  plane addresses in scalar registers, the LDS arrays on one row
//                 length, four planes a loop trip (no register moves): 106
//                 VGPRs instead of 122 (FP32 60 instead of 78: eight waves per
//                 SIMD).  A fifth FP64 wave per SIMD spills and runs slower.
//
// The RK stage is written in Shu-Osher form, algebraically identical to the
// reference's increments: phi1 = phi0 - dtau l(phi0);
// phi2 = 3/4 phi0 + 1/4 (phi1 - dtau l(phi1)); phi3 = 1/3 phi0 + 2/3 (phi2 - dtau l(phi2)).
// Stage 3 also reduces max |phi3 - phi0| (:46-62).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lsmp_device.h"
#include "lsmp_internal.h"

namespace lsmp {

namespace {

constexpr int NT = R3X * R3Y;                   // one thread per tile cell
constexpr int NHALO = P3X * P3Y - R3X * R3Y;    // LDS plane cells outside the tile
static_assert(NHALO <= 2 * NT, "at most two halo cells per thread");
static_assert(NT % 64 == 0, "whole waves");

// LDS position (row, col) of halo cell number t of the (R3X + 8) x (R3Y + 8)
// plane: four rows on top, four at the bottom, four columns left and right.
LSMP_DEV void halo_cell(int t, int &r, int &c)
{
    if (t < 4 * P3X) { r = t / P3X; c = t % P3X; }
    else if (t < 8 * P3X) { r = P3Y - 4 + (t - 4 * P3X) / P3X; c = (t - 4 * P3X) % P3X; }
    else { const int u = t - 8 * P3X; r = 4 + u / 8; c = u % 8 < 4 ? u % 8 : P3X - 8 + u % 8; }
}

// Element of a plane at a byte offset: the plane's address, the same in every
// lane, stays in scalar registers and the offset in one vector register (the
// empty statements, here and on the offsets in the plane loop, keep the
// compiler from adding the two into a vector pair per field: two registers
// and an addition per access).
template <typename T> using global_ptr = __attribute__((address_space(1))) T *;
template <typename T> LSMP_DEV T load_at(const T *plane_base, unsigned byte_off)
{
    unsigned long long b = (unsigned long long)plane_base;
    asm("" : "+s"(b));
    return *(global_ptr<const T>)((global_ptr<const char>)b + byte_off);
}
template <typename T> LSMP_DEV void store_at(T *plane_base, unsigned byte_off, T v)
{
    unsigned long long b = (unsigned long long)plane_base;
    asm("" : "+s"(b));
    *(global_ptr<T>)((global_ptr<char>)b + byte_off) = v;
}

// s_waitcnt vmcnt(0): the wave's loads and stores issued so far are done
LSMP_DEV void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

}  // namespace

// NB: the narrow band in FP32, which keeps the roundings of redis_exact (in FP64
// the tiles are all there is to it)
template <typename T, int STAGE, int BTN, bool NB>
__global__ __launch_bounds__(NT) void k_redis3d(const T *__restrict__ phi, T *__restrict__ phi_out,
                                                const T *__restrict__ phi0, const T *__restrict__ S0, RedisArgs ra,
                                                unsigned long long *ctl, const unsigned char *__restrict__ tiles,
                                                BandFields<T> bf, unsigned *__restrict__ blist,
                                                unsigned *__restrict__ bcount, int kc, RedisStep step)
{
    // rows of P3X slots: the plane with its halo, then Q of the x faces (row ty,
    // slot tx: of cell tx), then Q of the y faces (row ty: of cell ty).  One row
    // length for all three, so that a thread's places in them differ by constants.
    __shared__ T lds[(P3Y + R3Y + R3Y + 1) * P3X];
    constexpr int MX = P3Y * P3X, MY = (P3Y + R3Y) * P3X;
    static_assert(R3X + R3Y <= 64, "the first faces in one wave");
    // the workgroup's band cells, (plane - k0) * NT + thread, and their count
    __shared__ unsigned short lcell[BTN == 1 ? RKC * NT : 1];
    __shared__ unsigned lcount, lbase;
    static_assert(RKC * NT <= 65536, "local band-cell index in 16 bits");
    const int nx = ra.nx, ny = ra.ny, nz = ra.nz;
    // tiles in x-fastest order, renumbered so that each XCD takes a contiguous
    // run of them: the x and y halos of a tile are then mostly in its XCD's L2
    // (one grid dimension: the planes have no launch bound)
    const int gx = (nx + R3X - 1) / R3X, gy = (ny + R3Y - 1) / R3Y;
    const int tile_id = xcd_renumber((int)blockIdx.x, (int)gridDim.x);
    const int bx = tile_id % gx, by = (tile_id / gx) % gy, bz = tile_id / (gx * gy);
    // whether the pseudo-time loop has stopped: looked at once the run-up's loads
    // are on their way, before anything is written
    const bool lead = blockIdx.x == 0;
    auto stopped = [&]() { return STAGE == 1 ? redis_begin_step(ctl, step, lead) : ctl[1] != 0; };
    // narrow band: a workgroup with no cell of the tube keeps its cells.  Stage
    // 1 writes the step's output buffer and stage 2 the one stage 3 reads, so
    // both copy; stage 3 writes the buffer stage 1 filled, which holds them.
    if (tiles && !tiles[tile_id]) {
        if (stopped() || STAGE == 3) return;
        const int ci = bx * R3X + (int)threadIdx.x % R3X, cj = by * R3Y + (int)threadIdx.x / R3X;
        if (ci >= nx || cj >= ny) return;
        const size_t c0 = (size_t)cj * nx + ci, pl = (size_t)nx * ny;
        for (int k = bz * kc; k < min((bz + 1) * kc, nz); ++k)
            phi_out[(size_t)k * pl + c0] = phi[(size_t)k * pl + c0];
        return;
    }
    constexpr bool EXACT = redis_exact<T, NB>();
    // slopes are times 6 dx, ... until the Godunov sum (EXACT: scaled as they are formed)
    const T kx = EXACT ? (T)ra.inv12dx : (T)(2.0 * ra.inv12dx), ky = EXACT ? (T)ra.inv12dy : (T)(2.0 * ra.inv12dy),
            kz = EXACT ? (T)ra.inv12dz : (T)(2.0 * ra.inv12dz);
    auto face = [&](T sa, T sb, T sc, T sd, T hb, T hc, T e1, T e2, T &P, T &Q) {
        if constexpr (EXACT) weno_hj_face12(sa, sb, sc, sd, P, Q);
        else weno_hj_face(sa, sb, sc, sd, hb, hc, e1, e2, P, Q);
    };
    const T inv_w = (T)ra.inv_ls_wid, rdt = (T)ra.rdt;
    const int t = threadIdx.x;
    const int i0 = bx * R3X, j0 = by * R3Y, k0 = bz * kc;
    const int k1 = min(k0 + kc, nz);
    const int tx = t % R3X, ty = t / R3X;
    // cells past the domain edge hold the boundary cell (zero-gradient ghosts)
    const int gi = min(i0 + tx, nx - 1), gj = min(j0 + ty, ny - 1);
    const bool inner = i0 + tx < nx && j0 + ty < ny;
    const bool halo = t < NHALO, halo2 = t + NT < NHALO;
    int hr = 0, hc = 0, hr2 = 0, hc2 = 0;
    if (halo) halo_cell(t, hr, hc);
    if (halo2) halo_cell(t + NT, hr2, hc2);
    // byte offsets within a plane (a plane holds fewer than 2^28 cells); the
    // plane bases are uniform over the workgroup
    const size_t plane = (size_t)nx * ny;
    unsigned col = ((unsigned)gj * nx + gi) * (unsigned)sizeof(T);
    unsigned hcol = ((unsigned)clampi(j0 - 4 + hr, 0, ny - 1) * nx + clampi(i0 - 4 + hc, 0, nx - 1)) *
                          (unsigned)sizeof(T);
    unsigned hcol2 = ((unsigned)clampi(j0 - 4 + hr2, 0, ny - 1) * nx + clampi(i0 - 4 + hc2, 0, nx - 1)) *
                           (unsigned)sizeof(T);
    auto base = [&](const T *f, int p) { return f + (size_t)clampi(p, 0, nz - 1) * plane; };

    // the faces i+1/2 and j+1/2 read the LDS plane at the thread's own tile
    // position: past the domain edge it holds the boundary cell, as the halo
    // does.  One wave also takes the tile's first faces -- its lanes
    // 0..R3Y-1 the x face i0-1/2 of row u, lanes R3Y..R3Y+R3X-1 the y face
    // j0-1/2 of column u-R3Y (u the lane) -- a different wave from tile to
    // tile, so that the extra work spreads over the SIMDs of a CU
    const int fu = t - 64 * (tile_id % (NT / 64));
    const bool first_x = fu >= 0 && fu < R3Y, first_y = fu >= R3Y && fu < R3Y + R3X;
    int f_off = first_x ? (fu + 4) * P3X + 1 : (first_y ? P3X + 4 + (fu - R3Y) : 0);
    int f_dst = first_x ? MX + fu * P3X : MY + (first_y ? fu - R3Y : 0);
    int f_str = first_x ? 1 : P3X;
    const int own = ty * P3X + tx;   // the thread's cell, less 4 rows and 4 slots of halo
    T *const hdst = &lds[hr * P3X + hc], *const hdst2 = &lds[hr2 * P3X + hc2];

    T v[7];   // phi(k0-3 .. k0+3) of this cell's column
#pragma unroll
    for (int d = 0; d < 7; ++d) v[d] = load_at(base(phi, k0 - 3 + d), col);
    T halo_cur = halo ? load_at(base(phi, k0), hcol) : T(0);
    T halo2_cur = halo2 ? load_at(base(phi, k0), hcol2) : T(0);
    if (stopped()) return;
    T w0 = v[3], w1 = v[4], w2 = v[5], w3 = v[6];   // phi(p .. p+3)
    T wm1 = v[2], wm2 = v[1];                       // phi(p-1), phi(p-2) (EXACT)
    // z: second differences s(p-1), s(p), s(p+1), h(s(p)), e(p) and Q of face
    // p - 1/2, carried from plane to plane
    T za, zb, zc, zhb, ze, zq;
    {
        const T s2 = v[0] - T(2) * v[1] + v[2], s1 = v[1] - T(2) * v[2] + v[3];   // s(k0-2), s(k0-1)
        const T s0 = v[2] - T(2) * v[3] + v[4], sp = v[3] - T(2) * v[4] + v[5];   // s(k0), s(k0+1)
        za = s1;
        zb = s0;
        zc = sp;
        zhb = hj_h(zb);
        ze = zc - T(2) * zb + za;
        T unused;
        face(s2, s1, s0, sp, hj_h(s1), zhb, ze, s0 - T(2) * s1 + s2, unused, zq);
    }
    if (BTN == 1 && t == 0) lcount = 0;   // read after the loop's first barrier
    T lerr = T(0);
    // every load of the run-up is in, so that no plane waits for its own loads
    // where the loop's first entry would have to
    wait_loads();
    auto one_plane = [&](int pl) {
        // the plane index is the same in every lane: plane addresses are scalar
        const int p = __builtin_amdgcn_readfirstlane(pl);
        asm("" : "+v"(col), "+v"(hcol), "+v"(hcol2));
        // next plane's inputs, in flight while this one is computed
        const T w_next = load_at(base(phi, p + 4), col);
        const T halo_next = halo ? load_at(base(phi, p + 1), hcol) : T(0);
        const T halo2_next = halo2 ? load_at(base(phi, p + 1), hcol2) : T(0);
        // this plane's S0 and phi0, used after the two barriers
        const T s0_cur = load_at(base(S0, p), col);
        const T p0_cur = STAGE > 1 ? load_at(base(phi0, p), col) : T(0);

        // the previous plane's readers have passed its second barrier
        lds[own + 4 * P3X + 4] = w0;
        if (halo) *hdst = halo_cur;
        if (halo2) *hdst2 = halo2_cur;

        // z face p + 1/2: P is this plane's, Q the next one's
        const T zs_new = w1 - T(2) * w2 + w3;   // s(p + 2)
        const T zhc = hj_h(zc), ze_next = zs_new - T(2) * zc + zb;
        T zp, zq_next;
        face(za, zb, zc, zs_new, zhb, zhc, ze_next, ze, zp, zq_next);
        const T bz6 = hj_base(w0, w1, zb, zc);
        T zs1 = bz6 + zp, zs2 = (bz6 + ze) - zq;
        if constexpr (EXACT) {
            const T az = kz * central12(wm2, wm1, w1, w2);
            zs1 = az + kz * zp;
            zs2 = az - kz * zq;
        }
        __syncthreads();
        // x face i+1/2: P of this cell, Q of cell i+1
        T xs1, xs2, ys1, ys2;
        {
            const T *r = &lds[own + 4 * P3X + 4];
            const T m2 = r[-2], m1 = r[-1], c = w0, p1 = r[1], p2 = r[2], p3 = r[3];
            const T sa = m2 - T(2) * m1 + c, sb = m1 - T(2) * c + p1, sc = c - T(2) * p1 + p2, sd = p1 - T(2) * p2 + p3;
            const T e2 = sc - T(2) * sb + sa;
            T P, Q;
            face(sa, sb, sc, sd, hj_h(sb), hj_h(sc), sd - T(2) * sc + sb, e2, P, Q);
            lds[MX + own + 1] = Q;
            const T b6 = hj_base(c, p1, sb, sc);
            xs1 = b6 + P;
            xs2 = b6 + e2;
            if constexpr (EXACT) {
                xs2 = kx * central12(m2, m1, p1, p2);
                xs1 = xs2 + kx * P;
            }
        }
        // y face j+1/2
        {
            const T *r = &lds[own + 4 * P3X + 4];
            const T m2 = r[-2 * P3X], m1 = r[-P3X], c = w0, p1 = r[P3X], p2 = r[2 * P3X], p3 = r[3 * P3X];
            const T sa = m2 - T(2) * m1 + c, sb = m1 - T(2) * c + p1, sc = c - T(2) * p1 + p2, sd = p1 - T(2) * p2 + p3;
            const T e2 = sc - T(2) * sb + sa;
            T P, Q;
            face(sa, sb, sc, sd, hj_h(sb), hj_h(sc), sd - T(2) * sc + sb, e2, P, Q);
            lds[MY + own + P3X] = Q;
            const T b6 = hj_base(c, p1, sb, sc);
            ys1 = b6 + P;
            ys2 = b6 + e2;
            if constexpr (EXACT) {
                ys2 = ky * central12(m2, m1, p1, p2);
                ys1 = ys2 + ky * P;
            }
        }
        if (first_x || first_y) {
            asm("" : "+v"(f_off), "+v"(f_str), "+v"(f_dst));   // addresses formed here, not kept
            const T *f = &lds[f_off];
            const T v0 = f[0], v1 = f[f_str], v2 = f[2 * f_str], v3 = f[3 * f_str], v4 = f[4 * f_str],
                    v5 = f[5 * f_str];
            const T sa = v0 - T(2) * v1 + v2, sb = v1 - T(2) * v2 + v3, sc = v2 - T(2) * v3 + v4,
                    sd = v3 - T(2) * v4 + v5;
            T P, Q;
            face(sa, sb, sc, sd, hj_h(sb), hj_h(sc), sd - T(2) * sc + sb, sc - T(2) * sb + sa, P, Q);
            lds[f_dst] = Q;
        }
        __syncthreads();
        xs2 = EXACT ? xs2 - kx * lds[MX + own] : xs2 - lds[MX + own];
        ys2 = EXACT ? ys2 - ky * lds[MY + own] : ys2 - lds[MY + own];
        const T grad = EXACT ? godunov_sig(xs1, xs2, ys1, ys2, zs1, zs2, s0_cur, T(1), T(1), T(1))
                             : godunov_sig(xs1, xs2, ys1, ys2, zs1, zs2, s0_cur, kx, ky, kz);
        // lambda = 0: final off the band, replaced by k_redis3d_band on it
        const T l = s0_cur * grad - s0_cur;
        const T pn = rk_stage<T, STAGE>(w0, p0_cur, l, rdt);
        const bool band = BTN == 1 && inner && in_band_x(w0 * inv_w);
        // the next plane's inputs are in before this plane's stores go out:
        // a later wait for them would wait for the stores as well
        wait_loads();
        if (inner) {
            const size_t off = (size_t)p * plane;
            unsigned at = col;
            asm("" : "+v"(at));
            store_at(phi_out + off, at, pn);
            if (band) {
                const T del = band_delta(w0, inv_w);
                asm("" : "+v"(at));
                store_at(bf.gr + off, at, grad);
                store_at(bf.s2 + off, at, del * s0_cur * (grad - T(1)));
                store_at(bf.s3 + off, at, grad * del * del);
            } else if (STAGE == 3) {
                lerr = fmax(lerr, fabs(pn - p0_cur));
            }
        }
        if (BTN == 1) {
            // list this plane's band cells in LDS: one LDS atomic per wave
            const unsigned long long vote = __ballot(band);
            if (vote) {
                const unsigned below = __builtin_amdgcn_mbcnt_hi((unsigned)(vote >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((unsigned)vote, 0u));
                const int lead = __ffsll((long long)vote) - 1;
                unsigned at = 0;
                if (band && below == 0) at = atomicAdd(&lcount, (unsigned)__popcll(vote));
                at = __builtin_amdgcn_readlane(at, lead);
                if (band)
                    lcell[at + below] =
                        (unsigned short)((p - k0) * NT + t);
            }
        }
        wm2 = wm1;
        wm1 = w0;
        w0 = w1;
        w1 = w2;
        w2 = w3;
        w3 = w_next;
        za = zb;
        zb = zc;
        zc = zs_new;
        zhb = zhc;
        ze = ze_next;
        zq = zq_next;
        halo_cur = halo_next;
        halo2_cur = halo2_next;
    };
    // four planes a trip: the carried values then need no moves
    for (int pl = k0;;) {
        one_plane(pl);
        if (++pl >= k1) break;
        one_plane(pl);
        if (++pl >= k1) break;
        one_plane(pl);
        if (++pl >= k1) break;
        one_plane(pl);
        if (++pl >= k1) break;
    }
    if (BTN == 1) {
        // the workgroup's list onto the device list: one atomic
        __syncthreads();
        const unsigned nl = lcount;
        if (nl) {
            if (t == 0) lbase = atomicAdd(bcount, nl);
            __syncthreads();
            const unsigned at = lbase;
            for (unsigned e = t; e < nl; e += NT) {
                const unsigned lc = lcell[e], lt = lc % NT;
                blist[at + e] = (unsigned)((size_t)(k0 + (int)(lc / NT)) * plane) +
                                (unsigned)(j0 + (int)(lt / R3X)) * (unsigned)nx + (unsigned)(i0 + (int)(lt % R3X));
            }
        }
    }
    if (STAGE == 3) {
        double m = block_max((double)lerr);
        if (t == 0 && m > 0.0) atomic_max_nonneg(ctl_slot(ctl, step, (unsigned)tile_id), m);
    }
}

// The listed band cells: lambda from the 3x3x3 box sums of s2, s3 (centre
// weight 51, :409-448) in the reference's order -- in-plane sums row by row,
// then (plane k-1 + plane k) + plane k+1 -- and the cell's value.  Ghost cells
// of the box are the clamped interior cells (the zero-gradient fill of s2,
// s3).  Four lanes per listed cell: lanes 0..2 sum box planes k-1..k+1, lane
// 3 loads the cell itself and finishes it.  Consecutive stages alternate
// between two list lengths: this stage's (bcount) and the next one's (bnext),
// which this pass clears -- the previous stage's pass has read it, and the
// next stage's listing starts after this pass ends.  The stop flag, the list
// length, the list entries and the box loads of the first pass are in flight
// together: an entry at or past the length (stale, or never written) is
// clamped to a cell of the domain and its result dropped.
template <typename T, int STAGE>
__global__ __launch_bounds__(NT) void k_redis3d_band(const T *__restrict__ phi, T *__restrict__ phi_out,
                                                     const T *__restrict__ phi0, const T *__restrict__ S0,
                                                     RedisArgs ra, unsigned long long *ctl,
                                                     BandFields<T> bf, const unsigned *__restrict__ blist,
                                                     const unsigned *bcount, unsigned *bnext, RedisStep step)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *bnext = 0;
    const unsigned ncell = bcount[0];
    // stage 3: the maximum change in this workgroup's stripe, the stage
    // kernel's part of it complete now; a workgroup whose own maximum is not
    // above it skips the atomic (the 1,024 workgroups end together)
    unsigned long long *slot = ctl_slot(ctl, step, blockIdx.x);
    const unsigned long long stage_max = STAGE == 3 ? *slot : 0ull;
    const int nx = ra.nx, ny = ra.ny, nz = ra.nz;
    const T inv_w = (T)ra.inv_ls_wid, rdt = (T)ra.rdt;
    const unsigned plane = (unsigned)nx * (unsigned)ny, last = plane * (unsigned)nz - 1u;
    const int q = threadIdx.x & 3, g0 = (threadIdx.x & 63) & ~3;   // role, first lane of the four
    constexpr unsigned CPB = NT / 4;                                 // cells per workgroup and pass
    double lerr = 0.0;
    // the pass count is the same for every lane of the workgroup (shuffles)
    for (unsigned e0 = blockIdx.x * CPB;; e0 += gridDim.x * CPB) {
        const unsigned e = e0 + threadIdx.x / 4;
        // the list has room for every cell of the domain
        const unsigned c = min(blist[min(e, last)], last);
        // the stop flag (the stage kernel listed nothing) as a vector load,
        // behind the list entry, so that neither waits for the other
        const bool stopped = *reinterpret_cast<const volatile unsigned long long *>(ctl + 1) != 0;
        const unsigned rem = c % plane;
        const int k = (int)(c / plane), cj = (int)(rem / (unsigned)nx), ci = (int)(rem % (unsigned)nx);
        T part2 = T(0), part3 = T(0);
        T phc = T(0), s0 = T(0), grad = T(0), p0 = T(0), c2 = T(0), c3 = T(0);
        if (q < 3) {
            // box plane k-1+q: phi (band membership), s2 and s3 of its nine
            // cells, all loads in flight together; cells off the band contribute
            // nothing, whatever earlier stages left in s2 and s3 there
            const unsigned pb = (unsigned)clampi(k - 1 + q, 0, nz - 1) * plane;
            T pv[9], s2[9], s3[9];
#pragma unroll
            for (int jj = 0; jj < 3; ++jj)
#pragma unroll
                for (int ii = 0; ii < 3; ++ii) {
                    const unsigned at = pb + (unsigned)clampi(cj - 1 + jj, 0, ny - 1) * (unsigned)nx +
                                        (unsigned)clampi(ci - 1 + ii, 0, nx - 1);
                    pv[jj * 3 + ii] = phi[at];
                    s2[jj * 3 + ii] = bf.s2[at];
                    s3[jj * 3 + ii] = bf.s3[at];
                }
            if (stopped || e0 >= ncell) return;
#pragma unroll
            for (int r = 0; r < 9; ++r) {
                const bool inb = in_band_x(pv[r] * inv_w);
                part2 = part2 + (inb ? s2[r] : T(0));
                part3 = part3 + (inb ? s3[r] : T(0));
            }
        } else {
            phc = phi[c];
            s0 = S0[c];
            grad = bf.gr[c];
            c2 = bf.s2[c];
            c3 = bf.s3[c];
            if (STAGE > 1) p0 = phi0[c];
            if (stopped || e0 >= ncell) return;
        }
        const T a0 = __shfl(part2, g0, 64), a1 = __shfl(part2, g0 + 1, 64), a2 = __shfl(part2, g0 + 2, 64);
        const T b0 = __shfl(part3, g0, 64), b1 = __shfl(part3, g0 + 1, 64), b2 = __shfl(part3, g0 + 2, 64);
        if (q == 3 && e < ncell) {
            const T del = band_delta(phc, inv_w);
            const T la = T(51) * c2 + ((a0 + a1) + a2);
            const T lb = T(51) * c3 + ((b0 + b1) + b2);
            T lam = T(0);
            if (fabs(lb) > T(1.0e-12)) lam = la / lb * del;
            const T l = (s0 - lam) * grad - s0;
            const T pn = rk_stage<T, STAGE>(phc, p0, l, rdt);
            phi_out[c] = pn;
            if (STAGE == 3) lerr = fmax(lerr, (double)fabs(pn - p0));
        }
        if (e0 + gridDim.x * CPB >= ncell) break;
    }
    if (STAGE == 3) {
        double m = block_max(lerr);
        if (threadIdx.x == 0 && m > 0.0 && (unsigned long long)__double_as_longlong(m) > stage_max)
            atomic_max_nonneg(slot, m);
    }
}

static inline unsigned nb_of(int n, int b) { return (unsigned)((n + b - 1) / b); }

// workgroups of the band pass: four per CU of the device, four lanes a band
// cell (65536 cells a pass; a longer list takes more passes)
constexpr unsigned BAND_GRID = 1024;

// Planes a workgroup of the stage kernel marches, for `tiles` (x, y) tiles and
// nz planes.  A workgroup's march is a serial chain (1.1 us a plane with one
// workgroup on a CU, 2.6 us with four), so a grid that leaves the device
// idle is cut into shorter ones: the shortest that still fit one round of
// resident workgroups (1,024, four per CU).  us per pseudo-step with marches of
// 1, 2, 3, 4, 6, 8 and 16 planes (the rule's in brackets), FP64:
//   64^3        [50]  46   48   49   54   60   86
//   96^3         78   68   67  [65]  70   72   87
//   131x77x101   98   83   79   81  [81]  83  107
//   128^3       131  111  107  101  103 [101] 111
//   160^3       218  172  163  154  152 [151] 153
//   192^3       328  262  242  226  220 [217] 220
//   256^3       668  529  493  468  442  430 [416]
// Grids of several rounds take 8 planes where the tail of the last round counts and
// 16 from three rounds of 16, beyond which the three planes of run-up per march
// cost less than they save.
//
// FP32 holds twice the workgroups, so its marches are cut to two thousand, but
// not below three planes: 96^3 62, 53, [52], 52, 55, 58, 76; 131x77x101 76, 65, [62],
// 63, 66, 67, 88; 128^3 94, 79, 75, [73], 75, 74, 86.
static int stage_planes(unsigned tiles, int nz, bool fp32)
{
    constexpr int ROUND = 1024;
    auto fit = [&](int groups) {   // planes of the shortest marches that make so many workgroups
        const int blocks = std::max(1, groups / (int)tiles);
        return std::max(1, (nz + blocks - 1) / blocks);
    };
    int one = fit(ROUND);
    if (fp32) one = std::min(one, std::max(3, fit(2 * ROUND)));
    if (one <= 8) return one;
    return (size_t)tiles * nb_of(nz, RKC) >= (size_t)3 * ROUND ? RKC : 8;
}

template <typename T>
void launch_redis3d(hipStream_t st, int stage, int btn, const T *phi, T *phi_out, const T *phi0, const T *S0,
                    const RedisArgs &ra, unsigned long long *ctl, const unsigned char *tiles, const RedisBand<T> &bd,
                    bool band, RedisStep step)
{
    // the narrow band (tiles) marches RKC_NB planes per workgroup
    const int kc = tiles ? RKC_NB : stage_planes(nb_of(ra.nx, R3X) * nb_of(ra.ny, R3Y), ra.nz, sizeof(T) == 4);
    const dim3 g(nb_of(ra.nx, R3X) * nb_of(ra.ny, R3Y) * nb_of(ra.nz, kc));
#define LSMP_R3(S, B)                                                                                          \
    do {                                                                                                       \
        if (!band)                                                                                             \
            hipLaunchKernelGGL((tiles ? &k_redis3d<T, S, B, redis_exact<T, true>()> : &k_redis3d<T, S, B, false>), g, \
                               dim3(NT), 0, st, phi, phi_out, phi0, S0, ra, ctl, tiles, bd.f, bd.list, bd.count, kc, \
                               step);                                                                          \
        else if (B == 1)                                                                                       \
            hipLaunchKernelGGL((k_redis3d_band<T, S>), dim3(BAND_GRID), dim3(NT), 0, st, phi, phi_out, phi0,   \
                               S0, ra, ctl, bd.f, bd.list, bd.count, bd.next, step);                                \
    } while (0)
    if (btn) { if (stage == 1) LSMP_R3(1, 1); else if (stage == 2) LSMP_R3(2, 1); else LSMP_R3(3, 1); }
    else { if (stage == 1) LSMP_R3(1, 0); else if (stage == 2) LSMP_R3(2, 0); else LSMP_R3(3, 0); }
#undef LSMP_R3
}

template void launch_redis3d<double>(hipStream_t, int, int, const double *, double *, const double *, const double *,
                                     const RedisArgs &, unsigned long long *, const unsigned char *,
                                     const RedisBand<double> &, bool, RedisStep);
template void launch_redis3d<float>(hipStream_t, int, int, const float *, float *, const float *, const float *,
                                    const RedisArgs &, unsigned long long *, const unsigned char *,
                                    const RedisBand<float> &, bool, RedisStep);

}  // namespace lsmp
