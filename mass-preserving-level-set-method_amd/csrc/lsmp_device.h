// lsmp_device.h -- per-point numerics of the level-set transport step, shared
// by the gfx950 kernels.  Each function restates one reference formula; the
// association order of every sum and product is the reference's (Fortran
// evaluates left to right; x**2.0d0 is a square).
#pragma once
#include <hip/hip_runtime.h>

#define LSMP_DEV __device__ __forceinline__

namespace lsmp {

template <typename T> LSMP_DEV T sq(T x) { return x * x; }
template <typename T> LSMP_DEV T dabs(T x) { return fabs(x); }
LSMP_DEV int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Workgroups are handed to the 8 XCDs of the device in turn, each XCD with its
// own L2.  This renumbers workgroup b so that XCD x takes a contiguous range
// (the first nb % 8 XCDs one workgroup more): neighbouring strided lines, which
// share cache lines, then run on the same XCD at about the same time.
LSMP_DEV int xcd_renumber(int b, int nb)
{
    const int x = b % 8, i = b / 8, q = nb / 8, r = nb % 8;
    return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}
LSMP_DEV int xcd_block() { return xcd_renumber((int)blockIdx.x, (int)gridDim.x); }

// Pointwise flux split g = 1/2 (u + |u|) phi, f = 1/2 (u - |u|) phi
// (level_set_rk3_solver.f90:118-125).
template <typename T> LSMP_DEV void flux_split(T phi, T u, T &g, T &f)
{
    g = T(0.5) * (u + fabs(u)) * phi;
    f = T(0.5) * (u - fabs(u)) * phi;
}

// WENO-JS5 reconstruction of the positive flux at i+1/2 from g(i-2..i+2)
// (level_set_rk3_solver.f90:296-317).
template <typename T> LSMP_DEV T wenojs_g(T g0, T g1, T g2, T g3, T g4)
{
    const T EPS = T(1.0e-13);
    T b1 = T(13) * sq(g0 - T(2) * g1 + g2) + T(3) * sq(g0 - T(4) * g1 + T(3) * g2);
    T b2 = T(13) * sq(g1 - T(2) * g2 + g3) + T(3) * sq(g1 - g3);
    T b3 = T(13) * sq(g2 - T(2) * g3 + g4) + T(3) * sq(T(3) * g2 - T(4) * g3 + g4);
    T a1 = T(1) / sq(EPS + b1);
    T a2 = T(6) / sq(EPS + b2);
    T a3 = T(3) / sq(EPS + b3);
    T w1 = a1 / (a1 + a2 + a3);
    T w2 = a2 / (a1 + a2 + a3);
    T w3 = a3 / (a1 + a2 + a3);
    return w1 / T(3) * g0 - (T(7) * w1 + w2) / T(6) * g1 +
           (T(11) * w1 + T(5) * w2 + T(2) * w3) / T(6) * g2 +
           (T(2) * w2 + T(5) * w3) / T(6) * g3 - w3 / T(6) * g4;
}

// WENO-JS5 reconstruction of the negative flux at i+1/2 from f(i-1..i+3)
// (level_set_rk3_solver.f90:319-342).
template <typename T> LSMP_DEV T wenojs_f(T f0, T f1, T f2, T f3, T f4)
{
    const T EPS = T(1.0e-13);
    T b3 = T(13) * sq(f0 - T(2) * f1 + f2) + T(3) * sq(f0 - T(4) * f1 + T(3) * f2);
    T b2 = T(13) * sq(f1 - T(2) * f2 + f3) + T(3) * sq(f1 - f3);
    T b1 = T(13) * sq(f2 - T(2) * f3 + f4) + T(3) * sq(T(3) * f2 - T(4) * f3 + f4);
    T a1 = T(1) / sq(EPS + b1);
    T a2 = T(6) / sq(EPS + b2);
    T a3 = T(3) / sq(EPS + b3);
    T w1 = a1 / (a1 + a2 + a3);
    T w2 = a2 / (a1 + a2 + a3);
    T w3 = a3 / (a1 + a2 + a3);
    return w3 * (-f0 + T(5) * f1 + T(2) * f2) / T(6) +
           w2 * (T(2) * f1 + T(5) * f2 - f3) / T(6) +
           w1 * (T(11) * f2 - T(7) * f3 + T(2) * f4) / T(6);
}

// One CRWENO5 row of the positive-flux system from g(i-2..i+2)
// (level_set_rk3_solver.f90:362-381).
template <typename T>
LSMP_DEV void crweno_g_row(T g0, T g1, T g2, T g3, T g4, T &A, T &B, T &C, T &S)
{
    const T EPS = T(1.0e-13);
    const T c1 = T(0.2089141306), c2 = T(0.4999999998), c3 = T(0.2910858692);
    T b1 = T(13) * sq(g0 - T(2) * g1 + g2) + T(3) * sq(g0 - T(4) * g1 + T(3) * g2);
    T b2 = T(13) * sq(g1 - T(2) * g2 + g3) + T(3) * sq(g1 - g3);
    T b3 = T(13) * sq(g2 - T(2) * g3 + g4) + T(3) * sq(T(3) * g2 - T(4) * g3 + g4);
    T a1 = c1 * (T(1) + fabs(b3 - b1) / (EPS + b1));
    T a2 = c2 * (T(1) + fabs(b3 - b1) / (EPS + b2));
    T a3 = c3 * (T(1) + fabs(b3 - b1) / (EPS + b3));
    T w1 = a1 / (a1 + a2 + a3);
    T w2 = a2 / (a1 + a2 + a3);
    T w3 = a3 / (a1 + a2 + a3);
    A = (T(2) * w1 + w2) / T(3);
    B = (w1 + T(2) * (w2 + w3)) / T(3);
    C = w3 / T(3);
    S = w1 / T(6) * g1 + (T(5) * (w1 + w2) + w3) / T(6) * g2 + (w2 + T(5) * w3) / T(6) * g3;
}

// One CRWENO5 row of the negative-flux system from f(i-1..i+3)
// (level_set_rk3_solver.f90:388-407).
template <typename T>
LSMP_DEV void crweno_f_row(T f0, T f1, T f2, T f3, T f4, T &A, T &B, T &C, T &S)
{
    const T EPS = T(1.0e-13);
    const T c1 = T(0.2089141306), c2 = T(0.4999999998), c3 = T(0.2910858692);
    T b3 = T(13) * sq(f0 - T(2) * f1 + f2) + T(3) * sq(f0 - T(4) * f1 + T(3) * f2);
    T b2 = T(13) * sq(f1 - T(2) * f2 + f3) + T(3) * sq(f1 - f3);
    T b1 = T(13) * sq(f2 - T(2) * f3 + f4) + T(3) * sq(T(3) * f2 - T(4) * f3 + f4);
    T a1 = c1 * (T(1) + fabs(b3 - b1) / (EPS + b1));
    T a2 = c2 * (T(1) + fabs(b3 - b1) / (EPS + b2));
    T a3 = c3 * (T(1) + fabs(b3 - b1) / (EPS + b3));
    T w1 = a1 / (a1 + a2 + a3);
    T w2 = a2 / (a1 + a2 + a3);
    T w3 = a3 / (a1 + a2 + a3);
    A = (w3) / T(3);
    B = (w1 + T(2) * (w2 + w3)) / T(3);
    C = (w2 + T(2) * w1) / T(3);
    S = (T(5) * w3 + w2) / T(6) * f1 + (w3 + T(5) * (w2 + w1)) / T(6) * f2 + w1 / T(6) * f3;
}

// Reciprocal of a normal nonzero number (either sign): the hardware estimate
// refined by Newton steps (two in FP64, one in FP32), within an ulp or two of
// the correctly rounded 1/x.
LSMP_DEV double rcp_pos(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}
LSMP_DEV float rcp_pos(float x)
{
    float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}

// The same with one Newton step in FP64: the hardware estimate is good to
// about 5e-8, one step to about 2e-15 of 1/x -- enough for the WENO-HJ
// weights, which multiply a correction term that is itself small.
LSMP_DEV double rcp_w(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    return fma(r, fma(-x, r, 1.0), r);
}
LSMP_DEV float rcp_w(float x) { return rcp_pos(x); }

// Lane l - 1's and lane l + 1's value (wave_shr:1, wave_shl:1); the first and
// the last lane keep their own.
template <int CTRL> LSMP_DEV float lane_shift(float v)
{
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, false));
}
template <int CTRL> LSMP_DEV double lane_shift(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false));
}
template <typename T> LSMP_DEV T from_left(T v) { return lane_shift<0x138>(v); }
template <typename T> LSMP_DEV T from_right(T v) { return lane_shift<0x130>(v); }

// X of a tridiagonal system a X(-1) + b X + c X(+1) = d, one row a lane of groups of
// LANES (a = 0 in a group's first lane, c = 0 in its last), by parallel cyclic
// reduction.  A row divided by its b is handed to the neighbours as three
// values; a lane whose neighbour lies outside has a (c) = 0 by then and may read
// any finite row.  The couplings square with every step (0.55^K to begin with for
// interfaces K CRWENO rows apart on smooth data): once |a|, |c| <= TOL in every
// lane, leaving them out changes X by at most 2 TOL max |X| (half an ulp; FP32 a
// quarter), and the remaining steps are left out.
template <int LANES, typename T> LSMP_DEV T pcr_solve(T a, T b, T c, T d)
{
    constexpr T TOL = sizeof(T) == 8 ? T(0x1p-54) : T(0x1p-26);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int st = 1; st < LANES; st <<= 1) {
        const T r = rcp_pos(b);
        a *= r;
        c *= r;
        d *= r;
        if (__all(fabs(a) <= TOL && fabs(c) <= TOL)) return d;
        T am, cm, dm, ap, cq, dq;
        if (st == 1) {
            am = from_left(a); cm = from_left(c); dm = from_left(d);
            ap = from_right(a); cq = from_right(c); dq = from_right(d);
        } else {
            const int lm = lane - st, lp = lane + st;   // (modulo 64)
            am = __shfl(a, lm, 64); cm = __shfl(c, lm, 64); dm = __shfl(d, lm, 64);
            ap = __shfl(a, lp, 64); cq = __shfl(c, lp, 64); dq = __shfl(d, lp, 64);
        }
        b = (T(1) - cm * a) - ap * c;
        d = (d - dm * a) - dq * c;
        a = -am * a;
        c = -cq * c;
    }
    return d * rcp_pos(b);
}

// The same by every step of the reduction, four values a row (adv_exact): with the
// neighbours' reciprocals (DIV false) or divisions by them.
template <int LANES, bool DIV, typename T> LSMP_DEV T pcr_solve_full(T ra, T rb, T rc, T rd)
{
    const int lane = threadIdx.x & 63, s = lane & (LANES - 1);
#pragma unroll
    for (int st = 1; st < LANES; st <<= 1) {
        const bool hasm = s - st >= 0, hasp = s + st < LANES;
        const int lm = hasm ? lane - st : lane, lp = hasp ? lane + st : lane;
        const T ib = DIV ? rb : rcp_w(rb);
        const T am = __shfl(ra, lm, 64), im = __shfl(ib, lm, 64), cm = __shfl(rc, lm, 64), dm = __shfl(rd, lm, 64);
        const T ap = __shfl(ra, lp, 64), ip = __shfl(ib, lp, 64), cq = __shfl(rc, lp, 64), dq = __shfl(rd, lp, 64);
        const T k1 = !hasm ? T(0) : DIV ? ra / im : ra * im, k2 = !hasp ? T(0) : DIV ? rc / ip : rc * ip;
        const T na = -am * k1, nc = -cq * k2;
        const T nb = rb - cm * k1 - ap * k2, nd = rd - dm * k1 - dq * k2;
        ra = na;
        rb = nb;
        rc = nc;
        rd = nd;
    }
    return DIV ? rd / rb : rd * rcp_w(rb);
}

// sqrt of x >= 0 from the hardware reciprocal square root (good to about 6e-8)
// and one Newton step: good to about 5e-15 of sqrt(x); exactly 0 at x = 0.
LSMP_DEV double sqrt_w(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double s = x * y;
    const double r = fma(fma(-s, s, x), 0.5 * y, s);
    return x > 0.0 ? r : 0.0;
}
LSMP_DEV float sqrt_w(float x) { return __builtin_amdgcn_sqrtf(x); }
// the same to an ulp: a second step in FP64, the rounded square root in FP32
LSMP_DEV double sqrt_n(double x)
{
    const double y = __builtin_amdgcn_rsq(x), h = 0.5 * y, s = x * y;
    const double r = fma(fma(-s, s, x), h, s);
    return x > 0.0 ? fma(fma(-r, r, x), h, r) : 0.0;
}
LSMP_DEV float sqrt_n(float x) { return sqrt(x); }

// The g row up to a positive factor (the solvers use A, B, C and S of a row only
// together): with e_k = EPS + b_k and tau = |b3 - b1| the reference's weights
// a_k = c_k (1 + tau / e_k) are proportional to c_k (e_k + tau) prod_{m != k} e_m,
// so FP64 takes no reciprocal at all.  Equal to crweno_*_row() up to rounding
// of the weights.  The products need the FP64 exponent range: e_k lies in
// [1e-13, ~2e3], so a product of three can reach 1e-39, below FP32's normal
// range; the FP32 form keeps one reciprocal per weight and normalises.
LSMP_DEV void crweno_weights_fast(double b1, double b2, double b3, double &w1, double &w2, double &w3)
{
    const double EPS = 1.0e-13;
    const double c1 = 0.2089141306, c2 = 0.4999999998, c3 = 0.2910858692;
    const double tau = fabs(b3 - b1);
    const double e1 = EPS + b1, e2 = EPS + b2, e3 = EPS + b3;
    w1 = c1 * (e1 + tau) * (e2 * e3);
    w2 = c2 * (e2 + tau) * (e1 * e3);
    w3 = c3 * (e3 + tau) * (e1 * e2);
}
LSMP_DEV void crweno_weights_fast(float b1, float b2, float b3, float &w1, float &w2, float &w3)
{
    const float EPS = 1.0e-13f;
    const float c1 = 0.2089141306f, c2 = 0.4999999998f, c3 = 0.2910858692f;
    const float tau = fabsf(b3 - b1);
    const float a1 = c1 * (1.0f + tau * rcp_pos(EPS + b1));
    const float a2 = c2 * (1.0f + tau * rcp_pos(EPS + b2));
    const float a3 = c3 * (1.0f + tau * rcp_pos(EPS + b3));
    const float r = rcp_pos(a1 + a2 + a3);
    w1 = a1 * r;
    w2 = a2 * r;
    w3 = a3 * r;
}

template <typename T>
LSMP_DEV void crweno_g_row_fast(T g0, T g1, T g2, T g3, T g4, T &A, T &B, T &C, T &S)
{
    T b1 = T(13) * sq(g0 - T(2) * g1 + g2) + T(3) * sq(g0 - T(4) * g1 + T(3) * g2);
    T b2 = T(13) * sq(g1 - T(2) * g2 + g3) + T(3) * sq(g1 - g3);
    T b3 = T(13) * sq(g2 - T(2) * g3 + g4) + T(3) * sq(T(3) * g2 - T(4) * g3 + g4);
    T w1, w2, w3;
    crweno_weights_fast(b1, b2, b3, w1, w2, w3);
    // three times the row
    A = T(2) * w1 + w2;
    B = w1 + T(2) * (w2 + w3);
    C = w3;
    S = (w1 * g1 + (T(5) * (w1 + w2) + w3) * g2 + (w2 + T(5) * w3) * g3) * T(0.5);
}

// The normalised row itself, for the narrow band in FP32 (adv_exact).
LSMP_DEV void crweno_g_row_unit(float g0, float g1, float g2, float g3, float g4, float &A, float &B, float &C,
                                float &S)
{
    float b1 = 13.0f * sq(g0 - 2.0f * g1 + g2) + 3.0f * sq(g0 - 4.0f * g1 + 3.0f * g2);
    float b2 = 13.0f * sq(g1 - 2.0f * g2 + g3) + 3.0f * sq(g1 - g3);
    float b3 = 13.0f * sq(g2 - 2.0f * g3 + g4) + 3.0f * sq(3.0f * g2 - 4.0f * g3 + g4);
    float w1, w2, w3;
    crweno_weights_fast(b1, b2, b3, w1, w2, w3);
    const float third = float(1.0 / 3.0), sixth = float(1.0 / 6.0);
    A = (2.0f * w1 + w2) * third;
    B = (w1 + 2.0f * (w2 + w3)) * third;
    C = w3 * third;
    S = (w1 * g1 + (5.0f * (w1 + w2) + w3) * g2 + (w2 + 5.0f * w3) * g3) * sixth;
}

// FP32 in the narrow band keeps the rounding of the full reduction over normalised
// rows: the tube's tiles are the ones with a cell |phi| < W, and beyond its edge phi
// is +-W up to the rounding of the advection, so that other roundings would move
// the tube's edge by a tile here and there (0.2 dx in the tile's flat cells).  Every
// solve a line can take does so (tiles, a wave per line, paired, twisted).
template <typename T, bool NB> constexpr bool adv_exact() { return NB && sizeof(T) == 4; }
template <typename T, bool NB>
LSMP_DEV void crweno_row(T g0, T g1, T g2, T g3, T g4, T &A, T &B, T &C, T &S)
{
    if constexpr (adv_exact<T, NB>()) crweno_g_row_unit(g0, g1, g2, g3, g4, A, B, C, S);
    else crweno_g_row_fast(g0, g1, g2, g3, g4, A, B, C, S);
}

// WENO-HJ correction term (level_set_rk3_redis.f90:456-471).
template <typename T> LSMP_DEV T phyn(T a, T b, T c, T d)
{
    const T eps = T(1.0e-6);
    T is0 = T(13) * sq(a - b) + T(3) * sq(a - T(3) * b);
    T is1 = T(13) * sq(b - c) + T(3) * sq(b + c);
    T is2 = T(13) * sq(c - d) + T(3) * sq(T(3) * c - d);
    T alp0 = T(1) / sq(eps + is0);
    T alp1 = T(6) / sq(eps + is1);
    T alp2 = T(3) / sq(eps + is2);
    T w0 = alp0 / (alp0 + alp1 + alp2);
    T w2 = alp2 / (alp0 + alp1 + alp2);
    return w0 / T(3) * (a - T(2) * b + c) + (w2 - T(0.5)) / T(6) * (b - T(2) * c + d);
}

// The same WENO-HJ term with its five divisions folded into one reciprocal:
// with q_k = (eps + IS_k)^2 the reference's alp0 = 1/q0, alp1 = 6/q1,
// alp2 = 3/q2 normalise to w0 = q1 q2 / D and w2 = 3 q0 q1 / D with
// D = q1 q2 + 6 q0 q2 + 3 q0 q1.  Equal to phyn() up to rounding of the weights
// (q_k lies in [1e-12, 3e6], so D neither under- nor overflows in FP32).
// sbc = (b - c)^2 and scd = (c - d)^2 come from the caller: the two terms of
// one direction share them (squares of opposite differences are equal).
template <typename T> LSMP_DEV T phyn_fast(T a, T b, T c, T d, T sbc, T scd)
{
    const T eps = T(1.0e-6);
    T is0 = T(13) * sq(a - b) + T(3) * sq(a - T(3) * b);
    T is1 = T(13) * sbc + T(3) * sq(b + c);
    T is2 = T(13) * scd + T(3) * sq(T(3) * c - d);
    T q0 = sq(eps + is0), q1 = sq(eps + is1), q2 = sq(eps + is2);
    T q12 = q1 * q2, q01 = q0 * q1;
    T r = rcp_w(q12 + T(6) * (q0 * q2) + T(3) * q01);
    // w0/3 = q12 r/3 and (w2 - 1/2)/6 = q01 r/2 - 1/12
    T t0 = q12 * (r * T(1.0 / 3.0));
    T t2 = fma(q01, r * T(0.5), T(-1.0 / 12.0));
    return fma(t0, a - T(2) * b + c, t2 * (b - T(2) * c + d));
}

// WENO-HJ on a line with second differences s_m = phi(m+1) - 2 phi(m) + phi(m-1)
// (level_set_rk3_redis.f90:290-315, 456-471), everything times 6 dx:
//   6 dx D+(m) = b(m) + P(m+1/2),          b(m) = 6 (phi(m+1) - phi(m)) - s(m+1) - 2 s(m),
//   6 dx D-(m) = b(m) + e(m) - Q(m-1/2),   e(m) = s(m+1) - 2 s(m) + s(m-1),
// where the central part and the constant -1/2 of the weights are merged into
// b and b + e (each of third order, one-sided), and P, Q are the weighted third
// differences of a face, formed together: the indicators of P at m+1/2 and of
// Q there are those of s(m-1..m+2) in reversed roles.  An indicator plus eps
// is a sum of two squares,
//   13 (a - b)^2 + 3 (a - 3b)^2 = 16 ((a - 1.375 b)^2 + 0.609375 b^2),
//   13 (b - c)^2 + 3 (b + c)^2 = 16 ((b - 0.625 c)^2 + 0.609375 c^2),
// so that h(s) = 0.609375 s^2 + eps / 16 of the two middle differences serves
// all three of a face (hj_h; the common factor 16 drops out of the weights).
template <typename T> LSMP_DEV T hj_h(T s) { return fma(T(0.609375) * s, s, T(1.0e-6 / 16.0)); }

// P and Q of face m+1/2: sa..sd = s(m-1..m+2), hb = hj_h(sb), hc = hj_h(sc),
// e1 = e(m+1) = sd - 2 sc + sb, e2 = e(m) = sc - 2 sb + sa.  With q the squares of
// the indicators, P = (2 qJ qB e1 + 3 qA qJ e2) / Dp, Dp = qJ qB + 3 qA qJ +
// 6 qA qB, and Q the same with A and B, e1 and e2 exchanged.  FP64 takes both
// reciprocals from one (the product of the two denominators stays within
// [1e-58, 1e28]); FP32 denominators stay within [1e-28, 1e13].
template <typename T> struct HjFace {
    T dp, dm, yp, ym;   // P = yp / dp, Q = ym / dm
};
template <typename T> LSMP_DEV HjFace<T> weno_hj_parts(T sa, T sb, T sc, T sd, T hb, T hc, T e1, T e2)
{
    const T tA = fma(T(-1.375), sc, sd), tJ = fma(T(-0.625), sc, sb), tB = fma(T(-1.375), sb, sa);
    const T qA = sq(fma(tA, tA, hc)), qJ = sq(fma(tJ, tJ, hc)), qB = sq(fma(tB, tB, hb));
    const T pJB = qJ * qB, pAJ = qA * qJ, pAB = qA * qB;
    const T w = fma(T(6), pAB, pAJ + pJB);
    const T u1 = pJB * e1, u2 = pAJ * e2, t = u1 + u2;
    return {fma(T(2), pAJ, w), fma(T(2), pJB, w), fma(T(2), t, u2), fma(T(2), t, u1)};
}
template <typename T> LSMP_DEV void weno_hj_face(T sa, T sb, T sc, T sd, T hb, T hc, T e1, T e2, T &P, T &Q)
{
    const HjFace<T> f = weno_hj_parts(sa, sb, sc, sd, hb, hc, e1, e2);
    if constexpr (sizeof(T) == 8) {
        const T r = rcp_w(f.dp * f.dm);
        P = (f.dm * r) * f.yp;
        Q = (f.dp * r) * f.ym;
    } else {
        P = rcp_w(f.dp) * f.yp;
        Q = rcp_w(f.dm) * f.ym;
    }
}

// b(m) from phi(m), phi(m+1), s(m), s(m+1)
template <typename T> LSMP_DEV T hj_base(T c, T p1, T s0, T s1)
{
    return fma(T(-2), s0, fma(T(6), p1 - c, -s1));
}

// The same face times 12 d with its indicators over shared squares, and the central
// part times 12 d: FP32 in the narrow band (redis_exact) keeps these roundings, for
// the reason given at adv_exact.
LSMP_DEV void weno_hj_face12(float sa, float sb, float sc, float sd, float &plus, float &minus)
{
    const float eps = 1.0e-6f;
    const float bb = sb * sb, cc = sc * sc;
    const float fA = fma(40.0f, cc, fma(sd, fma(16.0f, sd, -44.0f * sc), eps));
    const float fJ = fma(16.0f, bb, fma(sc, fma(16.0f, sc, -20.0f * sb), eps));
    const float fB = fma(40.0f, bb, fma(sa, fma(16.0f, sa, -44.0f * sb), eps));
    const float qA = sq(fA), qJ = sq(fJ), qB = sq(fB);
    const float pJB = qJ * qB, pAJ = qA * qJ, pAB = qA * qB;
    const float dp = fma(3.0f, fma(2.0f, pAB, pAJ), pJB), dm = fma(3.0f, fma(2.0f, pAB, pJB), pAJ);
    const float e1 = sd - 2.0f * sc + sb, e2 = sc - 2.0f * sb + sa;
    const float u1 = pJB * e1, u2 = pAJ * e2;
    plus = fma(rcp_w(dp), fma(4.0f, u1, 6.0f * u2), -e2);
    minus = fma(rcp_w(dm), fma(4.0f, u2, 6.0f * u1), -e1);
}
LSMP_DEV float central12(float m2, float m1, float p1, float p2) { return fma(8.0f, p1 - m1, m2 - p2); }
template <typename T, bool NB> constexpr bool redis_exact() { return NB && sizeof(T) == 4; }

// D+ and D- times 6 d of one cell from phi(m-3 .. m+3), its two faces formed for it alone
template <typename T>
LSMP_DEV void weno_hj_cell(T m3, T m2, T m1, T c, T p1, T p2, T p3, T &dp6, T &dm6)
{
    const T sa = m3 - T(2) * m2 + m1, sb = m2 - T(2) * m1 + c, sc = m1 - T(2) * c + p1, sd = c - T(2) * p1 + p2,
            se = p1 - T(2) * p2 + p3;   // s(m-2) .. s(m+2)
    const T e0 = sc - T(2) * sb + sa, e1 = sd - T(2) * sc + sb, e2 = se - T(2) * sd + sc;   // e(m-1), e(m), e(m+1)
    const T hc = hj_h(sc);
    const HjFace<T> l = weno_hj_parts(sa, sb, sc, sd, hj_h(sb), hc, e1, e0);   // face m-1/2, for its Q
    const HjFace<T> r = weno_hj_parts(sb, sc, sd, se, hc, hj_h(sd), e2, e1);   // face m+1/2, for its P
    T P, Q;
    if constexpr (sizeof(T) == 8) {
        const T i = rcp_w(r.dp * l.dm);
        P = (l.dm * i) * r.yp;
        Q = (r.dp * i) * l.ym;
    } else {
        P = rcp_w(r.dp) * r.yp;
        Q = rcp_w(l.dm) * l.ym;
    }
    const T b6 = hj_base(c, p1, sc, sd);
    dp6 = b6 + P;
    dm6 = (b6 + e1) - Q;
}

// D+ and D- from the five second differences s_m = phi(m+1) - 2 phi(m) + phi(m-1),
// m = i-2..i+2, shared by both one-sided terms.
template <typename T>
LSMP_DEV void weno_hj_pm_fast(T m3, T m2, T m1, T c, T p1, T p2, T p3, T inv12d, T invd, T &dp, T &dm)
{
    const T a = inv12d * (-(m1 - m2) + T(7) * (c - m1) + T(7) * (p1 - c) - (p2 - p1));
    const T sm2 = m3 - T(2) * m2 + m1, sm1 = m2 - T(2) * m1 + c, s0 = m1 - T(2) * c + p1;
    const T sp1 = c - T(2) * p1 + p2, sp2 = p1 - T(2) * p2 + p3;
    // (sp1 - s0)^2 is is1 of D+ and is2 of D-; (s0 - sm1)^2 is2 of D+ and is1 of D-
    const T qp = sq(sp1 - s0), qm = sq(s0 - sm1);
    dp = a + invd * phyn_fast(sp2, sp1, s0, sm1, qp, qm);
    dm = a - invd * phyn_fast(sm2, sm1, s0, sp1, qm, qp);
}

// H and delta of ls_funs in FP64 without library calls: with theta = pi x / 2
// in (-pi/2, pi/2) for a cell of the band (x = phi / w), delta = cos(theta)^2 / w
// and sin(pi x) = 2 sin(theta) cos(theta), sine and cosine from their Taylor
// series (remainders below 2e-17).  Within 2.3e-16 of correctly rounded H and
// delta w.
LSMP_DEV void ls_funs_taylor(double phi, double w, double &H, double &D)
{
    const double eps = 1.0e-12;
    const double x = phi / w;
    H = x > 0.0 ? 1.0 : 0.0;
    D = 0.0;
    if (x > 1.0 - eps || x < -1.0 + eps) return;
    const double th = x * 1.570796326794896619231321691639751442, t = th * th;
    double c = 1.0 / 2432902008176640000.0;        // 1/20!
    c = fma(c, t, -1.0 / 6402373705728000.0);      // -1/18!
    c = fma(c, t, 1.0 / 20922789888000.0);         // 1/16!
    c = fma(c, t, -1.0 / 87178291200.0);           // -1/14!
    c = fma(c, t, 1.0 / 479001600.0);              // 1/12!
    c = fma(c, t, -1.0 / 3628800.0);               // -1/10!
    c = fma(c, t, 1.0 / 40320.0);                  // 1/8!
    c = fma(c, t, -1.0 / 720.0);                   // -1/6!
    c = fma(c, t, 1.0 / 24.0);                     // 1/4!
    c = fma(c, t, -0.5);                           // -1/2!
    c = fma(c, t, 1.0);
    double s = 1.0 / 51090942171709440000.0;       // 1/21!
    s = fma(s, t, -1.0 / 121645100408832000.0);    // -1/19!
    s = fma(s, t, 1.0 / 355687428096000.0);        // 1/17!
    s = fma(s, t, -1.0 / 1307674368000.0);         // -1/15!
    s = fma(s, t, 1.0 / 6227020800.0);             // 1/13!
    s = fma(s, t, -1.0 / 39916800.0);              // -1/11!
    s = fma(s, t, 1.0 / 362880.0);                 // 1/9!
    s = fma(s, t, -1.0 / 5040.0);                  // -1/7!
    s = fma(s, t, 1.0 / 120.0);                    // 1/5!
    s = fma(s, t, -1.0 / 6.0);                     // -1/3!
    s = fma(s, t, 1.0) * th;
    H = fmax(fmin(0.5 * ((1.0 + x) + 2.0 * (s * c) * 0.318309886183790671537767526745028724), 1.0), 0.0);
    D = c * c / w;
}

// Fourth-order central slope times 12 dx (level_set_rk3_redis.f90:290-293).
template <typename T> LSMP_DEV T central4(T m2, T m1, T c, T p1, T p2)
{
    return -(m1 - m2) + T(7) * (c - m1) + T(7) * (p1 - c) - (p2 - p1);
}

// D+ and D- along one direction from phi(i-3..i+3) (level_set_rk3_redis.f90:305-315).
template <typename T>
LSMP_DEV void weno_hj_pm(T m3, T m2, T m1, T c, T p1, T p2, T p3, T inv12d, T invd, T &dp, T &dm)
{
    T a = inv12d * central4(m2, m1, c, p1, p2);
    dp = a + invd * phyn(p3 - T(2) * p2 + p1, p2 - T(2) * p1 + c, p1 - T(2) * c + m1, c - T(2) * m1 + m2);
    dm = a - invd * phyn(m3 - T(2) * m2 + m1, m2 - T(2) * m1 + c, m1 - T(2) * c + p1, c - T(2) * p1 + p2);
}

// Godunov |grad phi| selected by the frozen sign S0 (level_set_rk3_redis.f90:341-360).
template <typename T, int DIM>
LSMP_DEV T godunov(T xs1, T xs2, T ys1, T ys2, T zs1, T zs2, T s0)
{
    T upm = -fmin(xs1, T(0)), upp = fmax(xs1, T(0));
    T umm = -fmin(xs2, T(0)), ump = fmax(xs2, T(0));
    T vpm = -fmin(ys1, T(0)), vpp = fmax(ys1, T(0));
    T vmm = -fmin(ys2, T(0)), vmp = fmax(ys2, T(0));
    if (DIM == 3) {
        T wpm = -fmin(zs1, T(0)), wpp = fmax(zs1, T(0));
        T wmm = -fmin(zs2, T(0)), wmp = fmax(zs2, T(0));
        if (s0 >= T(0)) return sqrt(sq(fmax(upm, ump)) + sq(fmax(vpm, vmp)) + sq(fmax(wpm, wmp)));
        return sqrt(sq(fmax(upp, umm)) + sq(fmax(vpp, vmm)) + sq(fmax(wpp, wmm)));
    } else {
        if (s0 >= T(0)) return sqrt(sq(fmax(upm, ump)) + sq(fmax(vpm, vmp)));
        return sqrt(sq(fmax(upp, umm)) + sq(fmax(vpp, vmm)));
    }
}

// delta != 0 only where ls_funs takes its middle branch
template <typename T> LSMP_DEV bool in_band_x(T x)
{
    return !(x > T(1) - T(1.0e-12)) && !(x < T(-1) + T(1.0e-12));
}

// delta of ls_funs for a cell of the band (its middle branch, |x| < 1 with
// x = phi / ls_wid): 0.5 (1 + cos(pi x)) / ls_wid = cos(theta)^2 / ls_wid with
// theta = pi x / 2 in (-pi/2, pi/2), cos from its Taylor series in theta^2 to
// the term in theta^20 (remainder below 2e-17 there).  Within 2.3e-16 of
// 0.5 (1 + cos(pi x)) evaluated with a correctly rounded cosine.
template <typename T> LSMP_DEV T band_delta(T phi, T inv_w)
{
    const T th = (phi * inv_w) * T(1.570796326794896619231321691639751442);
    const T t = th * th;
    T c = T(1.0 / 2432902008176640000.0);     // 1/20!
    c = fma(c, t, T(-1.0 / 6402373705728000.0));   // -1/18!
    c = fma(c, t, T(1.0 / 20922789888000.0));      // 1/16!
    c = fma(c, t, T(-1.0 / 87178291200.0));        // -1/14!
    c = fma(c, t, T(1.0 / 479001600.0));           // 1/12!
    c = fma(c, t, T(-1.0 / 3628800.0));            // -1/10!
    c = fma(c, t, T(1.0 / 40320.0));               // 1/8!
    c = fma(c, t, T(-1.0 / 720.0));                // -1/6!
    c = fma(c, t, T(1.0 / 24.0));                  // 1/4!
    c = fma(c, t, T(-0.5));                        // -1/2!
    c = fma(c, t, T(1));
    return c * c * inv_w;
}

// Godunov |grad phi| (level_set_rk3_redis.f90:341-360) from the one-sided
// slopes times 6 dx, 6 dy, 6 dz (2D: without the last pair); k = 1 / (6 dx), ...: with sigma the sign of
// S0, max(-min(D+, 0), max(D-, 0)) is max(-sigma D+, sigma D-, 0) per direction
// (and max(max(D+, 0), -min(D-, 0)) the same with sigma = -1).  Where S0 is a
// zero of either sign the pseudo-time right-hand side S0 (|grad| - 1) is zero.
template <typename T>
LSMP_DEV T godunov_sig(T xp, T xm, T yp, T ym, T zp, T zm, T s0, T kx, T ky, T kz)
{
    const T sx = copysign(kx, s0), sy = copysign(ky, s0), sz = copysign(kz, s0);
    const T gx = fmax(fmax(-(sx * xp), sx * xm), T(0));
    const T gy = fmax(fmax(-(sy * yp), sy * ym), T(0));
    const T gz = fmax(fmax(-(sz * zp), sz * zm), T(0));
    return sqrt_w(sq(gx) + sq(gy) + sq(gz));
}

template <typename T> LSMP_DEV T godunov_sig(T xp, T xm, T yp, T ym, T s0, T kx, T ky)
{
    const T sx = copysign(kx, s0), sy = copysign(ky, s0);
    const T gx = fmax(fmax(-(sx * xp), sx * xm), T(0));
    const T gy = fmax(fmax(-(sy * yp), sy * ym), T(0));
    return sqrt_n(sq(gx) + sq(gy));
}

// The stage's new value from the pseudo-time RHS l (Shu-Osher form).
template <typename T, int STAGE> LSMP_DEV T rk_stage(T phi_c, T p0, T l, T rdt)
{
    if (STAGE == 1) return phi_c - rdt * l;
    if (STAGE == 2) return T(0.75) * p0 + T(0.25) * (phi_c - rdt * l);
    return p0 * T(1.0 / 3.0) + T(2.0 / 3.0) * (phi_c - rdt * l);
}

// Smoothed Heaviside and delta (ns_solver/others.f90:18-31).
template <typename T> LSMP_DEV void ls_funs(T phi, T ls_wid, T &H, T &D)
{
    const T eps = T(1.0e-12);
    const T pi = T(3.141592653589793238462643383279502884);
    T x = phi / ls_wid;
    if (x > T(1) - eps) {
        H = T(1); D = T(0);
    } else if (x < T(-1) + eps) {
        H = T(0); D = T(0);
    } else {
        H = T(0.5) * ((T(1) + x) + sin(pi * x) / pi);
        D = T(0.5) * (T(1) + cos(pi * x)) / ls_wid;
    }
    H = fmax(fmin(H, T(1)), T(0));
}

// Heaviside used by the shape metric, without the clip (output.f90:233-248).
template <typename T> LSMP_DEV T heavyside(T x)
{
    const T eps = T(1.0e-12);
    const T pi = T(3.141592653589793238462643383279502884);
    if (x > T(1) - eps) return T(1);
    if (x < T(-1) + eps) return T(0);
    return T(0.5) * ((T(1) + x) + sin(pi * x) / pi);
}

// Wave- and block-wide reductions (64-lane wavefronts).
LSMP_DEV double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
LSMP_DEV double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// Block-wide sum of NV doubles; result valid in thread 0.  blockDim.x must be
// a multiple of 64 and at most 1024.
template <int NV> LSMP_DEV void block_sum(double (&v)[NV])
{
    __shared__ double red[16][NV];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = wave_sum(v[q]);
    if (lane == 0)
        for (int q = 0; q < NV; ++q) red[wid][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 0; q < NV; ++q) {
            double s = red[0][q];
            for (int w = 1; w < nw; ++w) s += red[w][q];
            v[q] = s;
        }
    }
    __syncthreads();
}

// Neumaier-compensated FP64 summation: s carries the rounded running sum and
// c the rounding errors of its additions (each recovered exactly), so s + c is
// the sum to about one rounding whatever the number of terms.
LSMP_DEV void csum_add(double &s, double &c, double x)
{
    const double t = s + x;
    c += fabs(s) >= fabs(x) ? (s - t) + x : (x - t) + s;
    s = t;
}

// Block-wide compensated sum of NV (s, c) pairs (blockDim.x a multiple of 64,
// at most 1024): pairs combine by adding their sums with csum_add and their
// compensations plainly; thread 0 gets s[q] = s + c of the block.
template <int NV> LSMP_DEV void block_sum_comp(double (&s)[NV], double (&c)[NV])
{
    __shared__ double red_s[16][NV], red_c[16][NV];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; ++q)
        for (int o = 32; o > 0; o >>= 1) {
            const double s2 = __shfl_xor(s[q], o, 64), c2 = __shfl_xor(c[q], o, 64);
            c[q] += c2;
            csum_add(s[q], c[q], s2);
        }
    if (lane == 0)
        for (int q = 0; q < NV; ++q) {
            red_s[wid][q] = s[q];
            red_c[wid][q] = c[q];
        }
    __syncthreads();
    if (threadIdx.x < NV) {   // a lane per quantity
        const int q = threadIdx.x;
        double ss = red_s[0][q], cc = red_c[0][q];
        for (int w = 1; w < nw; ++w) {
            cc += red_c[w][q];
            csum_add(ss, cc, red_s[w][q]);
        }
        s[0] = ss + cc;
    }
    if (threadIdx.x < 64)
#pragma unroll
        for (int q = NV - 1; q >= 0; --q) s[q] = __shfl(s[0], q, 64);
    __syncthreads();
}

// Compensated sum of the per-block partial triples partial[3 b + q], b < nblk,
// over the whole block (slot b to thread b, b + blockDim.x, ...); the totals
// land in acc of thread 0.  Fixed order: the result does not depend on timing.
LSMP_DEV void sum_partials3(const double *__restrict__ partial, int nblk, double (&acc)[3])
{
    // four slots' loads in flight, then their additions in slot order
    constexpr int AHEAD = 4;
    double cmp[3] = {0.0, 0.0, 0.0};
    acc[0] = acc[1] = acc[2] = 0.0;
    const int bd = blockDim.x;
    for (int b0 = threadIdx.x; b0 < nblk; b0 += AHEAD * bd) {
        double v[AHEAD][3];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int b = b0 + u * bd;
#pragma unroll
            for (int q = 0; q < 3; ++q) v[u][q] = b < nblk ? partial[3 * b + q] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (b0 + u * bd < nblk)
#pragma unroll
                for (int q = 0; q < 3; ++q) csum_add(acc[q], cmp[q], v[u][q]);
    }
    block_sum_comp<3>(acc, cmp);
}

// max of non-negative doubles through their bit patterns (ordered as integers)
LSMP_DEV void atomic_max_nonneg(unsigned long long *p, double v)
{
    atomicMax(p, (unsigned long long)__double_as_longlong(v));
}

LSMP_DEV double block_max(double v)
{
    __shared__ double red[16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int nw = (blockDim.x + 63) >> 6;
    v = wave_max(v);
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < nw; ++w) v = fmax(v, red[w]);
    __syncthreads();
    return v;
}

}  // namespace lsmp
