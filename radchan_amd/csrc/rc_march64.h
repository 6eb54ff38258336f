/*
 * rc_march64.h -- the full-FP64 march (param.h floatpoint 1, where the
 * reference compiles myfloat as double: param.h:64-65,158-166): ray
 * geometry, transmissivity, tallies and the per-ray constants in double;
 * the temperature field, the k/Ib tables and the band draws stay single
 * precision, as the reference's textures and float input are.
 *
 * Ray setup here (mc_gpu_noint.cu:115-186, :1381-1441); the march,
 * march_ray (:245-658) with its boundary conditions and the multigrid
 * hand-off (:210-224), is k_rays64's loop.  Every operation is IEEE double (+, -, *, /, sqrt, fma) or
 * the project-written expm1/exp and sin/cos of 2 pi u below, so the CPU
 * oracle's full-FP64 mode reproduces each ray bit for bit.
 */
#ifndef RC_MARCH64_H
#define RC_MARCH64_H

#include "rc_march.h"

namespace rc {

__device__ __forceinline__ double bits2d(uint64_t b) { return __longlong_as_double((long long)b); }

/* expm1(x) and exp(x) for x <= 0: x = n ln2 + r (Cody-Waite, two fma
 * steps), |r| <= ln2/2, expm1(r) by its Taylor series to r^13/13! (Horner),
 * scaled by 2^n, in two factors below 2^-1000 */
__device__ __forceinline__ void expm1_exp_d(double x, double &em1, double &e) {
    if (!(x < 0.0)) { em1 = x; e = 1.0; return; }
    if (x < -745.5) { em1 = -1.0; e = 0.0; return; }
    const double n = floor(x * 1.4426950408889634 + 0.5);
    double r = fma(-n, 6.93147180369123816490e-01, x);
    r = fma(-n, 1.90821492927058770002e-10, r);
    double p = fma(r, 1.0 / 6227020800.0, 1.0 / 479001600.0);
    p = fma(r, p, 1.0 / 39916800.0);
    p = fma(r, p, 1.0 / 3628800.0);
    p = fma(r, p, 1.0 / 362880.0);
    p = fma(r, p, 1.0 / 40320.0);
    p = fma(r, p, 1.0 / 5040.0);
    p = fma(r, p, 1.0 / 720.0);
    p = fma(r, p, 1.0 / 120.0);
    p = fma(r, p, 1.0 / 24.0);
    p = fma(r, p, 1.0 / 6.0);
    p = fma(r, p, 0.5);
    p = fma(r * r, p, r);
    const int ni = (int)n;
    if (ni < -1000) {
        const double s1 = bits2d((uint64_t)(ni + 600 + 1023) << 52);
        e = fma(s1, p, s1) * bits2d((uint64_t)(1023 - 600) << 52);
        em1 = -1.0;
        return;
    }
    const double s1 = bits2d((uint64_t)(ni + 1023) << 52);
    e = fma(s1, p, s1);
    em1 = (ni == 0) ? p : fma(s1, p, s1 - 1.0);
}

/* sin and cos of 2 pi u (u in [0,1], single precision): exact quadrant
 * split of 4u, Taylor polynomials to degree 17 / 18 on |y| <= pi/4 */
__device__ __forceinline__ void sincos2pi_d(float u, double &s, double &c) {
    const double x = 4.0 * (double)u;
    const double m = floor(x + 0.5);
    const double f = x - m;
    const double y = f * 1.5707963267948966;
    const double y2 = y * y;
    double ps = fma(y2, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
    ps = fma(y2, ps, 1.0 / 6227020800.0);
    ps = fma(y2, ps, -1.0 / 39916800.0);
    ps = fma(y2, ps, 1.0 / 362880.0);
    ps = fma(y2, ps, -1.0 / 5040.0);
    ps = fma(y2, ps, 1.0 / 120.0);
    ps = fma(y2, ps, -1.0 / 6.0);
    const double sp = fma(y * y2, ps, y);
    double pc = fma(y2, 1.0 / 6402373705728000.0, -1.0 / 20922789888000.0);
    pc = fma(y2, pc, 1.0 / 87178291200.0);
    pc = fma(y2, pc, -1.0 / 479001600.0);
    pc = fma(y2, pc, 1.0 / 3628800.0);
    pc = fma(y2, pc, -1.0 / 40320.0);
    pc = fma(y2, pc, 1.0 / 720.0);
    pc = fma(y2, pc, -1.0 / 24.0);
    pc = fma(y2, pc, 0.5);
    const double cp = fma(-y2, pc, 1.0);
    switch ((int)m & 3) {
        case 0: s = sp;  c = cp;  break;
        case 1: s = cp;  c = -sp; break;
        case 2: s = -sp; c = -cp; break;
        default: s = -cp; c = sp; break;
    }
}

/* a generated ray: its cell on the finest level, position and direction */
struct Ray64 {
    int ic, jc, kc;
    double xp, yp, zp, sx, sy, sz, isx, isy, isz;
};

/* per-ray constants: the ray's table row (k and Ib pairs of its band and
 * g), weight W = Ibmax ratioI, B(Ti) and its reciprocal */
struct En64 {
    uint32_t row;
    double W, Bi, rBi;
};

/* (B - Bi) / Bi, r = RN(1 / Bi): two residual corrections give the rounded
 * quotient (Markstein 1990), v_div_fixup the quotients of zeros, infinities
 * and NaN; between numbers made of float table entries nothing leaves the
 * normal range in between */
__device__ __forceinline__ double excess64(double B, double Bi, double r) {
    const double a = B - Bi;
    double q = a * r;
    q = fma(fma(-q, Bi, a), r, q);
    q = fma(fma(-q, Bi, a), r, q);
    return __builtin_amdgcn_div_fixup(q, Bi, a);
}

/* where in its row a temperature lies: clamp-to-edge linear interpolation
 * in double (the texture semantics of memory_copy_noint.cu:241-247) */
__device__ __forceinline__ void pos64(const DevSnap &sn, int nT, double T, int &t, double &a) {
    const double pos = (T - sn.Tnb0d) * sn.invdTd;
    if (!(pos > 0.0)) { t = 0; a = 0.0; }
    else if (pos >= (double)(nT - 1)) { t = nT - 1; a = 0.0; }
    else { t = (int)pos; a = pos - (double)t; }
}
/* K and B between two row entries */
__device__ __forceinline__ double lerp64(float v0, float v1, double a) {
    return (double)v0 + a * ((double)v1 - (double)v0);
}
__device__ __forceinline__ void kb64(const DevSnap &sn, const float2 *row, int nT, double T, double &K, double &B) {
    int t;
    double a;
    pos64(sn, nT, T, t, a);
    const float2 v0 = gld(row, t), v1 = gld(row, t + 1);
    K = lerp64(v0.x, v1.x, a);
    B = lerp64(v0.y, v1.y, a);
}

__device__ __forceinline__ void set_dir64(Ray64 &r, double sx, double sy, double sz) {
    r.sx = sx; r.sy = sy; r.sz = sz;
    r.isx = 1.0 / sx; r.isy = 1.0 / sy; r.isz = 1.0 / sz;
}

/* per-ray constants in double (:154-186, :1419-1424) */
__device__ __forceinline__ void energy64(const DevCommon &cm, const DevSnap &sn, uint32_t key, float Ti, bool surface,
                                         int bound, En64 &e) {
    e.row = key * (uint32_t)tab_stride(cm.nT);
    double Ki, Bi, Km, Bm;
    kb64(sn, sn.kb + e.row, cm.nT, (double)Ti, Ki, Bi);
    kb64(sn, sn.kb + e.row, cm.nT, (double)sn.Tmax, Km, Bm);
    e.Bi = Bi;
    e.rBi = 1.0 / Bi;
    e.W = surface ? (bound ? sn.Ibmax_e64 : sn.Ibmax_w64) * (Bi / Bm) : sn.Ibmax64 * (Bi / Bm) * (Ki / Km);
}

/* a fluid ray's start at the centre of cell (i,j,k): direction, position
 * and per-ray constants (kernel_fluid :115-186) */
__device__ __forceinline__ void fluid_setup64(const DevCommon &cm, const DevSnap &sn, int i, int j, int k,
                                              uint32_t cid, int v, int h, uint32_t key, bool have_key, float Ti,
                                              Ray64 &r, En64 &e) {
    const uint32_t tag = TAG_FLUID + 16u * (uint32_t)sn.snap;
    U4 u{0.f, 0.f, 0.f, 0.f};
    if (!have_key || !cm.sampler) u = draw4(cm.k0, cm.k1, (uint32_t)h, (uint32_t)v, cid, tag);
    if (!have_key) key = band_key(cm, sn, false, u.c, u.d);
    if (cm.sampler) {
        const uint4 sh = draw4_bits(cm.k0, cm.k1, SOBOL_SHIFT_H, (uint32_t)v, cid, tag);
        sobol_uniforms((uint32_t)h, sh.x, sh.y, u.a, u.b);
    }
    const double ct = 1.0 - 2.0 * (double)u.b;
    const double st = 2.0 * sqrt((double)u.b * (1.0 - (double)u.b));
    double sn2, cs2;
    sincos2pi_d(u.a, sn2, cs2);
    double sx = ct, sy = st * cs2, sz = st * sn2;
    if (sx == 0.0) sx = (double)1e-10f;
    if (sy == 0.0) sy = (double)1e-10f;
    if (sz == 0.0) sz = (double)1e-10f;
    set_dir64(r, sx, sy, sz);
    r.ic = i; r.jc = j; r.kc = k;
    r.xp = (double)gld(sn.x0, i); r.yp = (double)gld(sn.y0, j); r.zp = (double)gld(sn.z0, k);
    energy64(cm, sn, key, Ti, false, 0, e);
}

/* a ray's start at the centre of wall cell (j,k) (kernel_surface :1381-1462) */
__device__ __forceinline__ void surface_setup64(const DevCommon &cm, const DevSnap &sn, int bound, int j, int k,
                                                uint32_t cid, int v, int h, uint32_t key, bool have_key, float Tw,
                                                Ray64 &r, En64 &e) {
    const U4 u = draw4(cm.k0, cm.k1, (uint32_t)h, (uint32_t)v, cid,
                       (bound ? TAG_EAST : TAG_WEST) + 16u * (uint32_t)sn.snap);
    if (!have_key) key = band_key(cm, sn, true, u.c, u.d);
    const double a = sqrt(1.0 - (double)u.b), b = sqrt((double)u.b);
    double sn2, cs2;
    sincos2pi_d(u.a, sn2, cs2);
    const double st = bound ? a : b;
    double sx = bound ? -b : a, sy = st * cs2, sz = st * sn2;
    if (fabs(sx) <= 1e-10) sx = (double)((float)(1 - 2 * bound) * 1e-10f);
    if (fabs(sy) <= 1e-10) sy = (double)((float)((sy > 0.0) - (sy <= 0.0)) * 1e-10f);
    if (fabs(sz) <= 1e-10) sz = (double)((float)((sz > 0.0) - (sz <= 0.0)) * 1e-10f);
    set_dir64(r, sx, sy, sz);
    r.ic = bound ? cm.imax : 1; r.jc = j; r.kc = k;
    r.xp = bound ? (double)cm.Lx : 0.0; r.yp = (double)gld(sn.y0, j); r.zp = (double)gld(sn.z0, k);
    energy64(cm, sn, key, Tw, true, bound, e);
    /* on-face index adjustment (:1429-1441) */
    const DevLevel &L0 = sn.lev[0];
    const bool f0 = sx < 0.0, f1 = sy < 0.0, f2 = sz < 0.0;
    if (f0 && r.xp == (double)gld(L0.xu, r.ic - 1)) r.ic -= 1;
    if (f1 && r.yp == (double)((float)(r.jc - 1) * L0.dy)) r.jc -= 1;
    if (f2 && r.zp == (double)((float)(r.kc - 1) * L0.dz)) r.kc -= 1;
    if (!f0 && r.xp == (double)gld(L0.xu, r.ic)) r.ic += 1;
    if (!f1 && r.yp == (double)((float)r.jc * L0.dy)) r.jc += 1;
    if (!f2 && r.zp == (double)((float)r.kc * L0.dz)) r.kc += 1;
}

}  // namespace rc

#endif
