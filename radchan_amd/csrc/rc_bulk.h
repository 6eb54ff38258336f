/*
 * rc_bulk.h -- the bulk march of the batched solver: one ray per lane, every
 * lane of a wavefront one step at a time.
 *
 * The march is bound by VALU issue, so the ray's state is kept in the form
 * the step consumes, set once at pick-up, reflection or level change:
 *
 *  - the face the ray heads for along y and z as a float (face j at j dy,
 *    exact up to 2^24), the x face and the cell as byte offsets into the
 *    level's arrays, the table row as a byte offset: a step forms no address
 *    and converts no index;
 *  - per axis the value of that index at which the ray has left the grid, so
 *    leaving is one comparison, made only in the branch of the axis crossed;
 *  - lanes without a live ray are masked off the step, and a live ray's
 *    offsets are always a cell's or a wall entry's, so no load has a bound;
 *  - what happens once per ray (the dump tally, the finished ray's sums)
 *    waits until the lane's next pick-up, where it is done for all lanes
 *    that ended since.
 *
 * Every value is the one march_step_thread computes, so the tallies
 * are the plain march's to the bit (but for the sign of a zero).
 *
 * Measured (march kernel, nVar 2, against the step that recomputed indices
 * and addresses and stepped idle lanes too): 256x128x256, 360 bands, photmax
 * 100 200.1 -> 195.6 ms; four snapshots of 64x96x64 and 110x62x90 with BF16
 * tables 51.4 -> 38 ms; param.h's settings on 28x96x128, one run 106.2 -> 97.2
 * ms; with the ray generation, the queue and the exponent as they are now
 * 176.4, 34.5 and 89.8 ms.  A step's straight path is 86 vector instructions.
 * At 256x128x256 the gathers keep the texture-address units 0.88 busy, with
 * the vector issue at 0.75; at three levels (192x128x192) the issue is full.
 */
#ifndef RC_BULK_H
#define RC_BULK_H

#include "rc_march.h"

namespace rc {

/* lane mask <-> per-lane condition, without a vector instruction */
__device__ __forceinline__ bool lane_in(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

/* a load at a byte offset from a wavefront-uniform base */
template <class T> __device__ __forceinline__ T ld_off(const void *base, uint32_t off) {
    return *(const __attribute__((address_space(1))) T *)((rcd::rc_gchar *)base + off);
}

/* values of BulkRay::kt that are no table row: no pair loaded; the ray's next
 * step is a black wall's emission; the ray left through an open (bd 5) face */
enum { KT_NONE = -1, KT_WALL = -2, KT_LOST = -3 };

/* sizes of a grid level and where its x faces and table positions start */
struct BulkDim {
    int im, jm, km;
    uint32_t xoff, poff;
};

struct BulkRay {
    float xp, yp, zp, sx, sy, sz, isx, isy, isz, tra;
    float jf, kf;               /* the y and z face ahead: index jc - f1, kc - f2 */
    float jlim, klim;           /* their values once the ray has left the grid     */
    uint32_t ix4, xlim;         /* the same along x, 4 (xoff + ic - f0)            */
    uint32_t cell4;             /* 4 (poff + cell); at a wall, its entry           */
    int dx4, dcy4, dcz4;        /* steps of ix4 (and cell4) along x, of cell4 along y, z */
    float W, Bi, invBi;
    uint32_t rowb, rankb;       /* byte offsets of the ray's table rows            */
    int kt;                     /* the table pair held in k, or a KT_ value        */
    KbRaw k;
    float fac, dacc;            /* (B - Bi)/Bi of the last step; the tally         */
    int cap;                    /* the wavefront's step count at the level's step cap */
    uint32_t uh;                /* unit number | ray number << 16                  */
    int tid;
    float fx, pos;              /* the x face ahead and the cell's table position   */
    int lev;                    /* several levels: the level, and its spacings     */
    float dy, dz;
};

/* steps to the cap of a level, bounded so that the count cannot overflow */
__device__ __forceinline__ int bulk_cap(int maxs) { return min(maxs, 1 << 30); }

/* what the direction's signs decide at the cell with high x face ix4 and
 * indices (jc, kc): the faces ahead, where the ray leaves the grid, and the
 * cell's steps */
__device__ __forceinline__ void bulk_heads(const BulkDim &d, uint32_t ix4, float jc, float kc, BulkRay &b) {
    const bool nx = b.sx < 0.f, ny = b.sy < 0.f, nz = b.sz < 0.f;
    const int imjm4 = 4 * (int)__umul24((uint32_t)d.im, (uint32_t)d.jm);
    b.dx4 = nx ? -4 : 4;
    b.ix4 = nx ? ix4 - 4u : ix4;
    b.xlim = nx ? 4u * d.xoff - 4u : 4u * (d.xoff + (uint32_t)(d.im + 1));
    b.jf = jc + (ny ? -1.0f : 0.0f);
    b.kf = kc + (nz ? -1.0f : 0.0f);
    b.jlim = ny ? -1.0f : (float)(d.jm + 1);
    b.klim = nz ? -1.0f : (float)(d.km + 1);
    b.dcy4 = ny ? -4 * d.im : 4 * d.im;
    b.dcz4 = nz ? -imjm4 : imjm4;
}

/* the ray's place on a level: cell (ic, jc, kc), direction signs from s */
__device__ __forceinline__ void bulk_place(const BulkDim &d, int ic, int jc, int kc, BulkRay &b) {
    bulk_heads(d, 4u * (d.xoff + (uint32_t)ic), (float)jc, (float)kc, b);
    b.cell4 = 4u * (d.poff + (uint32_t)(ic - 1) +
                    __umul24((uint32_t)d.im, (uint32_t)(jc - 1) + __umul24((uint32_t)d.jm, (uint32_t)(kc - 1))));
}

/* the cell indices back from the bulk form */
__device__ __forceinline__ void bulk_cell(const BulkDim &d, const BulkRay &b, int &ic, int &jc, int &kc) {
    ic = (int)(b.ix4 / 4u - d.xoff) + (b.sx < 0.f ? 1 : 0);
    jc = (int)b.jf + (b.sy < 0.f ? 1 : 0);
    kc = (int)b.kf + (b.sz < 0.f ? 1 : 0);
}

/* The three boundary conditions (the outcomes of boundary_move): a periodic
 * face takes the ray to the opposite end; a specular face turns the
 * component round in the edge cell; a black (or bd 4) face makes the next
 * step the wall's emission at the wall's entry of the position array; a bd 5
 * face loses the ray.  Periodic faces come in pairs, so that test is
 * wavefront-uniform. */
template <class DF>
__device__ __forceinline__ void bulk_left_x(const DevCommon &cm, const DF &dim, BulkRay &b) {
    const BulkDim d = dim();
    const bool lo = b.dx4 < 0;
    if (cm.bd[FW] == 1) {
        const uint32_t w = 4u * (uint32_t)d.im, step = lo ? w : 0u - w;
        b.xp = lo ? cm.Lx : 0.f;
        b.ix4 += step;
        b.cell4 += step;
        return;
    }
    if ((lo ? cm.bd[FW] : cm.bd[FE]) == 3) {
        b.xp = lo ? 0.f : cm.Lx;
        b.sx = -b.sx;
        b.isx = -b.isx;
        b.cell4 -= (uint32_t)b.dx4;
        b.dx4 = -b.dx4;
        b.ix4 += 2u * (uint32_t)b.dx4;
        b.xlim = 8u * d.xoff + 4u * (uint32_t)d.im - b.xlim;
    } else {
        const uint32_t im = (uint32_t)d.im, jm = (uint32_t)d.jm, km = (uint32_t)d.km;
        const uint32_t j0 = (uint32_t)(int)b.jf - (b.sy < 0.f ? 0u : 1u), k0 = (uint32_t)(int)b.kf - (b.sz < 0.f ? 0u : 1u);
        const uint32_t nx = __umul24(jm, km);
        b.cell4 = 4u * (d.poff + __umul24(im, nx) + (lo ? 0u : nx) + j0 + __umul24(jm, k0));
        b.ix4 -= (uint32_t)b.dx4;
        b.kt = KT_WALL;
    }
}

template <class DF>
__device__ __forceinline__ void bulk_left_y(const DevCommon &cm, const DF &dim, BulkRay &b) {
    const BulkDim d = dim();
    const bool lo = b.sy < 0.f;
    if (cm.bd[FS] == 1) {
        const uint32_t w = 4u * __umul24((uint32_t)d.im, (uint32_t)d.jm);
        b.yp = lo ? cm.Ly : 0.f;
        b.jf = lo ? (float)(d.jm - 1) : 1.0f;
        b.cell4 += lo ? w : 0u - w;
        return;
    }
    if ((lo ? cm.bd[FS] : cm.bd[FN]) == 3) {
        b.yp = lo ? 0.f : cm.Ly;
        b.sy = -b.sy;
        b.isy = -b.isy;
        b.cell4 -= (uint32_t)b.dcy4;
        b.dcy4 = -b.dcy4;
        b.jf += lo ? 2.0f : -2.0f;
        b.jlim = (float)d.jm - b.jlim;
    } else {
        const uint32_t im = (uint32_t)d.im, jm = (uint32_t)d.jm, km = (uint32_t)d.km;
        const uint32_t i0 = b.ix4 / 4u - d.xoff - (b.dx4 < 0 ? 0u : 1u), k0 = (uint32_t)(int)b.kf - (b.sz < 0.f ? 0u : 1u);
        const uint32_t nx = __umul24(jm, km), ny = __umul24(im, km);
        b.cell4 = 4u * (d.poff + __umul24(im, nx) + 2u * nx + (lo ? 0u : ny) + i0 + __umul24(im, k0));
        b.kt = KT_WALL;
    }
}

template <class DF>
__device__ __forceinline__ void bulk_left_z(const DevCommon &cm, const DF &dim, BulkRay &b) {
    const BulkDim d = dim();
    const bool lo = b.sz < 0.f;
    if (cm.bd[FB] == 1) {
        const uint32_t w = 4u * __umul24((uint32_t)d.im, __umul24((uint32_t)d.jm, (uint32_t)d.km));
        b.zp = lo ? cm.Lz : 0.f;
        b.kf = lo ? (float)(d.km - 1) : 1.0f;
        b.cell4 += lo ? w : 0u - w;
        return;
    }
    const int bd = lo ? cm.bd[FB] : cm.bd[FT];
    if (bd == 3) {
        b.zp = lo ? 0.f : cm.Lz;
        b.sz = -b.sz;
        b.isz = -b.isz;
        b.cell4 -= (uint32_t)b.dcz4;
        b.dcz4 = -b.dcz4;
        b.kf += lo ? 2.0f : -2.0f;
        b.klim = (float)d.km - b.klim;
    } else if (bd == 5) {
        b.kt = KT_LOST;
        b.cell4 -= (uint32_t)b.dcz4;
    } else {
        const uint32_t im = (uint32_t)d.im, jm = (uint32_t)d.jm, km = (uint32_t)d.km;
        const uint32_t i0 = b.ix4 / 4u - d.xoff - (b.dx4 < 0 ? 0u : 1u), j0 = (uint32_t)(int)b.jf - (b.sy < 0.f ? 0u : 1u);
        const uint32_t nx = __umul24(jm, km), ny = __umul24(im, km), nz = __umul24(im, jm);
        b.cell4 = 4u * (d.poff + __umul24(im, nx) + 2u * (nx + ny) + (lo ? 0u : nz) + i0 + __umul24(im, j0));
        b.kt = KT_WALL;
    }
}

/* the x face ahead and the table position of the ray's cell */
__device__ __forceinline__ void bulk_load(const void *xu, const void *P, BulkRay &b) {
    b.fx = ld_off<float>(xu, b.ix4);
    b.pos = ld_off<float>(P, b.cell4);
}

/* One step of a live ray, whose x face and table position have been loaded
 * (bulk_load, or the step before): the table pair is asked for first, then
 * the next cell's values as soon as the geometry names it, so that those
 * loads are in flight during the absorption.  dy, dz: the level's spacings; xu, P: the bases
 * the offsets count from; dim(): the level's sizes, asked for only where a
 * ray left the grid.  Returns whether the ray's transmissivity has fallen to
 * tol or below (the dump tally is bulk_dump's), `wall` whether this was a
 * wall's emission, which is no step of the reference's march. */
template <int TM, class S, class DF>
__device__ __forceinline__ bool bulk_step(const DevCommon &cm, const S &sn, const DF &dim, const void *xu,
                                          const void *P, float dy, float dz, float tol, bool open, BulkRay &b,
                                          bool &wall) {
    const float fx = b.fx, pos = b.pos;
    wall = b.kt == KT_WALL;
    int t;
    ppos(pos, t, b.k.a);
    if (t != b.kt) {
        if (TM == TAB_BF16) {
            b.k.w = ld_off<uint32_t>(sn.kp16, b.rowb + 4u * (uint32_t)t);
            const rcd::rc_v4f v = ld_off<rcd::rc_v4f>(sn.bp, b.rankb + 16u * (uint32_t)t);
            b.k.q = make_float4(v.x, v.y, v.z, v.w);
        } else {
            const rcd::rc_v4f_a8 v = ld_off<rcd::rc_v4f_a8>(sn.kb, b.rowb + 8u * (uint32_t)t);
            b.k.q = make_float4(v.x, v.y, v.z, v.w);
        }
        b.kt = t;
    }
    /* the three face distances; the segment is their least (no NaN: the
     * directions' reciprocals are finite), ties cross z before y before x */
    const float fy = b.jf * dy, fz = b.kf * dz;
    const float dsx = (fx - b.xp) * b.isx;
    const float dsy = (fy - b.yp) * b.isy;
    const float dsz = (fz - b.zp) * b.isz;
    const float ds = fminf(fminf(dsx, dsy), dsz);
    const bool ex = ds == dsx, ey = ds == dsy, ez = ds == dsz;
    b.xp = ex ? fx : fmaf(ds, b.sx, b.xp);
    b.yp = ey ? fy : fmaf(ds, b.sy, b.yp);
    b.zp = ez ? fz : fmaf(ds, b.sz, b.zp);
    if (ez) {
        b.kf += __builtin_copysignf(1.0f, b.sz);
        b.cell4 += (uint32_t)b.dcz4;
        if (b.kf == b.klim) bulk_left_z(cm, dim, b);
    } else if (ey) {
        b.jf += __builtin_copysignf(1.0f, b.sy);
        b.cell4 += (uint32_t)b.dcy4;
        if (b.jf == b.jlim) bulk_left_y(cm, dim, b);
    } else {
        b.ix4 += (uint32_t)b.dx4;
        b.cell4 += (uint32_t)b.dx4;
        if (b.ix4 == b.xlim) bulk_left_x(cm, dim, b);
        b.fx = ld_off<float>(xu, b.ix4);
    }
    if (!wall) b.pos = ld_off<float>(P, b.cell4);
    /* absorption (phys_core_x), a wall's optical depth infinite */
    float K, B;
    kb_finish<TM>(b.k, K, B);
    float em1, exv;
    expm1_exp_step(K * ds, wall, em1, exv);
    b.fac = (B - b.Bi) * b.invBi;
    b.dacc += ((b.W * b.tra) * em1) * b.fac;
    b.tra = b.tra * exv;
    if (__builtin_expect(open, 0)) {
        asm volatile("");       /* a branch: as selects in every step, 2 % of a BF16 ensemble */
        if (b.kt == KT_LOST && !(b.tra < tol)) {      /* lost: ends without a dump */
            b.tra = 0.f;
            b.fac = 0.f;
        }
    }
    return !(b.tra > tol);
}

/* an ended ray's dump tally: the transmissivity below tol goes to the cell
 * it ended in */
__device__ __forceinline__ float bulk_dump(const BulkRay &b, float tol) {
    return b.tra < tol ? b.dacc - (b.W * b.tra) * b.fac : b.dacc;
}

}  // namespace rc

#endif
