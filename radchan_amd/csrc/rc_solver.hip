/*
 * rc_solver.hip -- MI355X (gfx950) narrow-band correlated-k OERM Monte Carlo
 * solver for the radiative source term div(q_r) of a channel flow, a drop-in
 * for RadChan's src/montecarlo path on one GPU.
 *
 * Reference path (RadChan): src/montecarlo/mc_gpu_noint.cu
 *   kernel_fluid :55-243, march_ray :245-658, mc_gpu_ :660-874,
 *   get_results_ :876-1021, find_band :1103-1169, wave_find :1234-1267,
 *   kernel_surface :1316-1482; tables src/montecarlo/memory_copy_noint.cu.
 *
 * Device data layout (all structure-of-arrays in HBM):
 *   per snapshot and grid level: the table positions of the cells
 *   [km][jm][im] (the temperature the reference samples with a texture at
 *   the mapped cell centre, mapped to the table's row coordinate) and of
 *   the black walls (DevLevel); x faces per level;
 *   tables in sorted band ("rank") order: kb[(rank*nQ+g)*S+t] = {k, Ib}
 *   pairs, S = tab_stride(nT), one 16-byte load per march step, the last
 *   row repeated so that the clamped top row needs no branch, then the
 *   fixed-temperature walls' entries.
 *
 * Variants:
 *   plain   -- the reference's launch shape: one thread per emitting cell,
 *              photmax rays in sequence, FP32 per-cell sums, a sort pre-pass
 *              per run (nVar launches of each kernel);
 *   batched -- see rc_batched.hip.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "rc_device.h"
#include "rc_internal.h"
#include "rc_kernels.h"
#include "rc_march.h"
#include "rc_radix.h"
#include "rc_march64.h"

using namespace rcd;

namespace rc {

/* ------------------------------------------------------------------------ */
/* set-up kernels                                                            */

/* linear texture fetch of the ghost-padded temperature volume at
 * unnormalised texel coordinates with clamp-to-edge addressing (the
 * reference's cudaFilterModeLinear + cudaAddressModeClamp texture,
 * memory_copy_noint.cu:131-168): texel i is centred at i + 0.5 */
__device__ float tex3_T(const float *__restrict__ T, int nx, int ny, int nz, float tx, float ty, float tz) {
    const int n[3] = {nx, ny, nz};
    const float crd[3] = {tx, ty, tz};
    int i0[3], i1[3];
    float w[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float b = crd[d] - 0.5f;
        const float fl = floorf(b);
        w[d] = b - fl;
        int lo = (int)fl, hi = lo + 1;
        lo = min(max(lo, 0), n[d] - 1);
        hi = min(max(hi, 0), n[d] - 1);
        i0[d] = lo; i1[d] = hi;
    }
    auto at = [&](int i, int j, int k) { return T[(size_t)i + (size_t)nx * ((size_t)j + (size_t)ny * (size_t)k)]; };
    const float c00 = lerp(at(i0[0], i0[1], i0[2]), at(i1[0], i0[1], i0[2]), w[0]);
    const float c10 = lerp(at(i0[0], i1[1], i0[2]), at(i1[0], i1[1], i0[2]), w[0]);
    const float c01 = lerp(at(i0[0], i0[1], i1[2]), at(i1[0], i0[1], i1[2]), w[0]);
    const float c11 = lerp(at(i0[0], i1[1], i1[2]), at(i1[0], i1[1], i1[2]), w[0]);
    const float c0 = lerp(c00, c10, w[1]);
    const float c1 = lerp(c01, c11, w[1]);
    return lerp(c0, c1, w[2]);
}

/* mapped texel coordinate of coarse index ic at ratio r (:334-336) */
__device__ __forceinline__ float tmap(int ic, int r) { return ((float)ic - 0.5f) * (float)r + 1.0f; }

/* how the table position of a black wall face is found: 0 not a black
 * wall, 1 the field's texture at the wall (adiabatic x walls, bd 4 z
 * walls), 2 the face's fixed temperature */
struct FaceModes {
    int m[6];
};

FaceModes face_modes(const rc_params &p) {
    FaceModes f{};
    for (int s = 0; s < 2; ++s) {
        const int adiab = s ? p.adiabe : p.adiabw;
        f.m[FW + s] = p.bd[FW + s] == 2 ? (adiab == 1 ? 1 : 2) : 0;
        f.m[FS + s] = p.bd[FS + s] == 2 ? 2 : 0;
        f.m[FB + s] = p.bd[FB + s] == 4 ? 1 : (p.bd[FB + s] == 2 ? 2 : 0);
    }
    return f;
}

/* per-level table positions (layout of DevLevel.P): cells at the texture
 * sample of the mapped cell centre (:334-338), adiabatic x walls at texel
 * x = 1.0 / imax + 1.0 (:391-399, :422-430), bd 4 z walls at the adjacent
 * cell's centre plane (:466-475, :504-513), fixed-temperature walls at
 * their face's fixed position */
__global__ void __launch_bounds__(256) k_level_P(const float *__restrict__ T0, int imax, int jmax, int kmax, int im,
                                                 int jm, int km, FaceModes fm, float Tnb0, float invdT, int nT,
                                                 float *__restrict__ P, float *__restrict__ Tout) {
    const int rx = imax / im, ry = jmax / jm, rz = kmax / km;
    const int nx = imax + 2, ny = jmax + 2, nz = kmax + 2;
    const size_t ncell = (size_t)im * jm * km;
    const size_t nfx = (size_t)jm * km, nfy = (size_t)im * km, nfz = (size_t)im * jm;
    const size_t total = level_pos_count(im, jm, km);
    for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < total; id += (size_t)gridDim.x * blockDim.x) {
        if (id < ncell) {
            const int i = (int)(id % im) + 1, j = (int)((id / im) % jm) + 1, k = (int)(id / ((size_t)im * jm)) + 1;
            const float Tc = tex3_T(T0, nx, ny, nz, tmap(i, rx), tmap(j, ry), tmap(k, rz));
            P[id] = table_pos(Tc, Tnb0, invdT, nT);
            if (Tout) Tout[id] = Tc;
            continue;
        }
        size_t q = id - ncell;
        float v = 0.f, tw = 0.f;
        if (q < 2 * nfx) {
            const int b = (int)(q / nfx);
            const size_t r = q % nfx;
            const int j = (int)(r % jm) + 1, k = (int)(r / jm) + 1;
            const int mode = fm.m[FW + b];
            if (mode == 1) {
                const float tx = b ? (float)imax + 1.0f : 1.0f;
                tw = tex3_T(T0, nx, ny, nz, tx, tmap(j, ry), tmap(k, rz));
                v = table_pos(tw, Tnb0, invdT, nT);
            } else if (mode == 2) {
                v = fixed_wall_pos(nT, FW + b);
            }
        } else if ((q -= 2 * nfx) < 2 * nfy) {
            const int b = (int)(q / nfy);
            if (fm.m[FS + b] == 2) v = fixed_wall_pos(nT, FS + b);
        } else {
            q -= 2 * nfy;
            const int b = (int)(q / nfz);
            const size_t r = q % nfz;
            const int i = (int)(r % im) + 1, j = (int)(r / im) + 1;
            const int mode = fm.m[FB + b];
            if (mode == 1) {
                const float tz = b ? (float)kmax + 0.5f : 1.5f;
                tw = tex3_T(T0, nx, ny, nz, tmap(i, rx), tmap(j, ry), tz);
                v = table_pos(tw, Tnb0, invdT, nT);
            } else if (mode == 2) {
                v = fixed_wall_pos(nT, FB + b);
            }
        }
        P[id] = v;
        if (Tout) Tout[id] = tw;
    }
}

/* cell (and adiabatic x-wall) temperatures of a level, e.g. the spline
 * restriction's, to table positions in P (and, for the FP64 path, kept in
 * Tout beside them) */
__global__ void __launch_bounds__(256) k_pos_from_T(const float *__restrict__ Tl, const float *__restrict__ Tw,
                                                    int im, int jm, int km, FaceModes fm, float Tnb0, float invdT,
                                                    int nT, float *__restrict__ P, float *__restrict__ Tout) {
    const size_t ncell = (size_t)im * jm * km, nfx = (size_t)jm * km;
    const size_t total = ncell + (Tw ? 2 * nfx : 0);
    for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < total; id += (size_t)gridDim.x * blockDim.x) {
        if (id < ncell) {
            P[id] = table_pos(Tl[id], Tnb0, invdT, nT);
            if (Tout) Tout[id] = Tl[id];
        } else {
            const size_t q = id - ncell;
            if (fm.m[FW + (int)(q / nfx)] == 1) {
                P[id] = table_pos(Tw[q], Tnb0, invdT, nT);
                if (Tout) Tout[id] = Tw[q];
            }
        }
    }
}

/* k and Ib of every table row at the snapshot's Tmax (the rays' emission
 * weights divide by them): one pass per field instead of one gather, a
 * table position and two interpolations per ray; and entries 3, 7 and 11 of
 * every g CDF of 16 */
__global__ void __launch_bounds__(256) k_rows_derived(DevCommon cm, const DevSnap *__restrict__ snaps) {
    const DevSnap &sn = snaps[blockIdx.y];
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= cm.nB * cm.nQ) return;
    float K, B;
    kb_at(sn, (uint32_t)row, key_rank(cm, (uint32_t)row), cm.nT, sn.Tmax, K, B);
    const_cast<float2 *>(sn.kbm)[row] = make_float2(K, B);
    if (sn.cdf_g4 && row < cm.nB) {
        const float *g = sn.cdf_g + 16 * (size_t)row;
        const_cast<float4 *>(sn.cdf_g4)[row] = make_float4(g[3], g[7], g[11], 0.f);
    }
}

/* ------------------------------------------------------------------------ */
/* the srt enumeration                                                       */

/* the radix sort's LDS: photmax keys (rounded up to 64) twice as 16 bits,
 * then two 256-bucket histograms; within 64 KiB up to 15 872 keys */
__host__ __device__ __forceinline__ bool sort_radix(int P) { return P > 256 && ((P + 63) & ~63) * 4 + 2048 <= 65536; }

/* the Philox stream of sort unit u: cell id, run and tag (explicit
 * (cell id, run, tag) triples, else fluid cells or the two walls' cells of
 * the slab) */
__device__ __forceinline__ void unit_stream(const DevCommon &cm, int u, int surface, const int32_t *ulist,
                                            uint32_t &cid, int &vv, uint32_t &tag) {
    if (ulist) {
        cid = (uint32_t)ulist[3 * u]; vv = ulist[3 * u + 1]; tag = (uint32_t)ulist[3 * u + 2];
    } else if (!surface) {
        cid = (uint32_t)u + (uint32_t)cm.imax * cm.jmax * (cm.zstart - 1); tag = TAG_FLUID;
    } else {
        const int b = u / cm.nsurf;
        cid = (uint32_t)(u % cm.nsurf) + (uint32_t)cm.jmax * (cm.zstart - 1); tag = b ? TAG_EAST : TAG_WEST;
    }
}

/* One workgroup (one wavefront) per (cell, run): draws photmax keys and
 * sorts them: in registers up to 256 keys (an LDS network took 0.53 ms for
 * 262 144 cells of 100 rays, this 0.19), in LDS by a bitonic network above the
 * radix sort's LDS, 15 872 keys, else by the two-pass LSD radix sort the
 * batched kernel uses (8-bit digits; O(photmax) like the reference's
 * histogram enumeration, where the network's stages grow as log^2).  The
 * sorted sequence is the one the reference's histogram enumeration
 * produces (kernel_find :1023-1049 + wave_find :1234-1267): ascending
 * sorted-band rank, then g; equal keys are identical draws, so any correct
 * sort gives the same sequence. */
__global__ void __launch_bounds__(64) k_sort_bands(DevCommon cm, const DevSnap *__restrict__ snaps, int s, int v,
                                                   int surface, int nunit, const int32_t *__restrict__ ulist,
                                                   uint16_t *__restrict__ keys) {
    extern __shared__ uint32_t lds[];
    const DevSnap &sn = snaps[s];
    const int P = cm.photmax;
    const int lane = threadIdx.x;
    if (sort_radix(P)) {
        /* keys in draw order at ka, after the low-byte pass at kb, the two
         * digit histograms after them */
        const int Pr = (P + 63) & ~63;
        uint16_t *const ka = reinterpret_cast<uint16_t *>(lds);
        uint16_t *const kb = ka + Pr;
        uint32_t *const hist = lds + Pr;
        for (int u = blockIdx.x; u < nunit; u += gridDim.x) {
            uint32_t cid, tag;
            int vv = v;
            unit_stream(cm, u, surface, ulist, cid, vv, tag);
            const uint32_t tagx = tag + 16u * (uint32_t)sn.snap;
            for (int w = lane; w < 512; w += 64) hist[w] = 0u;
            __syncthreads();
            for (int h = lane; h < P; h += 64) {
                const U4 r = draw4(cm.k0, cm.k1, (uint32_t)h, (uint32_t)vv, cid, tagx);
                const uint32_t key = band_key(cm, sn, tag != TAG_FLUID, r.c, r.d);
                ka[h] = (uint16_t)key;
                atomicAdd(&hist[key & 255u], 1u);
                atomicAdd(&hist[256u + (key >> 8)], 1u);
            }
            __syncthreads();
            radix_offsets(hist, lane);
            radix_first(ka, kb, hist, P, lane);
            radix_high(kb, ka, hist + 256, P, radix_high_bits(cm.nB * cm.nQ), lane);
            for (int h = lane; h < P; h += 64) keys[(size_t)u * P + h] = ka[h];
            __syncthreads();
        }
        return;
    }
    if (P <= 256) {
        for (int u = blockIdx.x; u < nunit; u += gridDim.x) {
            uint32_t cid, tag;
            int vv = v;
            unit_stream(cm, u, surface, ulist, cid, vv, tag);
            const uint32_t tagx = tag + 16u * (uint32_t)sn.snap;
            auto key = [&](int h) {
                if (h >= P) return 0xFFFFFFFFu;
                const U4 r = draw4(cm.k0, cm.k1, (uint32_t)h, (uint32_t)vv, cid, tagx);
                return band_key(cm, sn, tag != TAG_FLUID, r.c, r.d);
            };
            uint16_t *out = keys + (size_t)u * P;
            if (P <= 128) {
                uint32_t x[2] = {key(lane), key(lane + 64)};
                wave_sort<2>(x, lane);
                for (int r = 0; r < 2; ++r)
                    if (2 * lane + r < P) out[2 * lane + r] = (uint16_t)x[r];
            } else {
                uint32_t x[4] = {key(lane), key(lane + 64), key(lane + 128), key(lane + 192)};
                wave_sort<4>(x, lane);
                for (int r = 0; r < 4; ++r)
                    if (4 * lane + r < P) out[4 * lane + r] = (uint16_t)x[r];
            }
        }
        return;
    }
    int n2 = 1;
    while (n2 < P) n2 <<= 1;
    for (int u = blockIdx.x; u < nunit; u += gridDim.x) {
        uint32_t cid, tag;
        int vv = v;
        unit_stream(cm, u, surface, ulist, cid, vv, tag);
        const uint32_t tagx = tag + 16u * (uint32_t)sn.snap;
        for (int h = threadIdx.x; h < n2; h += blockDim.x) {
            uint32_t key = 0xFFFFFFFFu;
            if (h < P) {
                const U4 r = draw4(cm.k0, cm.k1, (uint32_t)h, (uint32_t)vv, cid, tagx);
                key = band_key(cm, sn, tag != TAG_FLUID, r.c, r.d);
            }
            lds[h] = key;
        }
        __syncthreads();
        for (int k = 2; k <= n2; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = threadIdx.x; i < n2; i += blockDim.x) {
                    const int ixj = i ^ j;
                    if (ixj > i) {
                        const uint32_t a = lds[i], b = lds[ixj];
                        const bool up = (i & k) == 0;
                        if ((a > b) == up) { lds[i] = b; lds[ixj] = a; }
                    }
                }
                __syncthreads();
            }
        for (int h = threadIdx.x; h < P; h += blockDim.x) keys[(size_t)u * P + h] = (uint16_t)lds[h];
        __syncthreads();
    }
}

/* ------------------------------------------------------------------------ */
/* plain variant: the reference's launch shape                               */

__global__ void __launch_bounds__(128) k_fluid_plain(DevCommon cm, const DevSnap *__restrict__ snaps, int s, int v,
                                                     const uint16_t *__restrict__ keys, double *__restrict__ de,
                                                     unsigned long long *__restrict__ stats) {
    const DevSnap &sn = snaps[s];
    int64_t steps = 0;
    int64_t rays = 0;
    for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < cm.ncell; n += gridDim.x * blockDim.x) {
        int i, j, k;
        cell_ijk(cm, n, i, j, k);
        const uint32_t cid = (uint32_t)n + (uint32_t)cm.imax * cm.jmax * (cm.zstart - 1);
        const float Ti = cell_T(cm, sn, i, j, k);
        float acc = 0.f;
        int st = 0;
        for (int h = 0; h < cm.photmax; ++h) {
            const uint32_t key = keys ? (uint32_t)keys[(size_t)n * cm.photmax + h] : 0u;
            acc += fluid_ray<false>(cm, sn, i, j, k, cid, v, h, key, keys != nullptr, Ti, st, nullptr);
        }
        steps += st;
        rays += cm.photmax;
        de[(size_t)n * cm.nVar + v] = (double)acc;
    }
    /* wavefront-reduced counters */
    for (int o = 32; o > 0; o >>= 1) {
        steps += __shfl_xor(steps, o);
        rays += __shfl_xor(rays, o);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&stat_line(stats)[0], (unsigned long long)rays);
        atomicAdd(&stat_line(stats)[1], (unsigned long long)steps);
    }
}

/* plain variant, one launch per band: the rays of sorted band `rank` of
 * every emitting cell (a contiguous range of the cell's sorted keys), added
 * to the cell's FP32 sum acc[n]; launched for every band in rank order, it
 * adds each cell's rays in the order k_fluid_plain does, so the sums are
 * the same to the bit */
__global__ void __launch_bounds__(128) k_fluid_band(DevCommon cm, const DevSnap *__restrict__ snaps, int s, int v,
                                                    int rank, const uint16_t *__restrict__ keys,
                                                    float *__restrict__ acc, unsigned long long *__restrict__ stats) {
    const DevSnap &sn = snaps[s];
    const int P = cm.photmax;
    const uint32_t klo = (uint32_t)rank * (uint32_t)cm.nQ, khi = klo + (uint32_t)cm.nQ;
    int64_t steps = 0, rays = 0;
    for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < cm.ncell; n += gridDim.x * blockDim.x) {
        const uint16_t *kk = keys + (size_t)n * P;
        /* first ray with key >= klo, and with key >= khi */
        int a = 0, b = P;
        while (a < b) { const int m = (a + b) >> 1; if ((uint32_t)kk[m] < klo) a = m + 1; else b = m; }
        int c = a, d = P;
        while (c < d) { const int m = (c + d) >> 1; if ((uint32_t)kk[m] < khi) c = m + 1; else d = m; }
        if (a == c) continue;
        int i, j, k;
        cell_ijk(cm, n, i, j, k);
        const uint32_t cid = (uint32_t)n + (uint32_t)cm.imax * cm.jmax * (cm.zstart - 1);
        const float Ti = cell_T(cm, sn, i, j, k);
        float sum = acc[n];
        int st = 0;
        for (int h = a; h < c; ++h) sum += fluid_ray<false>(cm, sn, i, j, k, cid, v, h, (uint32_t)kk[h], true, Ti, st, nullptr);
        acc[n] = sum;
        steps += st;
        rays += c - a;
    }
    for (int o = 32; o > 0; o >>= 1) {
        steps += __shfl_xor(steps, o);
        rays += __shfl_xor(rays, o);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&stat_line(stats)[0], (unsigned long long)rays);
        atomicAdd(&stat_line(stats)[1], (unsigned long long)steps);
    }
}

__global__ void k_acc_zero(float *__restrict__ acc, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) acc[i] = 0.f;
}

__global__ void k_acc_store(const float *__restrict__ acc, int n, int nVar, int v, double *__restrict__ de) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        de[(size_t)i * nVar + v] = (double)acc[i];
}

__global__ void __launch_bounds__(128) k_surface_plain(DevCommon cm, const DevSnap *__restrict__ snaps, int s, int v,
                                                       const uint16_t *__restrict__ keys, double *__restrict__ de,
                                                       unsigned long long *__restrict__ stats) {
    const DevSnap &sn = snaps[s];
    int64_t steps = 0, rays = 0;
    const int nsurf = cm.nsurf;
    for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < 2 * nsurf; n += gridDim.x * blockDim.x) {
        const int bound = n / nsurf, m = n % nsurf;
        if ((bound == 0 && !cm.adiab[0]) || (bound == 1 && !cm.adiab[1])) continue;
        const int j = m % cm.jmax + 1, k = m / cm.jmax + cm.zstart;
        const uint32_t cid = (uint32_t)m + (uint32_t)cm.jmax * (cm.zstart - 1);
        const float Tw = wall_T(cm, sn, bound, j, k);
        float acc = 0.f;
        int st = 0;
        for (int h = 0; h < cm.photmax; ++h) {
            const uint32_t key = keys ? (uint32_t)keys[(size_t)n * cm.photmax + h] : 0u;
            acc += surface_ray<false>(cm, sn, bound, j, k, cid, v, h, key, keys != nullptr, Tw, st, nullptr);
        }
        steps += st;
        rays += cm.photmax;
        de[(size_t)n * cm.nVar + v] = (double)acc;
    }
    for (int o = 32; o > 0; o >>= 1) {
        steps += __shfl_xor(steps, o);
        rays += __shfl_xor(rays, o);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&stat_line(stats)[0], (unsigned long long)rays);
        atomicAdd(&stat_line(stats)[1], (unsigned long long)steps);
    }
}

/* ------------------------------------------------------------------------ */
/* full-FP64 variant (floatpoint 1)                                          */

/* generated rays of a wavefront */
struct Rec64 {
    double sx[64], sy[64], sz[64], isx[64], isy[64], isz[64], W[64], Bi[64], rBi[64];
    float x[64], y[64], z[64];              /* the start is at single-precision coordinates */
    int ic[64], jc[64], kc[64];
    uint32_t row[64], id[64];
};
/* a ray being marched, handed from a lane to the whole wavefront */
struct Drain64 {
    double xp, yp, zp, sx, sy, sz, isx, isy, isz, tra, W, Bi, rBi, de;
    int ic, jc, kc, cnt, g;
    uint32_t row, id, pad;
};
/* LDS of coop64: factors or terms of the steps, transmissivities before them */
struct Chain64 {
    double x[64], tra[64];
};
/* rays left to a wavefront at which it stops marching them side by side */
constexpr int COOP64 = 8;
struct Lev64 {
    const float *xu, *T;
    int im, jm, km, maxs;
    float dy, dz;
};
__device__ __forceinline__ Lev64 lev64(const DevSnap &sn, int g) {
    const DevLevel &L = sn.lev[g];
    return Lev64{L.xu, sn.T_all + L.poff, L.im, L.jm, L.km, L.maxs, L.dy, L.dz};
}

/* LDS written by some lanes of the wavefront, then read by others */
__device__ __forceinline__ void wave_lds64() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
/* x of another lane of the quad (a DPP quad_perm) */
template <int PERM>
__device__ __forceinline__ double quad64(double x) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    return bits2d(((uint64_t)(uint32_t)__builtin_amdgcn_mov_dpp((int)(b >> 32), PERM, 0xF, 0xF, true) << 32) |
                  (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, PERM, 0xF, 0xF, true));
}

/* what a ray that leaves the grid through `face` (no periodic or specular
 * one) is tallied: a black wall's emission, from a fixed temperature's Ib
 * (the row's entry of the face) or the table at the wall's temperature
 * (adiabatic x walls, bd 4 z walls); nothing if lost */
__device__ __forceinline__ double wall64(const DevCommon &cm, const DevSnap &sn, const Lev64 &L, uint32_t row, int face,
                                         const Ray &r, double W, double tra, double Bi, double rBi) {
    const int bd = cm.bd[face];
    if (bd != 2 && bd != 4) return 0.0;
    double Bw;
    if ((face == FW && cm.adiab[0]) || (face == FE && cm.adiab[1]) || bd == 4) {
        double Kw;
        kb64(sn, sn.kb + row, cm.nT, (double)gld(L.T, wall_index(L, r, face)), Kw, Bw);
    } else {
        Bw = (double)gld(sn.kb, row + (uint32_t)(cm.nT + 1 + 2 * face)).y;
    }
    return W * tra * excess64(Bw, Bi, rBi);
}
/* indices on level g + 1 of those on level g (:215-223) */
__device__ __forceinline__ void coarsen64(const DevSnap &sn, int g, int &ic, int &jc, int &kc) {
    const DevLevel &L = sn.lev[g], &M = sn.lev[g + 1];
    const int ri = L.im / M.im, rj = L.jm / M.jm, rk = L.km / M.km;
    ic = (ic + ri - 1) / ri;
    jc = (jc + rj - 1) / rj;
    kc = (kc + rk - 1) / rk;
}

/* Units u0 .. u0 + nu - 1 (fluid cells, or wall cells of both walls) in runs
 * run0 .. run0 + nv - 1, run v's keys at keys + (v - run0) vkeys: ray q's
 * tally to ray[q], q = ((v - run0) nu + unit) photmax + h, for k_sum_rays64
 * to add up in ray order, which is the sum of a thread that traces its
 * cell's rays in turn, to the bit.  Free of that order, a wavefront takes
 * ranges of rays off a queue (one counter per XCD, as the batched kernel's),
 * generates them 64 at a time into LDS and has its lanes take the next
 * whenever REFILL64 of them are idle; its last COOP64 rays it marches
 * together (coop64).  (MG: several levels.)
 *
 * 64^3, 100 rays, 2 runs (302 M steps, the longest ray 21 000): a thread per
 * cell, its wavefront waiting for the longest of 64 rays and at last for
 * the longest of all, took 2 x 17.3 ms; both runs in one launch now take 7.6
 * ms, of which 4.6 are the bulk (FP64 arithmetic, about 150 instructions per
 * step) and the rest the last rays: a lone lane's step takes about 3000
 * clocks, coop64's 400 (15.3 ms per run without it).  REFILL64 4 to 16 and
 * STEPS64 1 to 4 are within 5 %; COOP64 4 to 16 within 1 %; 3 wavefronts per
 * SIMD instead of 4 (128 registers, 10 or 11 of them spilled, 46 with several
 * levels) 2 % slower; stopping the wavefront for a ray of over 1000 steps to
 * march it together at once, the same.  Thread per cell -> now elsewhere: 64^3,
 * 200 rays, 8 runs 201 -> 43 ms; 192x128x192, 100 rays, one run, one level
 * 319 -> 107 (two launches, the tallies' 2 GiB), three levels with walls
 * 108 -> 101, 8 runs 857 -> 797; param.h's settings on 28x96x128, 2 runs,
 * whose rays end after 3.4 steps and fill the lanes either way, 601 -> 578. */
constexpr int REFILL64 = 8, STEPS64 = 2;
static_assert(COOP64 * sizeof(Drain64) + sizeof(Chain64) <= sizeof(Rec64), "the drain's LDS");

__device__ __forceinline__ int uni64(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double lane64(double x, int l) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    return bits2d(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), l) << 32) |
                  (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l));
}

/* The rest of one ray by the whole wavefront, 64 steps at a time: the
 * geometry, which is serial, lane 4 q + a the axis a (every quad the same),
 * lane n keeping step n's cell and path; then table, exponential and excess
 * of all steps at once; then the transmissivities and the tally in step
 * order by one lane.  The operations on the ray are those of the loop in
 * k_rays64.  Returns the steps. */
template <bool MG>
__device__ int coop64(const DevCommon &cm, const DevSnap &sn, const Drain64 &r, uint32_t bds, double tl, Chain64 &ch,
                      double &de_out) {
    const int lane = threadIdx.x & 63, a = lane & 3;
    const double W = r.W, Bi = r.Bi, rBi = r.rBi;
    double tra = r.tra, de = r.de;
    /* the axis' position and direction; lane 3 of a quad is never crossed
     * (its face, position and direction stay 1e300, 0, 0 and 1) */
    double p = a == 0 ? r.xp : (a == 1 ? r.yp : (a == 2 ? r.zp : 0.0));
    double s = a == 0 ? r.sx : (a == 1 ? r.sy : (a == 2 ? r.sz : 0.0));
    double is = a == 0 ? r.isx : (a == 1 ? r.isy : (a == 2 ? r.isz : 1.0));
    int cnt = uni64(r.cnt), g = MG ? uni64(r.g) : 0, steps = 0;
    const uint32_t row = (uint32_t)uni64((int)r.row);
    Lev64 L = lev64(sn, g);
    /* What a step needs first is ready before it: the face ahead, f, and the
     * one after it, fn (index jn, as a float; past: its value once the grid
     * is left, lane 3: none; xn: the x axis').  u: the axis' index step, cs
     * its share of the cell index and du the share's step. */
    double f, fn;
    float xn, jn, past, uf, dyz;
    int nf, u, du, cs;
    auto neg = [&]() { return s < 0.0 ? 1 : 0; };
    auto xface = [&](int q) { return gld32(L.xu, (uint32_t)min(max(q, 0), L.im)); };
    auto enter = [&](int ci) {                  /* from the axis' cell index */
        const int j = ci - neg(), stride = a == 0 ? 1 : (a == 1 ? L.im : L.im * L.jm);
        nf = a == 0 ? L.im : (a == 1 ? L.jm : L.km);
        dyz = a == 1 ? L.dy : L.dz;
        u = 1 - 2 * neg();
        uf = (float)u;
        du = a == 3 ? 0 : u * stride;
        cs = a == 3 ? 0 : (ci - 1) * stride;
        past = a == 3 ? -9.f : (neg() ? -2.f : (float)(nf + 2));
        jn = (float)(j + u);
        f = a == 0 ? (double)xface(j) : (a == 3 ? 1e300 : (double)((float)j * dyz));
        xn = xface(j + u);
        fn = (double)(a == 0 ? xn : jn * dyz);
    };
    auto cell = [&]() { return (int)jn - u + neg(); };
    enter(a == 0 ? r.ic : (a == 1 ? r.jc : r.kc));
    for (;;) {
        int n = 0, end = -1;
        double pds = 0.0;
        uint32_t pc = 0;
        int nmax = min(64, L.maxs - cnt);
        do {
            const double d = (f - p) * is;
            double m = d, o = quad64<0xB1>(d);
            m = o < m ? o : m;
            o = quad64<0x4E>(m);
            m = o < m ? o : m;
            const bool eq = d == m;
            const int ea = (int)__ballot(eq) & 7;
            const double fo = f, pm = fma(m, s, p);
            f = eq ? fn : f;
            p = eq ? fo : pm;
            const int cq = cs + quad_lane<0xB1>(cs);
            const int c = cq + quad_lane<0x4E>(cq);
            if (lane == n) { pds = m; pc = (uint32_t)c; }
            ++n;
            jn += eq ? uf : 0.f;
            cs += eq ? du : 0;
            if (__builtin_expect(((0x14 >> ea) & 1) == 0, 0)) {
                /* x crossed, or faces of several axes at once: the tie
                 * rules, z before y before x (z if nothing compares) */
                const int ax = (0xAA52 >> (2 * ea)) & 3;
                const bool cr = a == ax;
                f = cr ? fn : fo;
                jn += cr == eq ? 0.f : (cr ? uf : -uf);
                cs += cr == eq ? 0 : (cr ? du : -du);
                if (ax == 0) xn = xface((int)jn);
            }
            fn = (double)(a == 0 ? xn : jn * dyz);
            const unsigned long long out = __ballot(jn == past);
            if (__builtin_expect(out != 0ull, 0)) {
                const int ax = (int)__builtin_ctzll(out) & 3, lo = __builtin_amdgcn_readlane(neg(), ax);
                const int face = 2 * ax + 1 - lo, bd = (int)(bds >> (4 * face)) & 15;
                if (bd == 1 || bd == 3) {                         /* periodic, specular: on from one of the sides */
                    const bool hi = (lo != 0) == (bd == 1);
                    int ci = cell();
                    if (a == ax) {
                        p = hi ? (double)(a == 0 ? cm.Lx : (a == 1 ? cm.Ly : cm.Lz)) : 0.0;
                        s = bd == 3 ? -s : s;
                        is = bd == 3 ? -is : is;
                        ci = hi ? nf : 1;
                    }
                    enter(ci);
                } else {
                    end = face;
                    nmax = n;
                }
            }
        } while (n < nmax);
        /* attenuation of the block's steps (:358-370) */
        double em = 0.0, ex = 1.0, fac = 0.0;
        if (lane < n) {
            int t;
            double al;
            pos64(sn, cm.nT, (double)gld(L.T, pc), t, al);
            const float2 v0 = gld(sn.kb, row + t), v1 = gld(sn.kb, row + t + 1);
            const double K = lerp64(v0.x, v1.x, al), B = lerp64(v0.y, v1.y, al), x = K * pds;
            fac = excess64(B, Bi, rBi);
            expm1_exp_d(-x, em, ex);
        }
        ch.x[lane] = ex;                                /* (1 beyond n) */
        wave_lds64();
        if (lane == 0)
            for (int k = 0; k < n; k += 8) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    ch.tra[k + q] = tra;
                    tra = tra * ch.x[k + q];
                }
            }
        wave_lds64();
        const double trb = ch.tra[lane], tral = trb * ex, lastt = W * tral * fac;
        const unsigned long long stop = __ballot(lane < n && !(tral > tl));
        const int m = stop ? (int)__builtin_ctzll(stop) + 1 : n;
        ch.x[lane] = lane < m ? W * trb * (-em) * fac : 0.0;
        wave_lds64();
        if (lane == 0)
            for (int k = 0; k < m; k += 8) {
#pragma unroll
                for (int q = 0; q < 8; ++q) de -= ch.x[k + q];
            }
        wave_lds64();
        de = lane64(de, 0);
        tra = lane64(tra, 0);
        if (stop) {
            tra = lane64(tral, m - 1);
            if (tra < tl) {
                de -= lane64(lastt, m - 1);
                tra = 0.0;
            }
        }
        steps += m;
        cnt += m;
        if (m == n && end >= 0) {
            const int ci = cell();
            const Ray rr{__builtin_amdgcn_readlane(ci, 0), __builtin_amdgcn_readlane(ci, 1), __builtin_amdgcn_readlane(ci, 2),
                         0, 0, 0};
            de -= wall64(cm, sn, L, row, end, rr, W, tra, Bi, rBi);
            break;
        }
        if (stop) break;
        if (cnt >= L.maxs) {
            if (!MG || g >= cm.grid_num - 1) break;
            const int ci = cell();
            int ic = __builtin_amdgcn_readlane(ci, 0), jc = __builtin_amdgcn_readlane(ci, 1),
                kc = __builtin_amdgcn_readlane(ci, 2);
            coarsen64(sn, g, ic, jc, kc);
            g += 1;
            cnt = 0;
            L = lev64(sn, g);
            enter(a == 0 ? ic : (a == 1 ? jc : kc));
        }
    }
    de_out = de;
    return steps;
}

template <bool SURF, bool MG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_rays64(DevCommon cm, const DevSnap *__restrict__ snaps, int s, int run0, int nv, const uint16_t *__restrict__ keys,
         size_t vkeys, int u0, int nu, int *__restrict__ queue, double *__restrict__ ray,
         unsigned long long *__restrict__ stats) {
    __shared__ Rec64 recs[4];
    const DevSnap &sn = snaps[s];
    const int lane = threadIdx.x & 63;
    Rec64 &q = recs[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
    const uint32_t P = (uint32_t)cm.photmax, total = (uint32_t)nv * (uint32_t)nu * P;
    const double tl = (double)(SURF ? cm.tollS : cm.toll);
    const Lev64 L0 = lev64(sn, 0);
    uint32_t bds = 0;                       /* 4 bits per face */
#pragma unroll
    for (int f = 0; f < 6; ++f) bds |= (uint32_t)cm.bd[f] << (4 * f);

    /* wavefront state: the queue's range, the generated rays */
    const int pwaves = max((int)gridDim.x * 4 / QPARTS, 1);
    int part = (int)(blockIdx.x % QPARTS), ptries = 0, plast = 0;
    uint32_t gpos = 0, gend = 0;
    int qn = 0, qh = 0;
    unsigned long long live = 0ull;
    int64_t steps = 0;

    /* lane state */
    bool alive = false;
    int ic = 1, jc = 1, kc = 1, cnt = 0, g = 0, f0 = 0, f1 = 0, f2 = 0, t = 0;
    double xp = 0, yp = 0, zp = 0, sx = 0, sy = 0, sz = 0, isx = 0, isy = 0, isz = 0, tra = 0, W = 0, Bi = 1, rBi = 1,
           de = 0, ta = 0;
    uint32_t row = 0, id = 0;
    float fxn = 0.f;
    float2 v0 = make_float2(0.f, 0.f), v1 = v0;
    Lev64 L = L0;

    /* the cell's temperature and the x face ahead, then its table entries */
    auto cell = [&]() {
        fxn = gld(L.xu, (uint32_t)(ic - f0));
        return gld(L.T, (uint32_t)(ic - 1) + (uint32_t)L.im * ((uint32_t)(jc - 1) + (uint32_t)L.jm * (uint32_t)(kc - 1)));
    };
    auto entries = [&](float T) {
        pos64(sn, cm.nT, (double)T, t, ta);
        v0 = gld(sn.kb, row + (uint32_t)t);
        v1 = gld(sn.kb, row + (uint32_t)t + 1u);
    };

    for (;;) {
        const int idle = 64 - __popcll(live);
        if (idle >= REFILL64) {
            if (qn == 0 && part >= 0) {
                while (gpos >= gend && part >= 0) {
                    const uint32_t pb = (uint32_t)((uint64_t)total * part / QPARTS);
                    const uint32_t pe = (uint32_t)((uint64_t)total * (part + 1) / QPARTS);
                    const int ask = min(max((int)((pe - pb) - plast) / (2 * pwaves), 64), 1024) & ~63;
                    int c0 = 0;
                    if (lane == 0) {
                        if (ptries) c0 = __hip_atomic_load(&queue[part * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if ((uint32_t)c0 < pe - pb) c0 = atomicAdd(&queue[part * QSTRIDE], ask);
                    }
                    c0 = __builtin_amdgcn_readfirstlane(c0);
                    if ((uint32_t)c0 < pe - pb) {
                        plast = c0 + ask;
                        gpos = pb + c0;
                        gend = min(gpos + ask, pe);
                    } else {
                        part = (part + 1) % QPARTS;
                        plast = 0;
                        if (++ptries >= QPARTS) part = -1;
                    }
                }
                if (gpos < gend) {
                    qn = (int)min(gend - gpos, 64u);
                    qh = 0;
                    if (lane < qn) {
                        const uint32_t x = gpos + lane, un = x / P, vi = un / (uint32_t)nu;
                        const int v = run0 + (int)vi, n = u0 + (int)(un - vi * (uint32_t)nu);
                        const int h = (int)(x - un * P);
                        const uint32_t key = keys ? (uint32_t)keys[vi * vkeys + (size_t)n * P + h] : 0u;
                        Ray64 r;
                        En64 e;
                        if (SURF) {
                            const int bound = n / cm.nsurf, w = n % cm.nsurf;
                            const int j = w % cm.jmax + 1, k = w / cm.jmax + cm.zstart;
                            const uint32_t cid = (uint32_t)(w + cm.jmax * (cm.zstart - 1));
                            surface_setup64(cm, sn, bound, j, k, cid, v, h, key, keys != nullptr,
                                            wall_T(cm, sn, bound, j, k), r, e);
                        } else {
                            int i, j, k;
                            cell_ijk(cm, n, i, j, k);
                            const uint32_t cid = (uint32_t)n + (uint32_t)cm.imax * cm.jmax * (cm.zstart - 1);
                            fluid_setup64(cm, sn, i, j, k, cid, v, h, key, keys != nullptr, cell_T(cm, sn, i, j, k), r, e);
                        }
                        q.sx[lane] = r.sx; q.sy[lane] = r.sy; q.sz[lane] = r.sz;
                        q.isx[lane] = r.isx; q.isy[lane] = r.isy; q.isz[lane] = r.isz;
                        q.x[lane] = (float)r.xp; q.y[lane] = (float)r.yp; q.z[lane] = (float)r.zp;
                        q.W[lane] = e.W; q.Bi[lane] = e.Bi; q.rBi[lane] = e.rBi;
                        q.ic[lane] = r.ic; q.jc[lane] = r.jc; q.kc[lane] = r.kc;
                        q.row[lane] = e.row; q.id[lane] = x;
                    }
                    gpos += qn;
                    wave_lds64();
                }
            }
            if (qn) {
                const int o = __builtin_amdgcn_mbcnt_hi((uint32_t)(~live >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)~live, 0u));
                if (!alive && o < qn) {
                    const int w = qh + o;
                    sx = q.sx[w]; sy = q.sy[w]; sz = q.sz[w];
                    isx = q.isx[w]; isy = q.isy[w]; isz = q.isz[w];
                    xp = (double)q.x[w]; yp = (double)q.y[w]; zp = (double)q.z[w];
                    W = q.W[w]; Bi = q.Bi[w]; rBi = q.rBi[w];
                    ic = q.ic[w]; jc = q.jc[w]; kc = q.kc[w];
                    row = q.row[w]; id = q.id[w];
                    f0 = sx < 0.0; f1 = sy < 0.0; f2 = sz < 0.0;
                    tra = 1.0;
                    de = 0.0;
                    cnt = 0;
                    alive = true;                           /* (toll < 1) */
                    if (MG) { g = 0; L = L0; }
                    entries(cell());
                }
                const int took = min(idle, qn);
                qn -= took;
                qh += took;
                wave_lds64();
            } else if (64 - idle <= COOP64) {
                break;
            }
        }
        for (int k = 0; k < STEPS64; ++k) {
            live = __ballot(alive);
            steps += __popcll(live);
            if (!alive) continue;
            /* one step of march_ray (one iteration of the loop at
             * mc_gpu_noint.cu:252-654) */
            const double fx = (double)fxn;
            const double fy = (double)((float)(jc - f1) * L.dy);
            const double fz = (double)((float)(kc - f2) * L.dz);
            const double dsx = (fx - xp) * isx, dsy = (fy - yp) * isy, dsz = (fz - zp) * isz;
            double ds = dsx;
            if (ds > dsy) ds = dsy;
            if (ds > dsz) ds = dsz;
            xp = (ds == dsx) ? fx : fma(ds, sx, xp);
            yp = (ds == dsy) ? fy : fma(ds, sy, yp);
            zp = (ds == dsz) ? fz : fma(ds, sz, zp);
            /* one index along the crossed axis, with the tie rules */
            const bool cx = dsx < dsy && dsx < dsz, cy = !(dsx < dsy) && dsy < dsz;
            const int d = cx ? f0 : (cy ? f1 : f2);
            ic += cx ? 1 - 2 * d : 0;
            jc += cy ? 1 - 2 * d : 0;
            kc += (cx || cy) ? 0 : 1 - 2 * d;
            const uint32_t at = (uint32_t)(cx ? ic : (cy ? jc : kc)) - 1u, lim = (uint32_t)(cx ? L.im : (cy ? L.jm : L.km));
            int end = -1;                           /* the face the ray ends at */
            if (at >= lim) {
                const int face = (cx ? FW : (cy ? FS : FB)) + (d ? 0 : 1);
                const int bd = (int)(bds >> (4 * face)) & 15;
                if (bd == 1 || bd == 3) {                         /* periodic, specular: on from one of the sides */
                    const bool hi = (d != 0) == (bd == 1);
                    const int ni = hi ? (int)lim : 1;
                    const double np = hi ? (double)(cx ? cm.Lx : (cy ? cm.Ly : cm.Lz)) : 0.0;
                    ic = cx ? ni : ic;
                    jc = cy ? ni : jc;
                    kc = (cx || cy) ? kc : ni;
                    xp = cx ? np : xp;
                    yp = cy ? np : yp;
                    zp = (cx || cy) ? zp : np;
                    if (bd == 3) {
                        if (cx) { sx = -sx; isx = -isx; f0 = sx < 0.0; }
                        else if (cy) { sy = -sy; isy = -isy; f1 = sy < 0.0; }
                        else { sz = -sz; isz = -isz; f2 = sz < 0.0; }
                    }
                } else {
                    end = face;
                }
            }
            const float2 w0 = v0, w1 = v1;
            const double wa = ta;
            float Tn = 0.f;
            if (end < 0) Tn = cell();
            /* attenuation and the reciprocity tally (:358-370) */
            const double K = lerp64(w0.x, w1.x, wa), B = lerp64(w0.y, w1.y, wa);
            const double x = K * ds, fac = excess64(B, Bi, rBi);
            double em, ex;
            expm1_exp_d(-x, em, ex);
            const double wta = W * tra * (-em);
            de -= wta * fac;
            tra = tra * ex;
            if (tra < tl) {
                de -= W * tra * fac;
                tra = 0.0;
            }
            if (end >= 0) {
                de -= wall64(cm, sn, L, row, end, Ray{ic, jc, kc, f0, f1, f2}, W, tra, Bi, rBi);
                tra = 0.0;
            }
            cnt += 1;
            alive = tra > tl;
            if (cnt >= L.maxs && alive) {
                /* still alive after the level's cap (:210-224): on to the
                 * next level, indices coarsened (:215-223) */
                alive = MG && g < cm.grid_num - 1;
                if (alive) {
                    coarsen64(sn, g, ic, jc, kc);
                    g += 1;
                    cnt = 0;
                    L = lev64(sn, g);
                    Tn = cell();
                }
            }
            if (alive) entries(Tn);
            else ray[id] = de;
        }
        live = __ballot(alive);
    }
    /* nothing left to generate and few rays marching: one after the other */
    Drain64 *dr = reinterpret_cast<Drain64 *>(&q);
    Chain64 &ch = *reinterpret_cast<Chain64 *>(dr + COOP64);
    if (alive) {
        const int o = __builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0u));
        dr[o] = Drain64{xp, yp, zp, sx, sy, sz, isx, isy, isz, tra, W, Bi, rBi, de, ic, jc, kc, cnt, g, row, id, 0u};
    }
    wave_lds64();
    const int nd = __popcll(live);
    for (int o = 0; o < nd; ++o) {
        double sum;
        steps += coop64<MG>(cm, sn, dr[o], bds, tl, ch, sum);
        if (lane == 0) ray[dr[o].id] = sum;
    }
    if (lane == 0) atomicAdd(&stat_line(stats)[1], (unsigned long long)steps);
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&stat_line(stats)[0], (unsigned long long)total);
}

/* each (unit, run)'s tallies added in ray order */
__global__ void __launch_bounds__(128) k_sum_rays64(const double *__restrict__ ray, int u0, int nu, int P, int nVar,
                                                    int run0, int nv, double *__restrict__ de) {
    for (int w = blockIdx.x * blockDim.x + threadIdx.x; w < nv * nu; w += gridDim.x * blockDim.x) {
        const int vi = w / nu, n = w - vi * nu;
        const double *r = ray + (size_t)w * P;
        double acc = 0.0;
#pragma unroll 8
        for (int h = 0; h < P; ++h) acc += r[h];
        de[(size_t)(u0 + n) * nVar + run0 + vi] = acc;
    }
}

/* traced rays: rays[5*q] = (i or bound, j, k, v, h); unit[q] indexes keys */
__global__ void __launch_bounds__(64) k_trace(DevCommon cm, const DevSnap *__restrict__ snaps, int surface,
                                              const int32_t *__restrict__ rays, const int32_t *__restrict__ unit,
                                              int n, const uint16_t *__restrict__ keys, rc_ray *__restrict__ out) {
    const DevSnap &sn = snaps[0];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int a = rays[5 * q], j = rays[5 * q + 1], k = rays[5 * q + 2], v = rays[5 * q + 3], h = rays[5 * q + 4];
    const bool hk = keys != nullptr;
    const uint32_t key = hk ? (uint32_t)keys[(size_t)unit[q] * cm.photmax + h] : 0u;
    int st = 0;
    if (!surface) {
        const uint32_t cid = (uint32_t)((a - 1) + cm.imax * ((j - 1) + cm.jmax * (k - 1)));
        fluid_ray<true>(cm, sn, a, j, k, cid, v, h, key, hk, cell_T(cm, sn, a, j, k), st, &out[q]);
    } else {
        const uint32_t cid = (uint32_t)((j - 1) + cm.jmax * (k - 1));
        surface_ray<true>(cm, sn, a, j, k, cid, v, h, key, hk, wall_T(cm, sn, a, j, k), st, &out[q]);
    }
}

/* mean over runs and the reference's variance 1/((n-1/2)(n-1)) sum (x-m)^2
 * (mc_gpu_noint.cu:234-239), reported as its square root (:984); 0 for a
 * single run */
__global__ void k_finalize(const double *__restrict__ de, int n, int nVar, float *__restrict__ mean,
                           float *__restrict__ sdev) {
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        double m = 0.0;
        for (int v = 0; v < nVar; ++v) m += de[(size_t)c * nVar + v];
        m /= nVar;
        double var = 0.0;
        if (nVar > 1) {
            for (int v = 0; v < nVar; ++v) {
                const double d = de[(size_t)c * nVar + v] - m;
                var += d * d;
            }
            var = var / (nVar - 0.5) / (nVar - 1);
        }
        mean[c] = (float)m;
        sdev[c] = (float)sqrt(var);
    }
}

/* ------------------------------------------------------------------------ */
/* launchers used by the session code                                        */

void launch_level_P(hipStream_t st, const float *T0, const rc_params &p, int g, float Tnb0, float invdT, int nT,
                    float *P, float *Tout) {
    const size_t n = level_pos_count(p.maxi[g], p.maxj[g], p.maxk[g]);
    const int blocks = (int)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_level_P, dim3(blocks), dim3(256), 0, st, T0, p.imax, p.jmax, p.kmax, p.maxi[g], p.maxj[g],
                       p.maxk[g], face_modes(p), Tnb0, invdT, nT, P, Tout);
}

void launch_pos_from_T(hipStream_t st, const rc_params &p, int g, const float *Tl, const float *Tw, float Tnb0,
                       float invdT, int nT, float *P, float *Tout) {
    const size_t n = (size_t)p.maxi[g] * p.maxj[g] * p.maxk[g] + (size_t)2 * p.maxj[g] * p.maxk[g];
    const int blocks = (int)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_pos_from_T, dim3(blocks), dim3(256), 0, st, Tl, Tw, p.maxi[g], p.maxj[g], p.maxk[g],
                       face_modes(p), Tnb0, invdT, nT, P, Tout);
}

void launch_rows_derived(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int nsnap) {
    hipLaunchKernelGGL(k_rows_derived, dim3((cm.nB * cm.nQ + 255) / 256, nsnap), dim3(256), 0, st, cm, snaps);
}

void launch_sort(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int s, int v, int surface, int nunit,
                 const int32_t *ulist, uint16_t *keys) {
    int n2 = 1;
    while (n2 < cm.photmax) n2 <<= 1;
    const size_t lds = sort_radix(cm.photmax) ? (size_t)((cm.photmax + 63) & ~63) * 4 + 2048
                       : cm.photmax <= 256       ? 0
                                                 : (size_t)n2 * 4;
    const int blocks = std::min(nunit, 1 << 20);
    hipLaunchKernelGGL(k_sort_bands, dim3(blocks), dim3(64), lds, st, cm, snaps, s, v, surface, nunit,
                       ulist, keys);
}

void launch_fluid_plain(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int s, int v, const uint16_t *keys,
                        double *de, unsigned long long *stats) {
    const int blocks = std::max(1, std::min((cm.ncell + 127) / 128, 1 << 20));
    hipLaunchKernelGGL(k_fluid_plain, dim3(blocks), dim3(128), 0, st, cm, snaps, s, v, keys, de, stats);
}

void launch_fluid_bands(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int s, int v, const uint16_t *keys,
                        float *acc, double *de, unsigned long long *stats) {
    const int blocks = std::max(1, std::min((cm.ncell + 127) / 128, 1 << 20));
    const int zb = std::max(1, std::min((cm.ncell + 255) / 256, 65536));
    hipLaunchKernelGGL(k_acc_zero, dim3(zb), dim3(256), 0, st, acc, cm.ncell);
    for (int rank = 0; rank < cm.nB; ++rank)
        hipLaunchKernelGGL(k_fluid_band, dim3(blocks), dim3(128), 0, st, cm, snaps, s, v, rank, keys, acc, stats);
    hipLaunchKernelGGL(k_acc_store, dim3(zb), dim3(256), 0, st, acc, cm.ncell, cm.nVar, v, de);
}

void launch_surface_plain(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int s, int v,
                          const uint16_t *keys, double *de, unsigned long long *stats) {
    const int blocks = std::max(1, std::min((2 * cm.nsurf + 127) / 128, 1 << 20));
    hipLaunchKernelGGL(k_surface_plain, dim3(blocks), dim3(128), 0, st, cm, snaps, s, v, keys, de, stats);
}

/* Input check and Tmax of a temperature field (imax+2)(jmax+2)(kmax+2) on
 * the device: out[0] |= 1 when an entry (ghosts included) is not a
 * positive finite number; out[1] = the largest interior temperature and
 * x-wall midpoint (T_0 + T_1)/2, (T_imax + T_imax+1)/2 of the interior rows
 * (mc_gpu_noint.cu:696-710), as float bits: positive floats order as their
 * bits.  out zero on entry. */
__global__ void __launch_bounds__(256) k_field_scan(const float *__restrict__ T, int imax, int jmax, int kmax,
                                                    uint32_t *__restrict__ out) {
    const uint32_t nx = (uint32_t)imax + 2u, ny = (uint32_t)jmax + 2u;
    const size_t n = (size_t)nx * ny * (size_t)(kmax + 2);
    uint32_t bad = 0u, m = 0u;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const float t = T[q];
        bad |= (t > 0.f && t <= 3.40282347e38f) ? 0u : 1u;
        const uint32_t row = (uint32_t)(q / nx), i = (uint32_t)(q - (size_t)row * nx);
        const uint32_t j = row % ny, k = row / ny;
        if (j >= 1u && j <= (uint32_t)jmax && k >= 1u && k <= (uint32_t)kmax && i >= 1u && i <= (uint32_t)imax) {
            float c = t;
            if (i == 1u) c = fmaxf(c, (T[q - 1] + t) * 0.5f);
            if (i == (uint32_t)imax) c = fmaxf(c, (t + T[q + 1]) * 0.5f);
            m = max(m, __float_as_uint(c));
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        bad |= (uint32_t)__shfl_xor((int)bad, o);
        m = max(m, (uint32_t)__shfl_xor((int)m, o));
    }
    /* the line of out takes about 90 atomics per microsecond: a wavefront
     * adds its maximum only where it exceeds the one there (256x128x256:
     * 377 us with one atomic per wavefront, now 62 us) */
    if ((threadIdx.x & 63) == 0) {
        if (bad) atomicOr(&out[0], 1u);
        if (m > __hip_atomic_load(&out[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&out[1], m);
    }
}

__global__ void k_zero_u32x2(uint32_t *p) {
    if (threadIdx.x < 2) p[threadIdx.x] = 0u;
}

void launch_field_scan(hipStream_t st, const float *T, int imax, int jmax, int kmax, uint32_t *out) {
    const size_t n = (size_t)(imax + 2) * (jmax + 2) * (kmax + 2);
    const int blocks = (int)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, 8192));
    hipLaunchKernelGGL(k_zero_u32x2, dim3(1), dim3(64), 0, st, out);
    hipLaunchKernelGGL(k_field_scan, dim3(blocks), dim3(256), 0, st, T, imax, jmax, kmax, out);
}

int launch_rays64(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int s, int v0, int nv, int surface,
                  const uint16_t *keys, size_t vkeys, double *ray, size_t nray, int *queue, double *de,
                  unsigned long long *stats) {
    const int ub = surface ? (cm.adiab[0] ? 0 : cm.nsurf) : 0;
    const int ue = surface ? (cm.adiab[1] ? 2 * cm.nsurf : cm.nsurf) : cm.ncell;
    const size_t P = (size_t)cm.photmax;
    int n = 0;
    for (int u = ub, nu = 0; u < ue; u += nu) {
        nu = (int)std::max<size_t>(1, std::min<size_t>(nray / nv / P, (size_t)(ue - u)));
        const int blocks = (int)std::min<size_t>((nv * nu * P + 255) / 256, 4 * 256);
        launch_zero_u64(st, reinterpret_cast<unsigned long long *>(queue), QUEUE_WORDS / 2);
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, st, cm, snaps, s, v0, nv, keys, vkeys, u, nu, queue, ray,
                               stats);
        };
        if (surface) { if (cm.grid_num > 1) go(k_rays64<true, true>); else go(k_rays64<true, false>); }
        else { if (cm.grid_num > 1) go(k_rays64<false, true>); else go(k_rays64<false, false>); }
        const int sb = (int)std::min<size_t>(((size_t)nv * nu + 127) / 128, 1 << 20);
        hipLaunchKernelGGL(k_sum_rays64, dim3(sb), dim3(128), 0, st, ray, u, nu, cm.photmax, cm.nVar, v0, nv, de);
        n += 3;
    }
    return n;
}

void launch_trace(hipStream_t st, const DevCommon &cm, const DevSnap *snaps, int surface, const int32_t *rays,
                  const int32_t *unit, int n, const uint16_t *keys, rc_ray *out) {
    hipLaunchKernelGGL(k_trace, dim3((n + 63) / 64), dim3(64), 0, st, cm, snaps, surface, rays, unit, n, keys, out);
}

void launch_finalize(hipStream_t st, const double *de, int n, int nVar, float *mean, float *sdev) {
    const int blocks = std::max(1, std::min((n + 255) / 256, 65536));
    hipLaunchKernelGGL(k_finalize, dim3(blocks), dim3(256), 0, st, de, n, nVar, mean, sdev);
}

}  // namespace rc
