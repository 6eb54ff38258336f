/*
 * rc_spline.hip -- restriction of the temperature field to a coarse grid
 * level by cubic splines (interp3D, src/montecarlo/spline.cpp:36-177), an
 * alternative to the texture average the reference's kernels use for the
 * coarse levels (mc_gpu_noint.cu:334-338; interp3D is not called there,
 * :694).
 *
 * interp3D interpolates the fine field to the coarse cell centres with
 * natural cubic splines along x (every fine (j, k) line), then y (every
 * coarse i, fine k), then z (every coarse (i, j)); the x walls take the
 * spline (along y, then z) of the face means (T_ghost + T_first)/2, and
 * the coarse ghost is 2 face - interior, so the coarse face mean is that
 * spline.  The arithmetic is the reference's spline/splint
 * (spline.cpp:180-226, Numerical Recipes): float data with the double
 * constants there, so that some products are formed in double and rounded
 * to float on assignment -- kept as written, the CPU restatement and this
 * kernel agree bit for bit.
 *
 * The sweeps along a line are serial, so a line's are one lane's, on values
 * in LDS.  All else is not: everything that depends on the grid alone (the
 * sweep's coefficients, the reciprocals of its divisors, each output's
 * interval and weights) is formed once per axis (k_spline_axis) instead of
 * by every line, and the slopes before the sweep and the outputs after it
 * are by all threads of the line's workgroup.  Quotients with a divisor b
 * known beforehand are a r with r = RN(1/b) and two residual corrections by
 * fma, which is the rounded quotient (Markstein 1990), 5 instructions instead
 * of the division's 11 to 14, checked against / on 3e8 random pairs and every
 * float divisor; lines or grids with values outside 1e-15..1e15, where a
 * residual could leave the normal range, divide.  Lines along x are read and
 * written with lanes along the line; along y and z consecutive lines are
 * consecutive addresses.  The x-wall passes run in the launches of the x and
 * z passes.
 *
 * Bound by the sweep's chain (9 dependent operations, 7 of them in FP64, per
 * point: about 300 clocks with the backward sweep) and the loads before it:
 * 192x128x192 to 96x64x96 with walls 1484 -> 159 us, of which x 70, y 27, z
 * 38 and the axes 20 us.  With coefficients per line and sweeps in global
 * memory it was 1484 us; with the sweep doing all the work 371 us, its
 * coefficients by scalar loads one point ahead (each wait also one for LDS)
 * 360 us, slopes and outputs by all threads 228 us, four points at a time
 * 159 us.
 *
 * Outputs: Tl [km][jm][im] cell temperatures and, when asked, Tw [2][km][jm]
 * the west/east face temperatures.  This runs once per snapshot and level,
 * before the march.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "rc_internal.h"
#include "rc_kernels.h"

namespace rc {
namespace {

/* what a line takes from its axis at point i: dx = x[i+1] - x[i], dx2 =
 * x[i+1] - x[i-1], p the forward sweep's divisor, their reciprocals, c its
 * y2 */
struct SplCoef {
    double dx2, rdx2, p, rp;
    float sig, c, dx, rdx;
};
/* an output's interval klo, klo + 1 and weights (spline.cpp:209-226) */
struct SplOut {
    int klo;
    float a, b, ca, cb, hh;
};
struct SplAxis {
    const SplCoef *k;       /* [n+1], i = 1..n-1                         */
    const SplOut *o;        /* [m+1], j = 1..m                           */
    const int *fast;        /* 1: the grid's divisors lie in 1e-12..1e12 */
    int n, m;
};

__device__ __forceinline__ float div_by(float a, float b, float r) {
    float q = a * r;
    q = fmaf(fmaf(-q, b, a), r, q);
    return fmaf(fmaf(-q, b, a), r, q);
}
__device__ __forceinline__ double div_by(double a, double b, double r) {
    double q = a * r;
    q = fma(fma(-q, b, a), r, q);
    return fma(fma(-q, b, a), r, q);
}

template <bool FAST, class T>
__device__ __forceinline__ T quot(T a, T b, T r) {
    return FAST ? div_by(a, b, r) : a / b;
}

/* The second derivatives of the spline through a line's y(1..n)
 * (spline.cpp:180-207 with yp1 = ypn = 1e30), in place of the differences of
 * its slopes, ui at U[i st], i = 2..n-1.  Four points at a time, so that what
 * does not hang on the point before overlaps, and the next four's inputs are
 * under way; points beyond the line's ends are worked on all the same, in the
 * rows U has there (SPL_PAD) and with whatever K holds.  The axis' entries,
 * the same for every lane, come by vector loads (the lines are in the CU's
 * cache since the slopes): a wait for a scalar load is a wait for every LDS
 * access too. */
constexpr int SPL_PAD = 7;
template <bool FAST>
__device__ __forceinline__ void spline_sweep(const SplAxis &ax, float *U, int st) {
    const int n = ax.n;
    int zero = 0;
    asm volatile("" : "+v"(zero));      /* keeps the loads from becoming scalar */
    const SplCoef *K = ax.k + zero;
    float up = 0.f, *w = U + 2 * st;
    U[st] = 0.f;
    {
        double dx2[4], rdx2[4], p[4], rp[4];
        float sig[4], ui[4];
        const SplCoef *k = K + 2;
        auto fetch = [&](const float *r) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                dx2[q] = k[q].dx2; rdx2[q] = k[q].rdx2; p[q] = k[q].p; rp[q] = k[q].rp;
                sig[q] = k[q].sig;
                ui[q] = r[q * st];
            }
            k += 4;
        };
        fetch(w);
        for (int i = 2; i <= n - 1; i += 4) {
            double v[4], pc[4], rc[4];
            float sc[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v[q] = quot<FAST>(6.0 * (double)ui[q], dx2[q], rdx2[q]);
                pc[q] = p[q]; rc[q] = rp[q]; sc[q] = sig[q];
            }
            fetch(w + 4 * st);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                up = (float)quot<FAST>(v[q] - (double)(sc[q] * up), pc[q], rc[q]);
                w[q * st] = up;
            }
            w += 4 * st;
        }
    }
    /* y2[n] = (un - qn u[n-1]) / (qn y2[n-1] + 1) with qn = un = 0 */
    const float qe = 0.0f, un = 0.0f;
    float z = FAST ? 0.0f : (float)((double)(un - qe * U[(n - 1) * st]) / ((double)(qe * K[n - 1].c) + 1.0));
    w = U + n * st;
    w[0] = z;
    w -= 4 * st;
    /* (entries of points below 0 would lie before the array) */
    float c[4], u[4];
    auto fetch = [&](int k0, const float *r) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            c[q] = K[max(k0 - q, 0)].c;
            u[q] = r[(3 - q) * st];
        }
    };
    fetch(n - 1, w);
    for (int k = n - 1; k >= 1; k -= 4) {
        float cc[4], uc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) { cc[q] = c[q]; uc[q] = u[q]; }
        fetch(k - 4, w - 4 * st);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            z = cc[q] * z + uc[q];
            w[(3 - q) * st] = z;
        }
        w -= 4 * st;
    }
}

/* the interval of x in xa[1..n] (spline.cpp:212-217) */
__device__ __forceinline__ int spl_interval(const float *xa, int n, float x) {
    int klo = 1, khi = n;
    while (khi - klo > 1) {
        const int k = (khi + klo) >> 1;
        if (xa[k] > x) khi = k; else klo = k;
    }
    return klo;
}

struct SplArgs {
    const float *T0;
    int imax, jmax, kmax, im, jm, km;
    SplAxis ax[3];
    float *tx;      /* [kmax][jmax][im] after the x pass  */
    float *txy;     /* [kmax][jm][im]   after the y pass  */
    float *by;      /* [2][kmax][jm]    face means along y */
    float *wk;      /* lines too long for LDS: y2, then u  */
    float *Tl, *Tw;
};

enum SplPass { SPL_X, SPL_Y, SPL_Z, SPL_WALL_Y, SPL_WALL_Z };

__host__ __device__ __forceinline__ int spl_axis(SplPass p) { return p == SPL_X ? 0 : (p == SPL_Y || p == SPL_WALL_Y ? 1 : 2); }
__host__ __device__ __forceinline__ size_t spl_lines(const SplArgs &a, SplPass p) {
    return p == SPL_X ? (size_t)a.jmax * a.kmax : p == SPL_Y ? (size_t)a.im * a.kmax : p == SPL_Z ? (size_t)a.im * a.jm
         : p == SPL_WALL_Y ? (size_t)2 * a.kmax : (size_t)2 * a.jm;
}
/* addresses of point 1 of line L in the pass's input and output, and their
 * steps along the line */
struct SplLine {
    const float *src, *src2;        /* src2: walls along y, the other side of the face mean */
    size_t ss;
    float *dst;
    size_t ds;
};
__device__ __forceinline__ SplLine spl_line(const SplArgs &a, SplPass p, size_t L) {
    SplLine l;
    l.src2 = nullptr;
    const size_t nx = (size_t)a.imax + 2, nxy = nx * (size_t)(a.jmax + 2);
    if (p == SPL_X) {                                   /* fine line (j, k) */
        const size_t j = L % a.jmax, k = L / a.jmax;
        l.src = a.T0 + 1 + nx * (j + 1) + nxy * (k + 1);
        l.ss = 1;
        l.dst = a.tx + L * a.im;
        l.ds = 1;
    } else if (p == SPL_Y) {                            /* line (coarse i, fine k) */
        const size_t i = L % a.im, k = L / a.im;
        l.src = a.tx + k * a.jmax * a.im + i;
        l.dst = a.txy + k * a.jm * a.im + i;
        l.ss = l.ds = a.im;
    } else if (p == SPL_Z) {                            /* line (coarse i, coarse j) */
        l.src = a.txy + L;
        l.dst = a.Tl + L;
        l.ss = l.ds = (size_t)a.jm * a.im;
    } else if (p == SPL_WALL_Y) {                       /* (side, fine k) of face means */
        const size_t side = L / a.kmax, k = L % a.kmax;
        l.src = a.T0 + (side ? (size_t)a.imax + 1 : 0) + nx + nxy * (k + 1);
        l.src2 = a.T0 + (side ? (size_t)a.imax : 1) + nx + nxy * (k + 1);
        l.ss = nx;
        l.dst = a.by + L * a.jm;
        l.ds = 1;
    } else {                                            /* (side, coarse j) */
        const size_t side = L / a.jm, j = L % a.jm;
        l.src = a.by + side * a.kmax * a.jm + j;
        l.dst = a.Tw + side * a.km * a.jm + j;
        l.ss = l.ds = a.jm;
    }
    return l;
}
__device__ __forceinline__ float spl_value(const SplLine &l, int i) {
    const float v = l.src[(size_t)(i - 1) * l.ss];
    return l.src2 ? (float)(0.5 * (double)(v + l.src2[(size_t)(i - 1) * l.ss])) : v;
}

/* one workgroup: `lpb` lines of pass pa, or, from block nb on, of pass pb;
 * values Y, and U, the slopes' differences and then the second derivatives,
 * in LDS at [i][line], padded by one line.  Everything but the sweep is by
 * all threads. */
constexpr int SPL_THREADS = 256, SPL_WAVES = SPL_THREADS / 64;
__global__ void __launch_bounds__(SPL_THREADS) k_spline_lines(SplArgs a, SplPass pa, int lpb, int nb, SplPass pb,
                                                              int lpb2) {
    extern __shared__ float spl_lds[];
    const bool second = (int)blockIdx.x >= nb;
    const SplPass p = second ? pb : pa;
    const int w = second ? lpb2 : lpb, st = w + 1, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SplAxis ax = a.ax[spl_axis(p)];
    const int n = ax.n, m = ax.m;
    const size_t L0 = (size_t)(second ? blockIdx.x - nb : blockIdx.x) * w;
    const int nl = (int)min((size_t)w, spl_lines(a, p) - L0);
    float *Y = spl_lds, *U = spl_lds + (size_t)(n + 1 + SPL_PAD) * st;
    const bool along = p == SPL_X || p == SPL_WALL_Y;   /* lines along memory: lanes along the line */
    const int col = tid % w, row = tid / w, rows = SPL_THREADS / w;     /* else lanes across lines */
    const SplLine mine = spl_line(a, p, L0 + min(along ? lane : col, nl - 1));
    auto line = [&](int l) {                            /* line l, the same for the wavefront */
        auto at = [&](const float *q) {
            const uint64_t v = reinterpret_cast<uint64_t>(q);
            return reinterpret_cast<float *>(
                ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32) |
                (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l));
        };
        return SplLine{at(mine.src), mine.src2 ? at(mine.src2) : nullptr, mine.ss, at(mine.dst), mine.ds};
    };
    float lo = 1e15f, hi = 1e-15f;
    auto keep = [&](int i, int l, float v) {
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
        Y[i * st + l] = v;
    };
    /* eight loads in flight per lane */
    if (along) {
        for (int l = wave; l < nl; l += 8 * SPL_WAVES)
            for (int i = 1 + lane; i <= n; i += 64) {
                float v[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = spl_value(line(min(l + q * SPL_WAVES, nl - 1)), i);
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (l + q * SPL_WAVES < nl) keep(i, l + q * SPL_WAVES, v[q]);
            }
    } else {
        for (int i = 1 + row; i <= n; i += 8 * rows) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = spl_value(mine, min(i + q * rows, n));
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (i + q * rows <= n) keep(i + q * rows, col, v[q]);
        }
    }
    const bool fast = __syncthreads_or(!(lo >= 1e-15f && hi <= 1e15f)) == 0 && *ax.fast != 0;
    if (col < nl)
#pragma unroll 4
        for (int i = 2 + row; i <= n - 1; i += rows) {
            const SplCoef &s1 = ax.k[i], &s0 = ax.k[i - 1];
            const float y0 = Y[(i - 1) * st + col], y1 = Y[i * st + col], y2 = Y[(i + 1) * st + col];
            U[i * st + col] = fast ? quot<true>(y2 - y1, s1.dx, s1.rdx) - quot<true>(y1 - y0, s0.dx, s0.rdx)
                                   : quot<false>(y2 - y1, s1.dx, s1.rdx) - quot<false>(y1 - y0, s0.dx, s0.rdx);
        }
    __syncthreads();
    if (tid < nl) {
        if (fast) spline_sweep<true>(ax, U + tid, st);
        else spline_sweep<false>(ax, U + tid, st);
    }
    __syncthreads();
    /* an output of line l (spline.cpp:209-226) */
    auto out = [&](const SplOut &o, int l) {
        const float *y = Y + o.klo * st + l, *z = U + o.klo * st + l;
        const float t1 = o.a * y[0] + o.b * y[st];
        const float t2 = (o.ca * z[0] + o.cb * z[st]) * o.hh;
        const double s6 = fast ? quot<true>((double)t2, 6.0, 1.0 / 6.0) : (double)t2 / 6.0;
        return (float)((double)t1 + s6);
    };
    if (along) {
        for (int j = 1 + lane; j <= m; j += 64) {
            const SplOut o = ax.o[j];
            for (int l = wave; l < nl; l += SPL_WAVES) line(l).dst[(size_t)(j - 1) * mine.ds] = out(o, l);
        }
    } else if (col < nl) {
#pragma unroll 4
        for (int j = 1 + row; j <= m; j += rows) mine.dst[(size_t)(j - 1) * mine.ds] = out(ax.o[j], col);
    }
}

/* lines of more points than LDS holds: a thread per line, the second
 * derivatives y2 and the sweep's u of line L at scratch [i][L], every
 * coefficient formed on the way (spline.cpp:180-226) */
__global__ void __launch_bounds__(64) k_spline_long(SplArgs a, SplPass p, const float *__restrict__ x,
                                                    const float *__restrict__ xc, int n, int m) {
    const size_t st = spl_lines(a, p), L = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (L >= st) return;
    const SplLine s = spl_line(a, p, L);
    auto y = [&](int i) { return spl_value(s, i); };
    float *y2 = a.wk + L, *u = a.wk + (size_t)(n + 1) * st + L;
    y2[st] = 0.0f;
    u[st] = 0.0f;
    for (int i = 2; i <= n - 1; ++i) {
        const float sig = (x[i] - x[i - 1]) / (x[i + 1] - x[i - 1]);
        const float q = (float)((double)(sig * y2[(i - 1) * st]) + 2.0);
        y2[i * st] = (float)(((double)sig - 1.0) / (double)q);
        const float ui = (y(i + 1) - y(i)) / (x[i + 1] - x[i]) - (y(i) - y(i - 1)) / (x[i] - x[i - 1]);
        u[i * st] = (float)((6.0 * (double)ui / (double)(x[i + 1] - x[i - 1]) - (double)(sig * u[(i - 1) * st])) /
                            (double)q);
    }
    const float qn = 0.0f, un = 0.0f;
    y2[n * st] = (float)((double)(un - qn * u[(n - 1) * st]) / ((double)(qn * y2[(n - 1) * st]) + 1.0));
    for (int k = n - 1; k >= 1; --k) y2[k * st] = y2[k * st] * y2[(k + 1) * st] + u[k * st];
    for (int j = 1; j <= m; ++j) {
        const int klo = spl_interval(x, n, xc[j]), khi = klo + 1;
        const float h = x[khi] - x[klo];
        const float b0 = (x[khi] - xc[j]) / h, b1 = (xc[j] - x[klo]) / h;
        const float t1 = b0 * y(klo) + b1 * y(khi);
        const float t2 = ((b0 * b0 * b0 - b0) * y2[klo * st] + (b1 * b1 * b1 - b1) * y2[khi * st]) * (h * h);
        s.dst[(size_t)(j - 1) * s.ds] = (float)((double)t1 + (double)t2 / 6.0);
    }
}

/* the axes' coefficients and outputs, a workgroup per axis: the divisions
 * by all threads, the chain of c and p (each from the one before) by one,
 * on sig values staged in LDS */
constexpr int AXIS_TILE = 2048;
struct AxisArgs {
    const float *x[3], *xc[3];
    SplCoef *k[3];
    SplOut *o[3];
    int *fast[3];
    int n[3], m[3];
};

__global__ void __launch_bounds__(256) k_spline_axis(AxisArgs a) {
    __shared__ float sig[AXIS_TILE], pv[AXIS_TILE], cv[AXIS_TILE];
    __shared__ int bad;
    __shared__ float cl;
    const int d = blockIdx.x, tid = threadIdx.x, n = a.n[d], m = a.m[d];
    const float *x = a.x[d], *xc = a.xc[d];
    SplCoef *k = a.k[d];
    if (tid == 0) { bad = 0; cl = 0.f; }
    __syncthreads();
    for (int i0 = 1; i0 <= n - 1; i0 += AXIS_TILE) {
        const int nt = min(AXIS_TILE, n - i0);
        for (int q = tid; q < nt; q += blockDim.x) {
            const int i = i0 + q;
            sig[q] = i >= 2 ? (x[i] - x[i - 1]) / (x[i + 1] - x[i - 1]) : 0.f;
        }
        __syncthreads();
        if (tid == 0) {
            float c = cl;
            for (int q = 0; q < nt; ++q) {
                const float p = (float)((double)(sig[q] * c) + 2.0);
                c = i0 + q >= 2 ? (float)(((double)sig[q] - 1.0) / (double)p) : 0.f;
                pv[q] = p;
                cv[q] = c;
            }
            cl = c;
        }
        __syncthreads();
        for (int q = tid; q < nt; q += blockDim.x) {
            const int i = i0 + q;
            SplCoef e;
            e.dx = x[i + 1] - x[i];
            e.rdx = 1.0f / e.dx;
            e.sig = sig[q];
            e.c = cv[q];
            e.dx2 = i >= 2 ? (double)(x[i + 1] - x[i - 1]) : 1.0;
            e.rdx2 = 1.0 / e.dx2;
            e.p = (double)pv[q];
            e.rp = 1.0 / e.p;
            k[i] = e;
            if (!(e.dx >= 1e-12f && e.dx2 <= 1e12 && e.p >= 1.0 && e.p <= 4.0)) bad = 1;
        }
        __syncthreads();
    }
    for (int j = 1 + tid; j <= m; j += blockDim.x) {
        const float xv = xc[j];
        const int klo = spl_interval(x, n, xv), khi = klo + 1;
        const float h = x[khi] - x[klo];
        SplOut o;
        o.klo = klo;
        o.a = (x[khi] - xv) / h;
        o.b = (xv - x[klo]) / h;
        o.ca = o.a * o.a * o.a - o.a;
        o.cb = o.b * o.b * o.b - o.b;
        o.hh = h * h;
        a.o[d][j] = o;
    }
    if (tid == 0) *a.fast[d] = !bad;
}

/* lines per workgroup whose values and U fit 54 KiB of LDS, so that three
 * workgroups share a CU and one's loads run beside another's sweep; 0: none,
 * more than SPL_NMAX points */
constexpr int SPL_NMAX = 2456;
inline size_t spl_block_lds(int n, int w) { return (size_t)(2 * (n + 1 + SPL_PAD)) * (w + 1) * 4; }
inline int spl_lines_per_block(int n) {
    for (int w = 64; w >= 4; w >>= 1)
        if (spl_block_lds(n, w) <= 55296u) return w;
    return n <= SPL_NMAX ? 2 : 0;
}
/* one axis' coefficients, flag and outputs (of lines up to SPL_NMAX) */
constexpr size_t SPL_AXIS_BYTES = ((size_t)(SPL_NMAX + 1) * (sizeof(SplCoef) + sizeof(SplOut)) + 16 + 15) / 16 * 16;
constexpr size_t SPL_AXES_FLOATS = 3 * SPL_AXIS_BYTES / 4;

}  // namespace

size_t spline_scratch_floats(int imax, int jmax, int kmax, int im, int jm, int km) {
    const size_t tx = (size_t)im * jmax * kmax, txy = (size_t)im * jm * kmax, by = (size_t)2 * kmax * jm;
    size_t wk = 2 * (size_t)(imax + 1) * jmax * kmax;
    wk = std::max(wk, 2 * (size_t)(jmax + 1) * im * kmax);
    wk = std::max(wk, 2 * (size_t)(kmax + 1) * im * jm);
    wk = std::max(wk, 2 * (size_t)(jmax + 1) * 2 * kmax);
    wk = std::max(wk, 2 * (size_t)(kmax + 1) * 2 * jm);
    return tx + txy + by + wk;
}

/* floats of the axes' coefficients (16-byte aligned) */
size_t spline_axes_floats() { return SPL_AXES_FLOATS; }

void launch_spline_level(hipStream_t st, const float *T0, const float *x0, const float *y0, const float *z0,
                         const float *xc, const float *yc, const float *zc, int imax, int jmax, int kmax, int im,
                         int jm, int km, float *Tl, float *Tw, float *scratch, float *axes) {
    SplArgs a;
    a.T0 = T0;
    a.imax = imax; a.jmax = jmax; a.kmax = kmax; a.im = im; a.jm = jm; a.km = km;
    const int n[3] = {imax, jmax, kmax}, m[3] = {im, jm, km};
    AxisArgs ax;
    const float *xf[3] = {x0, y0, z0}, *xo[3] = {xc, yc, zc};
    for (int d = 0; d < 3; ++d) {
        char *at = reinterpret_cast<char *>(axes) + d * SPL_AXIS_BYTES;
        ax.x[d] = xf[d];
        ax.xc[d] = xo[d];
        ax.n[d] = n[d] <= SPL_NMAX ? n[d] : 0;
        ax.m[d] = n[d] <= SPL_NMAX ? m[d] : 0;
        ax.k[d] = reinterpret_cast<SplCoef *>(at);
        at += (size_t)(SPL_NMAX + 1) * sizeof(SplCoef);
        ax.fast[d] = reinterpret_cast<int *>(at);
        ax.o[d] = reinterpret_cast<SplOut *>(at + 16);
        a.ax[d] = SplAxis{ax.k[d], ax.o[d], ax.fast[d], n[d], m[d]};
    }
    a.tx = scratch;
    a.txy = a.tx + (size_t)im * jmax * kmax;
    a.by = a.txy + (size_t)im * jm * kmax;
    a.wk = a.by + (size_t)2 * kmax * jm;
    a.Tl = Tl; a.Tw = Tw;
    hipLaunchKernelGGL(k_spline_axis, dim3(3), dim3(256), 0, st, ax);
    /* a pass, and a wall pass in the same launch; lines beyond LDS by
     * k_spline_long */
    auto run = [&](SplPass p, bool with, SplPass pw) {
        const int d = spl_axis(p), d2 = spl_axis(pw);
        const int w = spl_lines_per_block(n[d]), w2 = with ? spl_lines_per_block(n[d2]) : 0;
        const size_t nb = w ? (spl_lines(a, p) + w - 1) / w : 0, nb2 = w2 ? (spl_lines(a, pw) + w2 - 1) / w2 : 0;
        const size_t lds = std::max(w ? spl_block_lds(n[d], w) : 0, w2 ? spl_block_lds(n[d2], w2) : 0);
        if (nb + nb2)
            hipLaunchKernelGGL(k_spline_lines, dim3(nb + nb2), dim3(SPL_THREADS), lds, st, a, p, w, (int)nb, pw, w2);
        if (!w)
            hipLaunchKernelGGL(k_spline_long, dim3((spl_lines(a, p) + 63) / 64), dim3(64), 0, st, a, p, xf[d], xo[d],
                               n[d], m[d]);
        if (with && !w2)
            hipLaunchKernelGGL(k_spline_long, dim3((spl_lines(a, pw) + 63) / 64), dim3(64), 0, st, a, pw, xf[d2],
                               xo[d2], n[d2], m[d2]);
    };
    run(SPL_X, Tw != nullptr, SPL_WALL_Y);
    run(SPL_Y, false, SPL_WALL_Y);
    run(SPL_Z, Tw != nullptr, SPL_WALL_Z);
}

/* ---- the allocation-free entry point --------------------------------

rc_spline_restrict_noalloc works in `scratch`, a file-scope device array
of RC_SPLINE_NOALLOC_FLOATS floats (and the axes' coefficients, half a MiB
after them) that every GPU the library runs on holds until the process ends.  The host never passes the array's name to a kernel
(in host code it is a stand-in, not a device address): the device address
is looked up once per device with hipGetSymbolAddress, with that device
current, and kept in scratch_ptr[device]. */

namespace {

constexpr size_t kNoallocFloats = RC_SPLINE_NOALLOC_FLOATS;
static __device__ __align__(256) float scratch[kNoallocFloats + SPL_AXES_FLOATS];

constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
float *scratch_ptr[kMaxDevices] = {};

/* the device address of this device's scratch (nullptr and a message on failure) */
float *device_scratch(int dev) {
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("rc_spline_restrict_noalloc: device ordinal beyond 63");
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error(std::string("rc_spline_restrict_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
            return nullptr;
        }
        scratch_ptr[dev] = static_cast<float *>(p);
    }
    return scratch_ptr[dev];
}

/* working floats of the grid step: f[im0+1], then the centres x0, y0, z0
 * of level 0 and xc, yc, zc of the coarse level (n+2 each), rounded up to
 * 64 floats so the spline scratch after it stays 256-byte aligned */
size_t grid_floats(int im0, int jm0, int km0, int im, int jm, int km) {
    const size_t n = (size_t)(im0 + 1) + (im0 + 2) + (jm0 + 2) + (km0 + 2) + (im + 2) + (jm + 2) + (km + 2);
    return (n + 63) / 64 * 64;
}

struct GridArgs {
    int im0, jm0, km0, im, jm, km;
    float Lx, Ly, Lz;
    double fact_mesh;
    float *f, *x0, *y0, *z0, *xc, *yc, *zc;
};

/* centre c[j] of n uniform cells of length L, j = 0..n+1 with mirrored
 * ghosts (the y and z directions of Gridn::mk_grid, definitions.h:85-105) */
__device__ float uniform_centre(float L, int n, int j) {
    const float d = L * 1.0f / (float)n;
    if (j == 0) return -d / 2.0f;
    const int q = min(j, n);
    const float c = ((float)(q - 1) * d + (float)q * d) / 2.0f;
    return j == n + 1 ? c + d : c;
}

/* x centre x[i], i = 0..im+1, of a level with im cells from the fine faces
 * f[0..im0] (definitions.h:125-134) */
__device__ float x_centre(const float *f, int im0, int im, int i) {
    const int q = min(max(i, 1), im);
    const float hi = f[(size_t)q * im0 / im], lo = f[(size_t)(q - 1) * im0 / im];
    const float c = (float)(0.5 * (double)(hi + lo));
    return i == 0 ? -c : (i == im + 1 ? hi + (hi - c) : c);
}

/* Gridn::mk_grid (definitions.h:68-136) of level 0 and of the coarse
 * level by one workgroup: the cell widths and their scaling by all threads,
 * their running sum by one, on a tile in LDS; the operations of the host's
 * build_grid, so the centres are equal to its bit for bit */
constexpr int GRID_TILE = 4096;
__global__ void __launch_bounds__(256) k_level_grid(GridArgs a) {
    __shared__ float t[GRID_TILE];
    float *f = a.f;
    const int half = a.im0 / 2, tid = threadIdx.x, nt = blockDim.x;
    float run = 0.f;                     /* thread 0's */
    if (tid == 0) f[0] = 0.f;
    for (int i0 = 1; i0 <= half; i0 += GRID_TILE) {
        const int n = min(GRID_TILE, half - i0 + 1);
        for (int q = tid; q < n; q += nt) {
            const double r = (double)((float)(i0 + q) / (float)a.im0) - 0.5;
            t[q] = (float)(0.5 - a.fact_mesh * r * r);
        }
        __syncthreads();
        if (tid == 0)
            for (int q = 0; q < n; ++q) {
                run = run + t[q];
                t[q] = run;
            }
        __syncthreads();
        for (int q = tid; q < n; q += nt) f[i0 + q] = t[q];
        __syncthreads();
    }
    const double norm = (double)f[half];
    const double scale = (double)a.Lx / 2.;
    __syncthreads();
    for (int i = 1 + tid; i <= half; i += nt) f[i] = (float)(scale * (double)f[i] / norm);
    __syncthreads();
    for (int i = half + 1 + tid; i <= a.im0; i += nt) f[i] = a.Lx - f[a.im0 - i];
    __syncthreads();
    for (int i = tid; i <= a.im0 + 1; i += nt) a.x0[i] = x_centre(f, a.im0, a.im0, i);
    for (int i = tid; i <= a.im + 1; i += nt) a.xc[i] = x_centre(f, a.im0, a.im, i);
    for (int j = tid; j <= a.jm0 + 1; j += nt) a.y0[j] = uniform_centre(a.Ly, a.jm0, j);
    for (int k = tid; k <= a.km0 + 1; k += nt) a.z0[k] = uniform_centre(a.Lz, a.km0, k);
    for (int j = tid; j <= a.jm + 1; j += nt) a.yc[j] = uniform_centre(a.Ly, a.jm, j);
    for (int k = tid; k <= a.km + 1; k += nt) a.zc[k] = uniform_centre(a.Lz, a.km, k);
}

}  // namespace

}  // namespace rc

/* allocation-free rc_spline_restrict on device arrays (declared in
 * include/radchan.h): grid and spline work in this device's scratch,
 * asynchronous on `stream` */
extern "C" int rc_spline_restrict_noalloc(const rc_params *p, int level, const float *T, float *Tc, float *Tw,
                                          void *stream) {
    using namespace rc;
    if (!p || !T || !Tc) { set_error("rc_spline_restrict_noalloc: null argument"); return -1; }
    if (int e = check_params(*p)) return e;
    if (level < 1 || level >= p->grid_num) { set_error("rc_spline_restrict_noalloc: level in 1..grid_num-1"); return -2; }
    if (p->imax < 2 || p->jmax < 2 || p->kmax < 2) { set_error("cubic-spline restriction needs imax, jmax, kmax >= 2"); return -2; }
    const int im = p->maxi[level], jm = p->maxj[level], km = p->maxk[level];
    const size_t ng = grid_floats(p->imax, p->jmax, p->kmax, im, jm, km);
    const size_t need = ng + spline_scratch_floats(p->imax, p->jmax, p->kmax, im, jm, km);
    if (need > kNoallocFloats) {
        set_error("rc_spline_restrict_noalloc: the field needs " + std::to_string(need) +
                  " floats of scratch, beyond its fixed " + std::to_string(kNoallocFloats) +
                  " (use rc_spline_restrict)");
        return -2;
    }
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) { set_error("no HIP device available"); return -3; }
    float *w = device_scratch(dev);
    if (!w) return -3;
    GridArgs g;
    g.im0 = p->imax; g.jm0 = p->jmax; g.km0 = p->kmax; g.im = im; g.jm = jm; g.km = km;
    g.Lx = p->Lx; g.Ly = p->Ly; g.Lz = p->Lz; g.fact_mesh = p->fact_mesh;
    g.f = w;
    g.x0 = g.f + (p->imax + 1);
    g.y0 = g.x0 + (p->imax + 2);
    g.z0 = g.y0 + (p->jmax + 2);
    g.xc = g.z0 + (p->kmax + 2);
    g.yc = g.xc + (im + 2);
    g.zc = g.yc + (jm + 2);
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_level_grid, dim3(1), dim3(256), 0, st, g);
    launch_spline_level(st, T, g.x0, g.y0, g.z0, g.xc, g.yc, g.zc, p->imax, p->jmax, p->kmax, im, jm, km, Tc, Tw,
                        w + ng, w + kNoallocFloats);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error(std::string("rc_spline_restrict_noalloc: ") + hipGetErrorString(e)); return -4; }
    return 0;
}
