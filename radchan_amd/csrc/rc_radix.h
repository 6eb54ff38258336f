/* Sorts of 16-bit keys by one wavefront, shared by the batched kernel and the
 * plain variants' band sort: up to 256 keys in registers, else an LSD radix
 * sort of two passes of up to 8 bits (keys in HBM scratch, in LDS). */
#ifndef RC_RADIX_H
#define RC_RADIX_H

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rc_device.h"

namespace rc {

using namespace rcd;


/* bitonic sort of 64 R keys held in registers, element R lane + r in x[r]:
 * compare-exchanges at distances below R stay inside a lane; the stages at
 * distance R..32 R exchange with lane (lane ^ distance/R) (21 of them).  No
 * LDS traffic and no barrier.  Which of the two a lane keeps depends on two
 * bits of its index: 0 or all ones, the median's third operand, so that an
 * exchange is 2 instructions instead of 4 (minimum, maximum, select):
 * 192x128x192 at three levels, 100 rays per unit, 50.8 -> 50.3 ms. */
template <int R>
__device__ __forceinline__ void wave_sort(uint32_t (&x)[R], int lane) {
    /* the lane index as an opaque value, so that the per-stage masks
     * are formed here instead of being hoisted out of the caller's loop and
     * kept live across it */
    asm volatile("" : "+v"(lane));
    /* bit b of the element index R lane as all ones or 0 */
    auto bit = [&](int v, int b) { return (uint32_t)((v << (31 - b)) >> 31); };
#pragma unroll
    for (int kb = 1; (1 << kb) <= 64 * R; ++kb) {
        const int k = 1 << kb;
#pragma unroll
        for (int jb = kb - 1; jb >= 0; --jb) {
            const int j = 1 << jb;
            if (j < R) {
                /* descending where bit kb is set */
                const uint32_t down = k < R ? 0u : (k >= 64 * R ? 0u : bit(lane * R, kb));
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int p = r ^ j;
                    if (p > r) {
                        const uint32_t d = k < R ? ((r & k) ? ~0u : 0u) : down, u = x[r], w = x[p];
                        x[r] = umed3(u, w, d);
                        x[p] = umed3(u, w, ~d);
                    }
                }
            } else {
                const int v = lane * R;
                const uint32_t keep_max = bit(k >= 64 * R ? v : v ^ (v >> (kb - jb)), jb);
#pragma unroll
                for (int r = 0; r < R; ++r) x[r] = umed3(x[r], lane_xor(x[r], j / R), keep_max);
            }
        }
    }
}

/* the bits that keys below nkey use above their low eight */
__device__ __forceinline__ int radix_high_bits(int nkey) { return 32 - __clz((uint32_t)(nkey - 1) >> 8 | 1u); }

/* the bits of m below this lane */
__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

/* The two digit histograms (hist[0..255]: bits 0-7 of the keys,
 * hist[256..511]: bits 8-15) turned into exclusive prefix sums, each lane
 * holding 4 consecutive buckets of a histogram. */
__device__ __forceinline__ void radix_offsets(uint32_t *hist, int lane) {
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        uint32_t *hh = hist + 256 * half + 4 * lane;
        const uint32_t c0 = hh[0], c1 = hh[1], c2 = hh[2], c3 = hh[3];
        const uint32_t s = c0 + c1 + c2 + c3;
        uint32_t inc = s;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)inc, d);
            if (lane >= d) inc += y;
        }
        const uint32_t ex = inc - s;
        hh[0] = ex;
        hh[1] = ex + c0;
        hh[2] = ex + c0 + c1;
        hh[3] = ex + c0 + c1 + c2;
    }
    __syncthreads();
}

/* The first pass of the LSD sort, on the low digit: nothing has been ordered
 * yet, so equal digits may come in any order, and every key takes its place
 * from its digit's running offset by one LDS atomic (about 12 vector
 * instructions per 64 keys, against 75 of the stable pass below) */
__device__ __forceinline__ void radix_first(const uint16_t *src, uint16_t *dst, uint32_t *off, int n, int lane) {
#pragma unroll 1
    for (int h = lane; h < n; h += 64) {
        const uint32_t key = (uint32_t)src[h];
        dst[atomicAdd(&off[key & 255u], 1u)] = (uint16_t)key;
    }
    __syncthreads();
}

/* The stable pass on the high digit, of nbits <= 8 bits (the bits the keys
 * use above the low eight): key h goes to dst[off[digit] + (keys of that
 * digit before h)], off being the digit's running offset in LDS.  Keys are
 * taken 64 at a time in order; the lanes holding the same digit are found
 * by a ballot per bit, so the pass keeps the order of equal digits.  src and
 * dst are the wavefront's own scratch, in HBM or LDS.  One wavefront per
 * workgroup. */
__device__ __forceinline__ void radix_high(const uint16_t *src, uint16_t *dst, uint32_t *off, int n, int nbits,
                                           int lane) {
#pragma unroll 1
    for (int base = 0; base < n; base += 64) {
        const bool ok = base + lane < n;
        const uint32_t key = ok ? (uint32_t)src[base + lane] : 0u;
        {
            const uint32_t dig = key >> 8;
            unsigned long long m = __ballot(ok);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                if (b >= nbits) break;
                const unsigned long long bb = __ballot((dig >> b) & 1u);
                m &= ((dig >> b) & 1u) ? bb : ~bb;
            }
            if (ok) {
                const uint32_t o = off[dig];
                const uint32_t below = lanes_below(m);
                dst[o + below] = (uint16_t)key;
                if (below == 0) off[dig] = o + (uint32_t)__popcll(m);
            }
        }
    }
    __syncthreads();
}

}  // namespace rc

#endif
