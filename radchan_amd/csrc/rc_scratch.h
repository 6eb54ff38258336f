/*
 * rc_scratch.h -- how much device scratch a solve takes: what makes it
 * fastest where there is room, else what it cannot do without.
 *
 * Buf: ensure(n) holds n bytes or more afterwards and returns 0, or returns
 * an error and holds nothing (what it held is given back first); release();
 * bytes, what it holds.
 */
#ifndef RC_SCRATCH_H
#define RC_SCRATCH_H

#include <algorithm>
#include <cstddef>

namespace rc {

/* The FP64 solve's band keys, 16 bits each, run_keys per run (0: none), and
 * its rays' tallies, 8 bytes each, run_rays per run: the runs that a launch
 * takes together, 0 if there is no memory (`keys` or `ray` has said so).  The keys
 * of one run come first, since nothing goes without them; then the tallies of all runs,
 * 2 GiB at most, or a half, a quarter, .. of that, down to a unit's,
 * unit_rays (the launches are split to fit); then the other runs' keys. */
template <class Buf>
int fp64_scratch(Buf &keys, Buf &ray, size_t run_keys, size_t run_rays, size_t unit_rays, int nVar) {
    size_t want = std::max(std::min(run_rays * nVar, (size_t)1 << 28), unit_rays);
    for (;;) {
        if (run_keys && keys.ensure(run_keys * 2)) {
            if (!ray.bytes) return 0;
            ray.release();
            continue;
        }
        if (ray.bytes >= unit_rays * 8 || !ray.ensure(want * 8)) {
            const int runs = (int)std::max<size_t>(1, std::min<size_t>(nVar, ray.bytes / 8 / run_rays));
            if (!run_keys || runs == 1 || !keys.ensure(run_keys * runs * 2)) return runs;
            if (!keys.ensure(run_keys * 2)) return 1;
            ray.release();
        }
        if (want == unit_rays) return 0;
        want = std::max(want / 2, unit_rays);
    }
}

/* The batched launches' sort scratch: 16-bit keys, `fluid` and `walls` of
 * them.  1: both beside each other, so that the walls' launch may run while
 * the fluid's does; 0: room for the larger, one launch after the other; < 0:
 * neither.  refused: the size there was no memory for (0: none yet), which
 * is not asked for again on every solve. */
template <class Buf>
int sort_scratch(Buf &b, size_t fluid, size_t walls, size_t &refused) {
    const size_t both = (fluid + walls) * 2, one = std::max(fluid, walls) * 2;
    if (both == 0 || b.bytes >= both) return 1;
    if (!refused || both < refused) {
        if (!b.ensure(both)) return 1;
        if (both != one) refused = both;
    }
    return b.ensure(one) ? -1 : 0;
}

}  // namespace rc

#endif
