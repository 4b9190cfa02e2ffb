// Test helper: the float grid's id windows (IdWindows) over a sorted list of
// the ids within an owner's reach.  Returns the passes over the candidates, or
// -1 if the windows do not cover every id once, in order, within the cap.
#include <algorithm>

#include "boids_internal.h"

extern "C" int64_t window_passes(const uint32_t* ids, uint32_t m, uint32_t n, uint32_t cap)
{
    int64_t passes = 0;
    uint32_t served = 0;
    for (boids::IdWindows w(n, cap); w.more(); ++passes) {
        const uint32_t lo = w.lo, hi = w.width < n - lo ? lo + w.width : n;
        if (lo >= hi || passes > (1 << 20)) return -1;
        const uint32_t a = (uint32_t)(std::lower_bound(ids, ids + m, lo) - ids);
        const uint32_t b = (uint32_t)(std::lower_bound(ids, ids + m, hi) - ids);
        if (!w.take(b - a)) continue;
        if (a != served || b - a > cap) return -1;
        served = b;
    }
    return served == m ? passes : -1;
}
