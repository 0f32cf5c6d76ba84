// search_window.hpp -- how a search tile keeps a larger window in LDS: arithmetic of one window, the
// same on the host (tests/cpp/window_tests.hip) and in the tile (search_tile.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace setops {

// A larger window in LDS: n elements from pool index g, in cl chunks of 16 bytes: whole (m == 0), or as
// ns samples, the first elements of lines (g >> 5) + m, + 2m, ...
struct LargeWindow {
    uint64_t g;
    uint32_t lo, hi;  // pair-relative, lo <= hi
    uint32_t cl, m, ns;
};

// The window [lo, hi) of the larger set at pool index `base`, searched for `probes` values: staged whole
// up to `stage` elements per probe, else sampled with at most `sample` samples per probe (and
// `min_sample`).  lo and hi are found by two searches that know nothing of each other: in a set that is
// not sorted they may cross, and the window is then empty.
__host__ __device__ __forceinline__ LargeWindow large_window(uint64_t base, uint32_t lo, uint32_t hi, uint32_t probes,
                                                             uint32_t stage, uint32_t sample, uint32_t min_sample)
{
    LargeWindow w{base + lo, lo, hi > lo ? hi : lo, 0, 0, 0};
    const uint32_t n = w.hi - w.lo;
    if (n == 0) return w;
    if (n <= stage * probes) {
        w.cl = ((uint32_t)(w.g & 3) + n + 3) / 4;
        return w;
    }
    const uint32_t heads = (uint32_t)(((w.g + n - 1) >> 5) - (w.g >> 5));  // lines after the first
    const uint32_t most = sample * probes > min_sample ? sample * probes : min_sample;
    w.m = (heads + most - 1) / most;
    if (w.m == 0) w.m = 1;
    w.ns = heads / w.m;
    w.cl = (w.ns + 3) / 4;
    if (w.cl == 0) w.cl = 1;
    return w;
}

// The range [at, end) of LDS words that a probe of a staged window of n words from word lb searches.  The
// lifting reads word y - 1 for at <= y <= end, also where at == end: an empty window, which may begin at
// word 0, takes the range [1, 1) of a probe without a window.
struct LiftRange {
    uint32_t at, end;
};
__host__ __device__ __forceinline__ LiftRange lift_range(uint32_t lb, uint32_t n)
{
    return n ? LiftRange{lb, lb + n} : LiftRange{1, 1};
}
// ... its next position at most `step` further
__host__ __device__ __forceinline__ uint32_t lift_to(const LiftRange &r, uint32_t step)
{
    return r.at + step < r.end ? r.at + step : r.end;
}

} // namespace setops
