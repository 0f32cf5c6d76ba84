// Host tests of the search tile's window arithmetic (search_window.hpp): runs on the CPU.
#include <cstdio>
#include <cstdlib>

#include "../../simd_set_operations_amd/csrc/search_window.hpp"

static int failures = 0;
#define CHECK(cond, ...)                            \
    do {                                            \
        if (!(cond)) {                              \
            if (failures++ < 10) {                  \
                std::printf("FAILED %s: ", #cond);  \
                std::printf(__VA_ARGS__);           \
                std::printf("\n");                  \
            }                                       \
        }                                           \
    } while (0)

static uint64_t state = 88172645463325252ull;
static uint64_t rnd(uint64_t n)
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return state % n;
}

// Every element a window's staging or sampling reads lies inside the larger set, and the chunks hold it,
// whichever bounds the two searches return.
static void windows()
{
    const uint32_t per_probe[][2] = {{13, 4}, {6, 4}, {2, 2}, {4, 4}, {9, 4}};  // stage, sample
    for (int i = 0; i < 2000000; i++) {
        const uint64_t base = rnd(2) ? rnd(100) : rnd(1ull << 36);
        const uint32_t size = (uint32_t)(rnd(4) ? 1 + rnd(5000) : 1 + rnd(0xFFFFFFFEull));
        const uint32_t lo = (uint32_t)rnd((uint64_t)size + 1), hi = (uint32_t)rnd((uint64_t)size + 1);
        const uint32_t probes = 1 + (uint32_t)rnd(1024), *k = per_probe[rnd(5)];
        const setops::LargeWindow w = setops::large_window(base, lo, hi, probes, k[0], k[1], 24);
        const uint64_t first = base + lo, end = base + (hi > lo ? hi : lo);
        CHECK(w.lo == lo && w.lo <= w.hi && w.hi <= size && base + w.hi == end, "lo %u hi %u", lo, hi);
        CHECK(w.g == first, "lo %u hi %u", lo, hi);
        if (first == end) {
            CHECK(w.cl == 0 && w.m == 0 && w.ns == 0, "empty window, lo %u hi %u: cl %u", lo, hi, w.cl);
        } else if (w.m == 0) {
            CHECK(4ull * w.cl >= (first & 3) + (end - first) && w.cl <= (k[0] * probes + 6) / 4, "cl %u", w.cl);
        } else {
            CHECK(4ull * w.cl >= w.ns && w.ns <= (k[1] * probes > 24 ? k[1] * probes : 24), "cl %u ns %u", w.cl, w.ns);
            // the last sample's line begins inside the window, and fewer than m lines follow it
            const uint64_t line = (first >> 5) + (uint64_t)w.ns * w.m;
            CHECK(w.ns == 0 || 32 * line < end, "ns %u m %u", w.ns, w.m);
            CHECK(((end - 1) >> 5) - line < w.m, "ns %u m %u", w.ns, w.m);
        }
    }
}

// The words that the lifting reads and the value it finds, over windows anywhere in the staged words, empty ones
// and the first word included.
static void lifting()
{
    static uint32_t words[4096];
    for (uint32_t i = 0; i < 4096; i++) words[i] = 3 * i + 1;
    for (int i = 0; i < 500000; i++) {
        const uint32_t n = (uint32_t)(rnd(3) ? rnd(40) : rnd(3000)), lb = rnd(3) ? 0u : (uint32_t)rnd(4096 - n);
        const uint32_t x = (uint32_t)rnd(3 * 4096 + 2), steps = (uint32_t)rnd(13);  // the wave's, at least log2 n
        setops::LiftRange r = setops::lift_range(lb, n);
        CHECK(r.at <= r.end && r.end <= 4096, "lb %u n %u", lb, n);
        uint32_t levels = 0;
        while (n >> levels) levels++;
        for (int bit = (int)(steps > levels ? steps : levels) - 1; bit >= 0; bit--) {
            const uint32_t y = setops::lift_to(r, 1u << bit);
            CHECK(y >= 1 && y <= 4096, "lb %u n %u: reads word %d", lb, n, (int)y - 1);
            if (y >= 1 && y <= 4096 && words[y - 1] < x) r.at = y;
        }
        uint32_t lower = lb;
        while (lower < lb + n && words[lower] < x) lower++;
        CHECK(n == 0 ? r.at == r.end : r.at == lower, "lb %u n %u x %u: %u", lb, n, x, r.at);
    }
}

int main()
{
    windows();
    lifting();
    std::printf("%d failures\n", failures);
    return failures ? 1 : 0;
}
