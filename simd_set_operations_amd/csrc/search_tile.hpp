// search_tile.hpp -- probe-per-element tile kernel for skewed pairs (gfx950).
//
// The search policy of the reference's galloping / binary_search_intersect
// (setops/src/intersect/galloping.rs:7-49): every element of the smaller set ("probe") is looked
// up in the larger set.  Units are probes (tile_plan.hpp, POLICY_SEARCH), so a tile carries
// U = NT*KS probes whatever the sizes of the larger sets.  Per tile:
//   1. segment table; stage the probe windows in LDS (the smaller side of each pair, which may
//      be A or B -- orientation does not change the result, A∩B ascending),
//   2. narrow the larger set of a pair that other tiles share to [lo, hi): lower bound of the
//      segment's first probe and upper bound of its last probe, by a wave-cooperative 64-way
//      partition search,
//   3. stage the larger windows in LDS, whole where they are short, else the first element of every
//      m-th line, while they fit (a prefix of the segments); the rest are searched in global memory,
//   4. each lane looks up its KS probes: in windows staged whole by binary lifting, in sampled windows
//      and through the B-pool index by groups of lanes that read the line found, the same for every
//      entry.  The search mode tells the entries apart where a window found no room (and for further
//      sets): galloping (exponential then binary, galloping.rs:7-30), binary search
//      (binary_search_intersect, galloping.rs:32-49) or block galloping with a full compare of the
//      last block (simd_galloping.rs:49-107), each probe from the window's start,
//   5. block scan of hits, results (probe values; BSR: base and state AND) staged in order,
//      tile and per-pair counts -- the same outputs as the merge tile kernel.
#pragma once

#include "search_window.hpp"
#include "tile_plan.hpp"

namespace setops {

template <int NT, int KS, int MAXSEG, int CAPB, bool BSR>
struct SearchSmem {
    static constexpr int U = NT * KS;
    static constexpr int PKEYS = U + 8 * MAXSEG + 16;
    static constexpr int LKEYS = CAPB + 16;
    uint32_t pkey[PKEYS];               // probe windows
    uint32_t pst[BSR ? PKEYS : 4];
    uint32_t lkey[LKEYS];               // staged larger windows
    uint32_t lst[BSR ? LKEYS : 4];
    uint32_t seg_u[MAXSEG + 1];
    uint32_t seg_la[MAXSEG];            // LDS index of the segment's first probe
    uint32_t seg_wa[MAXSEG];            // probes in the window
    uint32_t seg_lo[MAXSEG];            // narrowed larger window [lo, hi), pair-relative
    uint32_t seg_hi[MAXSEG];
    uint32_t seg_lb[MAXSEG];            // LDS index of lkey[lo] (or of its samples), or kNotStaged
    uint32_t seg_m[MAXSEG];             // lines per sample of a sampled window, 0: staged whole
    // bit0: pair starts here, bit1: ends here, bit2: larger side is A; from bit 8: samples
    uint32_t seg_flags[MAXSEG];
    uint32_t narrow[4];                 // first segment's narrowed window, last segment's
    uint64_t seg_lbase[MAXSEG];         // pool index of the larger set's first element
    uint32_t lane_mask[NT];
    uint32_t lane_pfx[NT];
    uint32_t scan_scratch[NT / kWave];
    uint32_t wave_el[NT / kWave];
    uint32_t win_c[MAXSEG + 1];
    uint64_t win_g[MAXSEG];
    uint32_t win_src[MAXSEG];
    uint32_t xlo[kMaxExtraSets];  // further sets (single pair): the tile's probe range in each
    uint32_t xhi[kMaxExtraSets];
    // top level of the B-pool index over the tile's larger B sets: top[j - top_j0] = B[kTopStride j]
    alignas(16) uint32_t top[kTopCap];
    unsigned long long red64[NT / kWave][2];
};

constexpr uint32_t kNotStaged = 0xFFFFFFFFu;
constexpr uint32_t kNoNarrow = 16 * 3072;  // larger sets searched through the B-pool index unnarrowed

// Lower bound of x in arr[lo, hi) starting from lo: galloping (probe lo+1, lo+3, lo+7, ... then
// binary search in the last gap) or plain binary search.  Works on LDS or global arrays.
template <bool GALLOP, class Arr>
__device__ __forceinline__ uint32_t lower_bound_from(const Arr &arr, uint32_t lo, uint32_t hi, uint32_t x)
{
    if constexpr (GALLOP) {
        uint32_t step = 1, prev = lo;
        uint32_t cur = lo;
        while (cur < hi && arr(cur) < x) {
            prev = cur + 1;
            cur = (step >= hi - lo) ? hi : lo + step;
            step <<= 1;
        }
        lo = prev;
        hi = cur;  // arr[prev-1] < x <= arr[cur] (or cur == hi)
    }
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (arr(mid) < x) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Search modes of the probes: binary search, galloping, or galloping over blocks with a full
// compare of the last block (simd_galloping).
enum : int { SM_BINARY = 0, SM_GALLOP = 1, SM_BLOCK = 2 };
constexpr uint32_t kBlockPool = 32;  // block of a pool window: one 128-byte span, nine 16-byte loads

// Blocks [lo + W b, lo + W b + W) of arr[lo, hi): the first block whose last element is >= x, found
// by galloping over the blocks' last elements (blocks 0, 1, 2, 4, 8, ...) and a binary search of the
// blocks the gallop leaves -- gallop_wide and binary_search_wide of simd_galloping.rs:196-243 with
// GPU-sized blocks.  Returns the block, or the block count when every element is < x.
template <uint32_t W, class Arr>
__device__ __forceinline__ uint32_t gallop_blocks(const Arr &arr, uint32_t lo, uint32_t hi, uint32_t x)
{
    const uint32_t nbk = (hi - lo + W - 1) / W;
    auto last = [&](uint32_t b) {
        const uint32_t e = lo + W * b + W;
        return arr((e < hi ? e : hi) - 1);
    };
    uint32_t bl = 0, bh = 0, step = 1;
    while (bh < nbk && last(bh) < x) {
        bl = bh + 1;
        bh = (step >= nbk) ? nbk : step;
        step <<= 1;
    }
    while (bl < bh) {  // blocks < bl end below x; block bh (if any) ends at >= x
        const uint32_t mid = (bl + bh) >> 1;
        if (last(mid) < x) bl = mid + 1; else bh = mid;
    }
    return bl;
}

// Lower bound of x in L[lo, hi) by block galloping over a window of a resident pool, L = P + g, P
// readable up to pool elements and 16-byte aligned; the block that can hold x is counted in full
// (block_compare, simd_galloping.rs:272-296), W independent reads in place of the last log2(W)
// dependent steps: the last block is read as the aligned 16-byte chunks that cover it (one
// round trip).  Also reports whether the window holds x.  Pool values are compared XOR f (x is
// already in that space).
__device__ __forceinline__ uint32_t lower_bound_block_pool(const uint32_t *__restrict__ P, uint64_t pool, uint64_t g,
                                                           uint32_t lo, uint32_t hi, uint32_t x, uint32_t f, bool &found)
{
    constexpr uint32_t W = kBlockPool;
    const uint32_t *__restrict__ L = P + g;
    auto arr = [&](uint32_t i) { return L[i] ^ f; };
    const uint32_t b = gallop_blocks<W>(arr, lo, hi, x);
    const uint32_t s0 = lo + W * b;
    found = false;
    if (s0 >= hi) return hi;
    const uint64_t q0 = g + s0, q1 = g + ((hi - s0 < W) ? hi : s0 + W);
    const uint64_t c0 = q0 & ~3ull;
    uint32_t lt = 0;
    bool eq = false;
#pragma unroll
    for (int c = 0; c < (int)(W / 4) + 1; c++) {
        const uint64_t e = c0 + 4ull * (uint64_t)c;
        if (e < q1) {
            const uint4 v = load_chunk(P, pool, e);
            const uint32_t w[4] = {v.x ^ f, v.y ^ f, v.z ^ f, v.w ^ f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint64_t q = e + (uint64_t)j;
                const bool in = q >= q0 && q < q1;
                lt += (in && w[j] < x) ? 1u : 0u;
                eq |= in && w[j] == x;
            }
        }
    }
    found = eq;
    return s0 + lt;
}

constexpr uint64_t kNoPos = ~0ull;

// Entries <= x among arr[lo, hi) of a sorted array of n entries, hi - lo <= 16: the aligned 16-byte
// chunks that cover the range load together (one round trip).
__device__ __forceinline__ uint32_t count_le16(const uint32_t *__restrict__ arr, uint64_t n, uint64_t lo, uint64_t hi,
                                               uint32_t x)
{
    uint32_t cnt = 0;
    const uint64_t c0 = lo & ~3ull;
#pragma unroll
    for (int c = 0; c < 5; c++) {
        const uint64_t e = c0 + 4ull * (uint64_t)c;
        if (e < hi) {
            const uint4 v = load_chunk(arr, n, e);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint64_t q = e + (uint64_t)j;
                cnt += (q >= lo && q < hi && w[j] <= x) ? 1u : 0u;
            }
        }
    }
    return cnt;
}

// Pool index of x in B[g0, g1), or kNoPos, using idx[k] = B[32k] ^ f (every 32nd pool element, in
// the compare space) and, when given, the middle level mid[m] = idx[16 m]: a binary search over
// the middle-level entries inside the range, then the 16 index entries under the one found (one
// round trip), or, without the middle level, a binary search over the index entries; then the
// only 32-element line that can hold x, compared in full (eight 16-byte loads).  The range is
// sorted (one set), so the entries inside it are too.
__device__ __forceinline__ uint64_t index_probe(const uint32_t *__restrict__ B, uint64_t pool,
                                                const uint32_t *__restrict__ idx, const uint32_t *__restrict__ mid,
                                                uint64_t g0, uint64_t g1, uint32_t x, uint32_t f)
{
    if (g0 >= g1) return kNoPos;
    const uint64_t kb = (g0 + 31) / 32, ke = (g1 + 31) / 32;  // entries with 32k in [g0, g1)
    uint64_t k;                                                // first entry > x
    if (mid) {
        const uint64_t mb = (kb + kMidIdx - 1) / kMidIdx, me = (ke + kMidIdx - 1) / kMidIdx;
        uint64_t lo = mb, hi = me;  // first middle entry > x
        while (lo < hi) {
            const uint64_t m = (lo + hi) >> 1;
            if (mid[m] <= x) lo = m + 1; else hi = m;
        }
        // the first index entry > x lies in [L, H], at most 16 entries
        const uint64_t L = (lo > mb) ? kMidIdx * (lo - 1) + 1 : kb;
        const uint64_t H = (lo < me) ? kMidIdx * lo : ke;
        k = L + count_le16(idx, (pool + 31) / 32, L, H, x);
    } else {
        uint64_t lo = kb, hi = ke;
        while (lo < hi) {
            const uint64_t m = (lo + hi) >> 1;
            if (idx[m] <= x) lo = m + 1; else hi = m;
        }
        k = lo;
    }
    if (k == 0) return kNoPos;  // kb == 0 and x < B[0] = B[g0]
    const uint64_t base = 32 * (k - 1);  // the line [base, base+32) holds every candidate
    uint64_t hit = kNoPos;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const uint64_t e = base + 4ull * c;
        const uint4 v = load_chunk(B, pool, e);
        const uint32_t w[4] = {v.x ^ f, v.y ^ f, v.z ^ f, v.w ^ f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t q = e + (uint64_t)j;
            if (q >= g0 && q < g1 && q < pool && w[j] == x) hit = q;
        }
    }
    return hit;
}

// ---- wave-cooperative index lookups --------------------------------------------------------------
// A lookup through the B-pool index with its top level in LDS (every kTopStride-th element) searches
// the top level in LDS, then makes three dependent global reads: a 64-byte window of the middle
// level (every kMidStride-th element), a 64-byte window of the index (every 32nd element) and the
// 128-byte line of B that can hold x.  Read by the probe's own lane, each window is four or eight
// 16-byte loads to one line, and each load instruction of a wave touches 64 different lines: the
// vector memory pipeline looks every one of them up separately, and on resident pools that, not
// HBM, bounds the search tile.  Here a group of lanes reads one probe's window, one 16-byte chunk
// per lane, so an instruction reads 16 whole 64-byte windows (groups of 4) or 8 whole 128-byte lines
// (groups of 8); the probes' arguments reach the groups, and the counts come back, through
// cross-lane permutes.  Every lane of the wave must call these together.

__device__ __forceinline__ uint32_t lane_perm(uint32_t v, uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(src << 2), (int)v);
}

// The value of the lane 1 or 2 away in its group of four (xor), and of lane 7 - i of its eight, by DPP.
__device__ __forceinline__ uint32_t quad_xor1(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t quad_xor2(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t half_mirror(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false);
}

// For the probe x of every lane: entries <= x among positions [lo, hi) of the 16-entry block blk of
// arr (entries 16 blk .. 16 blk + 15, arr holding n entries); lh = lo | hi << 8, 0 for no window.
// Round r serves lanes 16 r .. 16 r + 15, one per group of 4 lanes; all four loads are in flight
// together.
__device__ __forceinline__ uint32_t coop_count16(const uint32_t *__restrict__ arr, uint64_t n, uint32_t blk, uint32_t lh,
                                                 uint32_t x)
{
    const uint32_t lane = lane_id();
    const uint32_t c = lane & 3u;  // the chunk this lane reads of the block it serves
    uint4 v[4];
    uint32_t plh[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t p = 16u * (uint32_t)r + (lane >> 2);  // the lane whose probe is served
        const uint32_t pb = lane_perm(blk, p);
        plh[r] = lane_perm(lh, p);
        v[r] = plh[r] ? load_chunk(arr, n, 16ull * pb + 4u * c) : make_uint4(0u, 0u, 0u, 0u);
    }
    uint32_t res = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t p = 16u * (uint32_t)r + (lane >> 2);
        const uint32_t px = lane_perm(x, p);
        const uint32_t lo = plh[r] & 0xFFu, hi = plh[r] >> 8;
        const uint32_t w[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
        uint32_t k = 0;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint32_t e = 4u * c + j;
            k += (e >= lo && e < hi && w[j] <= px) ? 1u : 0u;
        }
        k += quad_xor1(k);
        k += quad_xor2(k);
        const uint32_t t = lane_perm(k, 4u * (lane & 15u));  // lane 16 r + i reads group i
        if ((lane >> 4) == (uint32_t)r) res = t;
    }
    return res;
}

// The positions [from, to) of a 32-element line as a mask, from <= 31, to <= 32.
__device__ __forceinline__ uint32_t line_mask(uint32_t from, uint32_t to)
{
    return to > from ? (~0u >> (32u - to)) & (~0u << from) : 0u;
}

// For the probe x of every lane (in the compare space): the position of x in the 32-element line
// `line` of B (or of A, with AB and `a`; elements 32 line .. 32 line + 31) among the positions vm (0:
// no probe), or 32 when absent.  Without POS only whether x is there: 0 or 32.  Round r serves
// lanes 8 r .. 8 r + 7, one per group of 8 lanes; all eight loads are in flight together.
template <bool POS, bool AB>
__device__ __forceinline__ uint32_t coop_find32(const PairBatch &in, uint32_t line, uint32_t vm, bool a, uint32_t x)
{
    const uint32_t lane = lane_id();
    const uint32_t c = lane & 7u;
    uint4 v[8];
    uint32_t pvm[8];
    const uint64_t am = AB ? ballot(a) : 0ull;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint32_t p = 8u * (uint32_t)r + (lane >> 3);
        const uint32_t pl = lane_perm(line, p);
        pvm[r] = lane_perm(vm, p);
        const bool pa = AB && ((am >> p) & 1u);
        v[r] = pvm[r] ? load_chunk(pa ? in.A : in.B, pa ? in.a_pool : in.b_pool, 32ull * pl + 4u * c)
                      : make_uint4(0u, 0u, 0u, 0u);
    }
    uint32_t res = 32;
    const uint32_t xf = x ^ in.sflip;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint32_t px = lane_perm(xf, 8u * (uint32_t)r + (lane >> 3));
        const uint32_t eq = (v[r].x == px ? 1u : 0u) | (v[r].y == px ? 2u : 0u) | (v[r].z == px ? 4u : 0u) |
                            (v[r].w == px ? 8u : 0u);
        const uint32_t hit = eq & (pvm[r] >> (4u * c));  // one bit at most (a set holds x at most once)
        if constexpr (POS) {
            uint32_t h = hit ? 4u * c + (uint32_t)__builtin_ctz(hit) + 1u : 0u;  // position + 1
            h |= quad_xor1(h);
            h |= quad_xor2(h);
            h |= half_mirror(h);  // the other four lanes of the eight
            const uint32_t t = lane_perm(h, 8u * (lane & 7u));  // lane 8 r + i reads group i
            if ((lane >> 3) == (uint32_t)r) res = t ? t - 1u : 32u;
        } else {
            // group i of round r answers lane 8 r + i
            const uint64_t b = ballot(hit != 0);
            if ((lane >> 3) == (uint32_t)r) res = ((b >> (8u * (lane & 7u))) & 0xFFu) ? 0u : 32u;
        }
    }
    return res;
}

// Pool index of x in B[g0, g1) (without POS: any index of its line), or kNoPos, for the probe of every
// lane of the wave (on = false: no probe), through the top level top[j - tj0] = B[kTopStride j] in
// LDS, the middle level in.b_mid[m] = in.b_idx[kMidIdx m] and the index in.b_idx[k] = B[32 k] (values
// in the compare space), with the global reads made by groups of lanes.  The windows it reads
// each lie in one aligned block: the middle-level entries over one top-level interval are those of
// one 16-entry block (top entries are every 16th middle entry), likewise the index entries under one
// middle-level interval, and the candidates of B one 32-element line.
template <bool POS>
__device__ __forceinline__ uint64_t coop_index_probe_top(const PairBatch &in, bool on, const uint32_t *top, uint64_t tj0,
                                                         uint64_t g0, uint64_t g1, uint32_t x)
{
    on = on && g0 < g1;
    uint64_t L = 0, H = 0, mb = 0, me = 0;
    if (on) {
        const uint64_t kb = (g0 + 31) / 32, ke = (g1 + 31) / 32;
        const uint64_t jb = (kb + kTopIdx - 1) / kTopIdx, je = (ke + kTopIdx - 1) / kTopIdx;
        uint64_t lo = jb, hi = je;  // first top entry > x
        while (lo < hi) {
            const uint64_t m = (lo + hi) >> 1;
            if (top[m - tj0] <= x) lo = m + 1; else hi = m;
        }
        L = (lo > jb) ? kTopIdx * (lo - 1) + 1 : kb;
        H = (lo < je) ? kTopIdx * lo : ke;
        mb = (L + kMidIdx - 1) / kMidIdx;
        me = (H + kMidIdx - 1) / kMidIdx;
    }
    // middle level: [mb, me) inside block mb / 16
    const uint32_t mblk = (uint32_t)(mb >> 4);
    const uint32_t mlh = (on && me > mb) ? (uint32_t)(mb & 15u) | ((uint32_t)(me - 16ull * mblk) << 8) : 0u;
    const uint32_t mc = coop_count16(in.b_mid, (in.b_pool + kMidStride - 1) / kMidStride, mblk, mlh, x);
    uint64_t L2 = 0, H2 = 0;
    if (on) {
        const uint64_t ms = mb + mc;
        L2 = (ms > mb) ? kMidIdx * (ms - 1) + 1 : L;
        H2 = (ms < me) ? kMidIdx * ms : H;
    }
    // index: [L2, H2) inside block L2 / 16; the first entry > x is L2 + count
    const uint32_t iblk = (uint32_t)(L2 >> 4);
    const uint32_t ilh = (on && H2 > L2) ? (uint32_t)(L2 & 15u) | ((uint32_t)(H2 - 16ull * iblk) << 8) : 0u;
    const uint32_t ic = coop_count16(in.b_idx, (in.b_pool + 31) / 32, iblk, ilh, x);
    // B: the line [32(kk-1), 32 kk) holds every candidate; positions inside [g0, g1) and the pool
    const uint64_t kk = L2 + ic;
    const bool bon = on && kk > 0;
    const uint64_t base = bon ? 32 * (kk - 1) : 0;
    uint32_t vm = 0;
    if (bon) {
        const uint64_t e1 = min(g1, in.b_pool);
        vm = line_mask(g0 > base ? (uint32_t)min(g0 - base, (uint64_t)31) : 0u,
                       e1 > base && base + 32 > g0 ? (uint32_t)min(e1 - base, (uint64_t)32) : 0u);
    }
    const uint32_t pos = coop_find32<POS, false>(in, (uint32_t)(base >> 5), vm, false, x);
    return (vm && pos < 32) ? base + pos : kNoPos;
}

template <int NT, int KS, int MAXSEG, int CAPB, bool BSR, bool COUNT_ONLY, int SMODE, bool DIRECT = false>
__global__ __launch_bounds__(NT, 4) void search_tile_kernel(PairBatch in, TilePlan plan, TileOut out, uint32_t tile0)
{
    static_assert(KS >= 1 && KS <= 31, "lane masks hold KS bits");
    constexpr int U = NT * KS;
    constexpr int NW = NT / kWave;
    using Smem = SearchSmem<NT, KS, MAXSEG, CAPB, BSR>;
    __shared__ Smem sm;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t wave = tid / kWave;

    {
        // one tile per workgroup (a loop over tiles here costs ~20% on the merge kernel)
        const uint32_t t = tile0 + blockIdx.x;
        if (t >= plan.ntiles) return;
        // ---- 1. segment table, probe windows -------------------------------------------------------
        // DIRECT (the launch for plan.direct: one pair, or a batch of at most NT pairs): nothing
        // planned the tiles.  A batch's pair p owns the units (probes and padding) from the sum over
        // the pairs before it (a block scan, one pair per thread), and a tile's pairs are those its
        // unit range meets.  plan.single is uniform: every thread takes the branch or none.
        static_assert(!DIRECT || !BSR, "a direct tile holds plain pairs");
        constexpr bool direct = DIRECT;
        const bool dbatch = direct && !plan.single;
        if (direct && t == 0 && tid == 0 && out.error) *out.error = 0;  // before the flags below
        const uint64_t u0 = (uint64_t)t * U;
        uint32_t ulen = (uint32_t)((u0 + U < plan.utotal) ? U : plan.utotal - u0);
        uint32_t d_first = 0, d_last = 0;
        if constexpr (DIRECT) {
            if (!plan.single) {
                // pair tid's first unit and units go to LDS (the probe-key space, staged later)
                // for the segment table; the tile's first and last pairs after them
                if (tid == 0) {
                    sm.pkey[2 * NT] = ~0u;
                    sm.pkey[2 * NT + 1] = ~0u;
                }
                const bool own = tid < in.P;
                const uint32_t v = own ? (uint32_t)pair_units(in, plan.policy, plan.c0, tid) : 0u;
                uint32_t tu = 0;
                const uint32_t pu = block_exclusive_scan<NT>(v, sm.scan_scratch, &tu);
                // the device sizes must give the units the host planned for (as the plan checks)
                if (t == 0 && tid == 0 && out.error && (uint64_t)tu != plan.utotal) atomicOr(out.error, 4u);
                if (own) {
                    sm.pkey[2 * tid] = pu;
                    sm.pkey[2 * tid + 1] = v;
                    const uint64_t ue = u0 + ulen - 1;  // the tile's last unit
                    if (pu <= u0 && u0 < (uint64_t)pu + v) sm.pkey[2 * NT] = tid;
                    if (pu <= ue && ue < (uint64_t)pu + v) sm.pkey[2 * NT + 1] = tid;
                }
                __syncthreads();  // also: the scratch is scanned again below
                d_first = sm.pkey[2 * NT];
                d_last = sm.pkey[2 * NT + 1];
            }
        }
        const uint32_t p_first = direct ? d_first : plan.tile_first[t];
        const uint32_t p_last = direct ? d_last : plan.tile_last[t];
        uint32_t nseg = p_last - p_first + 1;
        bool bad = p_last < p_first || nseg > (uint32_t)MAXSEG || p_last >= in.P;
        if (bad) nseg = 0;
        if (t == 0 && tid == 0 && out.error && !direct && plan.uoff[in.P] != plan.utotal) atomicOr(out.error, 4u);
        if (dbatch && tid == 0) {  // the tile maps the placement reads
            plan.tile_first[t] = bad ? 0u : p_first;
            plan.tile_last[t] = bad ? ~0u : p_last;
        }
        uint32_t seg_pu = 0;  // direct batch: the segment's pair's first unit
        uint32_t cp = 0;
        uint64_t gp = 0;
        uint32_t swap = 0;
        // the span of the tile's larger B sets, for the top level of the B-pool index (1b)
        unsigned long long gmin = ~0ull, gmax = 0;
        if (tid < nseg) {
            SegWin w;
            if (dbatch) {
                const uint32_t p = p_first + tid;
                seg_pu = sm.pkey[2 * p];
                w = search_direct_window(in, p, seg_pu, sm.pkey[2 * p + 1], u0, ulen);
            } else {
                w = direct ? direct_window(plan) : seg_window(in, plan, t, p_first, nseg, tid, ulen);
            }
            swap = (w.nb < w.na) ? 1u : 0u;  // probes come from the smaller side
            gp = (swap ? w.b : w.a) + w.i0;
            const uint32_t n = (uint32_t)(w.i1 - w.i0);
            cp = n ? ((uint32_t)(gp & 3) + n + 3) / 4 : 0u;
            sm.seg_u[tid] = w.u;
            sm.seg_wa[tid] = n;
            sm.seg_flags[tid] = w.flags | (swap << 2);
            sm.seg_lbase[tid] = swap ? w.a : w.b;
            sm.seg_hi[tid] = (uint32_t)(swap ? w.na : w.nb);  // larger size until narrowed
            if (!swap && w.nb > 0) {
                gmin = w.b;
                gmax = w.b + w.nb;
            }
        }
        if (in.b_top) {
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                gmin = min(gmin, (unsigned long long)__shfl_xor(gmin, d, kWave));
                gmax = max(gmax, (unsigned long long)__shfl_xor(gmax, d, kWave));
            }
            if (lane == 0) {
                sm.red64[wave][0] = gmin;
                sm.red64[wave][1] = gmax;
            }
        }
        uint32_t tot = 0;
        const uint32_t pfx = block_exclusive_scan<NT>(cp, sm.scan_scratch, &tot);
        if (4u * tot + 8u > (uint32_t)Smem::PKEYS) bad = true;  // not reachable by the unit bound
        if (tid < nseg) {
            sm.win_c[tid] = pfx;
            sm.win_g[tid] = gp & ~3ull;
            sm.win_src[tid] = swap;
            sm.seg_la[tid] = 4u * pfx + (uint32_t)(gp & 3);
        }
        if (tid == 0) {
            sm.win_c[nseg] = tot;
            sm.seg_u[nseg] = ulen;
        }
        __syncthreads();
        // ---- 1b. top level of the B-pool index over the tile's larger B sets, loaded together with
        // the probe windows (one round trip for both) ---------------------------------------------------
        bool top_ok = false;
        uint64_t tj0 = 0;
        uint64_t tn = 0;
        if (in.b_top && !bad) {
            gmin = ~0ull;
            gmax = 0;
#pragma unroll
            for (int k = 0; k < NW; k++) {
                gmin = min(gmin, sm.red64[k][0]);
                gmax = max(gmax, sm.red64[k][1]);
            }
            if (gmax > gmin) {
                // entries j with kTopStride j in [gmin, gmax)
                tj0 = (gmin + kTopStride - 1) / kTopStride;
                tn = (gmax + kTopStride - 1) / kTopStride - tj0;
                top_ok = tn <= (uint64_t)kTopCap;
            }
        }
        if (bad) {
            nseg = 0;
            ulen = 0;
            if (tid == 0 && out.error) atomicOr(out.error, 2u);
        } else {
            // the top level goes straight to LDS (4 bytes per lane, a wave's row of 64 entries per
            // load), in flight with the windows' loads and holding no registers meanwhile
            if (top_ok) {
                for (uint32_t r = tid - lane; r < (uint32_t)tn; r += NT)  // r: the wave's row (uniform)
                    if (r + lane < (uint32_t)tn)
                        __builtin_amdgcn_global_load_lds(in.b_top + tj0 + r + lane, sm.top + r, 4, 0, 0);
            }
            constexpr int QP = (Smem::PKEYS + 4 * NT - 1) / (4 * NT);
            stage_windows<NT, QP>(in.A, in.a_pool, in.B, in.b_pool, sm.win_c, sm.win_g, sm.win_src, nseg, sm.pkey,
                                  in.sflip);
            if constexpr (BSR)
                stage_windows<NT, QP>(in.As, in.a_pool, in.Bs, in.b_pool, sm.win_c, sm.win_g, sm.win_src, nseg, sm.pst,
                                      0u);
            if (top_ok) __builtin_amdgcn_s_waitcnt(0);  // the direct-to-LDS loads have landed
        }
        __syncthreads();

        // ---- 2. narrow the larger sets of the pairs that other tiles share ----------------------------
        // At most the first and the last segment are parts of a pair; their probes reach only a
        // part of the larger set, whose bounds four waves find, one 64-way search each.  A pair that
        // lies whole in the tile searches its whole larger set: narrowing one would cost two
        // searches of dependent reads, one pair after another (a tile of 130 small pairs waited for
        // 33 of them).  A larger set longer than kNoNarrow in an indexed pool whose top level is
        // staged is not narrowed either: every probe finds its line through the index.
        static_assert(NW == 4, "one wave per bound");
        auto through_index = [&](uint32_t swapped, uint32_t nl) {
            return top_ok && in.b_idx && !swapped && nl > kNoNarrow;
        };
        auto partial = [&](uint32_t s) {
            const uint32_t f = sm.seg_flags[s];
            return sm.seg_wa[s] && (f & 3u) != 3u && !through_index((f >> 2) & 1u, sm.seg_hi[s]);
        };
        if (nseg) {
            const uint32_t s = wave < 2 ? 0u : nseg - 1;
            if ((wave < 2 || s != 0) && partial(s)) {
                const bool large_is_a = (sm.seg_flags[s] >> 2) & 1u;
                const uint32_t *__restrict__ L = (large_is_a ? in.A : in.B) + sm.seg_lbase[s];
                const uint32_t nl = sm.seg_hi[s], f = in.sflip;
                const uint32_t v = sm.pkey[sm.seg_la[s] + ((wave & 1u) ? sm.seg_wa[s] - 1 : 0u)];
                const bool up = (wave & 1u) != 0;
                const uint32_t r = (uint32_t)group_partition_point<kWave>(0, nl, lane, 0, [&](uint64_t x) {
                    const uint32_t y = L[x] ^ f;
                    return up ? y <= v : y < v;
                });
                if (lane == 0) sm.narrow[wave] = r;
            }
        }
        __syncthreads();

        // ---- 3. stage or sample the larger windows while they fit -------------------------------------
        // A window of at most kStage elements per probe is staged whole.  Of a longer one LDS gets
        // the first element of every m-th 128-byte line: at most kSample samples per probe, each
        // line's read when it is the one that can hold a probe (4b).  So a probe costs at most kSample
        // lines of samples (fewer through the index) and one line of the set, in two round trips,
        // where a gallop or binary search from the window's start reads a line per level.  The limits
        // are what LDS holds beside four workgroups per CU.  (3,000 pairs of larger sets of 2^12 to
        // 2^16 elements and ratios up to 4,096: the whole batch 279 us with narrowed windows searched
        // in global memory, 239 us sampled, 208 us with the staged ones searched as in 4a.)
        uint32_t nst = 0;   // segments whose windows fit
        uint32_t ltot = 0;  // chunks of staged and sampled windows (0: every probe goes through the index)
        constexpr uint32_t kStage = CAPB / U - 1, kSample = CAPB / U > 5 ? 4 : CAPB / U - 1, kMinSample = 24;
        {
            LargeWindow lw{};
            uint32_t src = 0;
            bool idx = false;
            if (tid < nseg) {
                const uint32_t k = sm.seg_wa[tid], f = sm.seg_flags[tid];
                uint32_t lo = 0, hi = k ? sm.seg_hi[tid] : 0u;
                idx = through_index((f >> 2) & 1u, sm.seg_hi[tid]);
                if (partial(tid) && (tid == 0 || tid == nseg - 1)) {
                    lo = sm.narrow[tid == 0 ? 0 : 2];
                    hi = sm.narrow[tid == 0 ? 1 : 3];
                }
                src = ((f >> 2) & 1u) ? 0u : 1u;  // pool of the larger side
                const uint64_t base = sm.seg_lbase[tid];
                if (idx) lw = LargeWindow{base + lo, lo, hi, 0, 0, 0};
                else lw = large_window(base, lo, hi, k, kStage, kSample, kMinSample);
            }
            const uint32_t cl = lw.cl, m = lw.m;
            const uint64_t gl = lw.g;
            const uint32_t lpfx = block_exclusive_scan<NT>(cl, sm.scan_scratch, &ltot);
            const bool fits = lpfx + cl <= (uint32_t)(CAPB / 4);
            // the segments that fit form a prefix; their count is the number of fitting threads
            {
                const uint64_t bal = ballot(tid < nseg && fits);
                if (lane == 0) sm.wave_el[wave] = (uint32_t)__popcll(bal);
            }
            __syncthreads();
            for (int k = 0; k < NW; k++) nst += sm.wave_el[k];
            if (tid < nseg) {
                sm.seg_lo[tid] = lw.lo;
                sm.seg_hi[tid] = lw.hi;
                sm.seg_m[tid] = m;
                sm.seg_flags[tid] |= lw.ns << 8;
                if (fits) {
                    sm.win_c[tid] = lpfx;
                    sm.win_g[tid] = m ? gl : gl & ~3ull;
                    sm.win_src[tid] = src;
                    sm.seg_lb[tid] = idx ? kNotStaged : 4u * lpfx + (m ? 0u : (uint32_t)(gl & 3));
                } else {
                    sm.seg_lb[tid] = kNotStaged;
                }
                if (tid + 1 == nst) sm.win_c[nst] = lpfx + cl;
            }
            if (tid == 0 && nst == 0) sm.win_c[0] = 0;
            __syncthreads();
            if (nst) {
                constexpr int QL = (CAPB + 4 * NT - 1) / (4 * NT);
                stage_or_sample<NT, QL>(in, sm.win_c, sm.win_g, sm.win_src, sm.seg_m, sm.seg_flags, nst, sm.lkey);
                if constexpr (BSR)
                    stage_windows<NT, QL>(in.As, in.a_pool, in.Bs, in.b_pool, sm.win_c, sm.win_g, sm.win_src, nst,
                                          sm.lst, 0u, sm.seg_m);
            }
            __syncthreads();
        }

        // ---- 3b. further sets (a single pair, plain sets: small_adaptive over k sets) -----------------
        // Every probe found in the pair's larger set is also looked up in each further set in turn
        // (adaptive.rs:107-147); each further set is narrowed to the tile's probe range here, one
        // wave per set, and each lane gallops forward through it from there.
        uint32_t xcur[kMaxExtraSets];
        const uint32_t nx = (!BSR && nseg == 1 && sm.seg_wa[0] > 0) ? in.nx : 0u;
        if (nx) {
            const uint32_t vf = sm.pkey[sm.seg_la[0]], vl = sm.pkey[sm.seg_la[0] + sm.seg_wa[0] - 1];
            for (uint32_t j = wave; j < nx; j += NW) {
                const uint32_t *__restrict__ X = in.xsets[j];
                const uint64_t nxj = in.xlens[j];
                const uint32_t f = in.sflip;
                const uint32_t lo = (uint32_t)group_partition_point<kWave>(0, nxj, lane, 0,
                                                                           [&](uint64_t i) { return (X[i] ^ f) < vf; });
                const uint32_t hi = (uint32_t)group_partition_point<kWave>(
                    lo, nxj, lane, 0, [&](uint64_t i) { return (X[i] ^ f) <= vl; });
                if (lane == 0) {
                    sm.xlo[j] = lo;
                    sm.xhi[j] = hi;
                }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < (uint32_t)kMaxExtraSets; j++) xcur[j] = (j < nx) ? sm.xlo[j] : 0u;
        }

        // ---- 4. lookups --------------------------------------------------------------------------
        const uint32_t ub = tid * KS;
        uint32_t hmask = 0, nelems = 0;
        uint32_t svals[BSR ? KS : 1];
        uint32_t s0 = 0;
        if (ub < ulen) {
            uint32_t lo = 0, hi = nseg;  // largest s with seg_u[s] <= ub
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (sm.seg_u[mid] <= ub) lo = mid; else hi = mid;
            }
            s0 = lo;
        }
        // fmask: the lane's probes found (bit k); BSR also keeps their states in the larger set.  A set
        // holds x at most once, so where a search starts does not change what it finds.  (Four probes
        // per lane: the loops of 4a and 4b are not unrolled, so that a lookup's registers are held once.)
        constexpr int UK = (BSR || KS <= 2) ? KS : 1;
        uint32_t fmask = 0;
        uint32_t lstate[BSR ? KS : 1];
        // 4a. probes of windows staged whole: binary lifting in LDS with the wave's common steps, the KS
        // searches in lockstep, so that their reads overlap (two probes, windows of up to 3,000
        // elements: 2,900 cycles where galloping through them in turn takes 6,500)
        if (ltot) {
            LiftRange r[KS];
            uint32_t xv[KS], nmax = 0, s = s0;
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const uint32_t u = ub + (uint32_t)k;
                r[k] = lift_range(0, 0);
                xv[k] = 0;
                if (u < ulen) {
                    while (u >= sm.seg_u[s + 1]) s++;
                    const uint32_t e = u - sm.seg_u[s], lb = sm.seg_lb[s];
                    if (e < sm.seg_wa[s] && lb != kNotStaged && sm.seg_m[s] == 0) {
                        const uint32_t n = sm.seg_hi[s] - sm.seg_lo[s];
                        xv[k] = sm.pkey[sm.seg_la[s] + e];
                        r[k] = lift_range(lb, n);
                        nmax = max(nmax, n);
                    }
                }
            }
            const uint32_t L = wave_max_u32(32u - (uint32_t)__clz(nmax));
            for (int bit = (int)L - 1; bit >= 0; bit--) {
#pragma unroll
                for (int k = 0; k < KS; k++) {
                    const uint32_t y = lift_to(r[k], 1u << bit);
                    // (at its window's end, or without one, a probe stays: y == at)
                    if (sm.lkey[y - 1] < xv[k]) r[k].at = y;
                }
            }
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const bool found = r[k].at < r[k].end && sm.lkey[r[k].at] == xv[k];
                fmask |= found ? 1u << k : 0u;
                if constexpr (BSR) lstate[k] = found ? sm.lst[r[k].at] : 0u;
            }
        }
        // 4b. probes of sampled windows, the whole wave together, the k-th probe of every lane at once:
        // the samples at most x give the m lines that can hold it, a search over those lines' first
        // elements (m > 1) the one line, which a group of lanes reads.
        if (ltot) {
            uint32_t s = s0;
#pragma unroll UK
            for (int k = 0; k < KS; k++) {
                const uint32_t u = ub + (uint32_t)k;
                uint32_t x = 0, line = 0, vm = 0;
                bool in_a = false;
                if (u < ulen) {
                    while (u >= sm.seg_u[s + 1]) s++;
                    const uint32_t e = u - sm.seg_u[s];
                    const uint32_t m = sm.seg_m[s], lb = sm.seg_lb[s];
                    if (m && lb != kNotStaged && e < sm.seg_wa[s]) {
                        x = sm.pkey[sm.seg_la[s] + e];
                        const uint32_t f = sm.seg_flags[s];
                        const bool large_is_a = (f >> 2) & 1u;
                        const uint64_t base = sm.seg_lbase[s];
                        const uint64_t g0 = base + sm.seg_lo[s], g1 = base + sm.seg_hi[s];
                        uint32_t lo = 0, hi = f >> 8;  // samples at most x
                        while (lo < hi) {
                            const uint32_t mid = (lo + hi) >> 1;
                            if (sm.lkey[lb + mid] <= x) lo = mid + 1; else hi = mid;
                        }
                        line = (uint32_t)(g0 >> 5) + lo * m;
                        if (m > 1) {
                            const uint32_t end = (uint32_t)((g1 - 1) >> 5) + 1;
                            uint32_t n = min(m, end - line);  // the last of n lines whose first element is at most x
                            while (n > 1) {
                                const uint32_t h = n >> 1, q = line + h;
                                const uint32_t y = (in.b_idx && !large_is_a)
                                                       ? in.b_idx[q]
                                                       : (large_is_a ? in.A : in.B)[32ull * q] ^ in.sflip;
                                if (y <= x) {
                                    line = q;
                                    n -= h;
                                } else {
                                    n = h;
                                }
                            }
                        }
                        const uint64_t l0 = 32ull * line;
                        const uint32_t from = g0 > l0 ? (uint32_t)(g0 - l0) : 0u;
                        vm = line_mask(from, (uint32_t)min(g1 - l0, (uint64_t)32));
                        in_a = large_is_a;
                    }
                }
                if (ballot(vm != 0) != 0) {  // wave-uniform
                    const uint32_t pos = coop_find32<BSR, true>(in, line, vm, in_a, x);
                    if (vm && pos < 32) {
                        fmask |= 1u << k;
                        if constexpr (BSR) lstate[k] = (in_a ? in.As : in.Bs)[32ull * line + pos];
                    }
                }
            }
        }
        // probes answered through the indexed B pool with its top level staged, likewise
        if (top_ok && in.b_idx) {
            // one probe per lane at a time (two at once measured no faster at two probes per lane and
            // slower at four, where the registers of the second cost occupancy)
            uint32_t s = s0;
#pragma unroll UK
            for (int k = 0; k < KS; k++) {
                const uint32_t u = ub + (uint32_t)k;
                bool on = u < ulen;
                uint32_t x = 0;
                uint64_t g0 = 0, g1 = 0;
                if (on) {
                    while (u >= sm.seg_u[s + 1]) s++;
                    const uint32_t e = u - sm.seg_u[s];
                    on = e < sm.seg_wa[s] && sm.seg_lb[s] == kNotStaged && !((sm.seg_flags[s] >> 2) & 1u);
                    if (on) {
                        x = sm.pkey[sm.seg_la[s] + e];
                        g0 = sm.seg_lbase[s] + sm.seg_lo[s];
                        g1 = sm.seg_lbase[s] + sm.seg_hi[s];
                    }
                }
                if (ballot(on) != 0) {  // wave-uniform
                    const uint64_t q = coop_index_probe_top<BSR>(in, on, sm.top, tj0, g0, g1, x);
                    if (q != kNoPos) {
                        fmask |= 1u << k;
                        if constexpr (BSR) lstate[k] = in.Bs[q];
                    }
                }
            }
        }
        // 4c. probes of windows that found no room in LDS, each by its lane
        if (nst < nseg && ub < ulen) {
            uint32_t s = s0;
#pragma unroll UK
            for (int k = 0; k < KS; k++) {
                const uint32_t u = ub + (uint32_t)k;
                if (u >= ulen) break;
                while (u >= sm.seg_u[s + 1]) s++;
                const uint32_t e = u - sm.seg_u[s];
                const bool large_is_a = (sm.seg_flags[s] >> 2) & 1u, idx = in.b_idx && !large_is_a;
                if (e >= sm.seg_wa[s] || sm.seg_lb[s] != kNotStaged || (idx && top_ok)) continue;
                const uint32_t x = sm.pkey[sm.seg_la[s] + e], lo = sm.seg_lo[s], hi = sm.seg_hi[s];
                const uint64_t g = sm.seg_lbase[s];
                bool found;
                uint64_t q = 0;
                if (idx) {
                    // the index, then one 128-byte line
                    q = index_probe(in.B, in.b_pool, in.b_idx, in.b_mid, g + lo, g + hi, x, in.sflip);
                    found = q != kNoPos;
                } else if constexpr (SMODE == SM_BLOCK) {
                    q = g + lower_bound_block_pool(large_is_a ? in.A : in.B, large_is_a ? in.a_pool : in.b_pool, g, lo,
                                                   hi, x, in.sflip, found);
                } else {
                    const uint32_t *__restrict__ L = (large_is_a ? in.A : in.B) + g;
                    const uint32_t f = in.sflip;
                    auto arr = [&](uint32_t i) { return L[i] ^ f; };
                    const uint32_t pos = lower_bound_from<SMODE == SM_GALLOP>(arr, lo, hi, x);
                    found = pos < hi && arr(pos) == x;
                    q = g + pos;
                }
                if (found) {
                    fmask |= 1u << k;
                    if constexpr (BSR) lstate[k] = (large_is_a ? in.As : in.Bs)[q];
                }
            }
        }
        hmask = fmask;
        if constexpr (BSR) {
            // a base match is a result when the state AND is non-zero
            uint32_t s = s0;
#pragma unroll
            for (int k = 0; k < KS; k++) {
                svals[k] = 0;
                if ((fmask >> k) & 1u) {
                    const uint32_t u = ub + (uint32_t)k;
                    while (u >= sm.seg_u[s + 1]) s++;
                    svals[k] = sm.pst[sm.seg_la[s] + (u - sm.seg_u[s])] & lstate[k];
                    nelems += __popc(svals[k]);
                    if (!svals[k]) hmask &= ~(1u << k);
                }
            }
        }
        if constexpr (!BSR) {
            // further sets of a single pair, in order; the first one that lacks x ends the lookup
            if (nx) {
                for (uint32_t m = fmask; m; m &= m - 1) {
                    const uint32_t k = __builtin_ctz(m);
                    const uint32_t x = sm.pkey[sm.seg_la[0] + (ub + k - sm.seg_u[0])], f = in.sflip;
                    bool found = true;
#pragma unroll
                    for (uint32_t j = 0; j < (uint32_t)kMaxExtraSets; j++) {
                        if (!found || j >= nx) continue;
                        const uint32_t *__restrict__ X = in.xsets[j];
                        auto xarr = [&](uint32_t i) { return X[i] ^ f; };
                        const uint32_t xh = sm.xhi[j];
                        const uint32_t xp = lower_bound_from<SMODE != SM_BINARY>(xarr, xcur[j], xh, x);
                        xcur[j] = xp;
                        found = xp < xh && xarr(xp) == x;
                    }
                    if (!found) hmask &= ~(1u << k);
                }
            }
        }
        if constexpr (!BSR) {
            // k-set groups: each hit is looked up in its pair's further sets in B, in order; the
            // first that lacks it drops it (small_adaptive's walk, adaptive.rs:107-147, one element
            // at a time: each lookup searches the whole further set).  A pass of its own after the
            // lookups, so its state is not live beside theirs.
            if (in.x_off && hmask) {
                uint32_t s = s0;
                for (int k = 0; k < KS; k++) {
                    if (!((hmask >> k) & 1u)) continue;
                    const uint32_t u = ub + (uint32_t)k;
                    while (u >= sm.seg_u[s + 1]) s++;
                    const uint32_t x = sm.pkey[sm.seg_la[s] + (u - sm.seg_u[s])];
                    const uint64_t p = (uint64_t)p_first + s;
                    const uint64_t j1 = in.x_off[p + 1];
                    bool found = true;
                    for (uint64_t j = in.x_off[p]; found && j < j1; j++) {
                        // a range is read only inside the pool (and its index)
                        const uint64_t g1 = min(in.x_end[j], in.b_pool), g0 = min(in.x_beg[j], g1);
                        if (in.b_idx) {
                            found = index_probe(in.B, in.b_pool, in.b_idx, in.b_mid, g0, g1, x, in.sflip) != kNoPos;
                        } else if (g1 > g0) {
                            const uint32_t n = (uint32_t)(g1 - g0);
                            if constexpr (SMODE == SM_BLOCK) {
                                (void)lower_bound_block_pool(in.B, in.b_pool, g0, 0u, n, x, in.sflip, found);
                            } else {
                                const uint32_t *__restrict__ X = in.B + g0;
                                const uint32_t f = in.sflip;
                                auto xarr = [&](uint32_t i) { return X[i] ^ f; };
                                const uint32_t xp = lower_bound_from<false>(xarr, 0u, n, x);
                                found = xp < n && xarr(xp) == x;
                            }
                        } else {
                            found = false;
                        }
                    }
                    if (!found) hmask &= ~(1u << k);
                }
            }
        }
        const uint32_t nwords = __popc(hmask);
        if constexpr (!BSR) nelems = nwords;

        // ---- 5. tile scan, staged outputs, counts ------------------------------------------------------
        const uint32_t pfx2 = block_exclusive_scan<NT>(nwords, sm.scan_scratch, &tot);
        sm.lane_mask[tid] = hmask;
        sm.lane_pfx[tid] = pfx2;
        if constexpr (BSR) {
            uint32_t el = nelems;
#pragma unroll
            for (int dd = 1; dd < kWave; dd <<= 1) el += __shfl_xor(el, dd, kWave);
            if (lane == 0) sm.wave_el[wave] = el;
        }
        __syncthreads();
        if constexpr (!COUNT_ONLY) {
            uint32_t *dk = plan.stage + (uint64_t)t * plan.stage_words;
            uint32_t *ds = dk + plan.stage_words / 2;
            uint32_t pos = pfx2;
            // the one tile of a direct run writes to the caller's output: no further than its capacity
            // (device sizes beyond the planned ones, flagged above, may find more results than it has room
            // for).  Of a run of several tiles nothing beyond the capacity is placed.
            const uint32_t room = (uint32_t)min(out.cap, (uint64_t)U);
            uint32_t s = s0;
#pragma unroll
            for (int k = 0; k < KS; k++) {
                const uint32_t u = ub + (uint32_t)k;
                if (hmask & (1u << k)) {
                    while (u >= sm.seg_u[s + 1]) s++;
                    if (DIRECT && pos >= room) break;
                    dk[pos] = sm.pkey[sm.seg_la[s] + (u - sm.seg_u[s])] ^ in.sflip;  // the value as given
                    if constexpr (BSR) ds[pos] = svals[k];
                    pos++;
                }
            }
        }
        if (tid == 0) {
            uint32_t el = tot;
            if constexpr (BSR) {
                el = 0;
                for (int k = 0; k < NW; k++) el += sm.wave_el[k];
            }
            plan.tile_count[t] = tot;
            plan.tile_elems[t] = el;
            if (plan.one_tile) {  // one tile: its counts are the totals, its results the output
                if (out.totals) {
                    out.totals[0] = tot;
                    out.totals[1] = el;
                }
                if (out.out_off) out.out_off[in.P] = tot;
            }
        }
        if (tid < nseg) {
            auto before = [&](uint32_t x) -> uint32_t {
                if (x >= ulen) return tot;
                const uint32_t l = x / KS, k = x % KS;
                return sm.lane_pfx[l] + __popc(sm.lane_mask[l] & ((1u << k) - 1u));
            };
            const uint32_t c0v = before(sm.seg_u[tid]);
            const uint32_t c = before(sm.seg_u[tid + 1]) - c0v;
            const uint32_t f = sm.seg_flags[tid];
            const uint64_t p = (uint64_t)p_first + tid;
            if (f & 1u) {
                plan.pair_local[p] = c0v;
                if (dbatch) plan.uoff[p] = seg_pu;  // for the placement (no plan wrote it)
            }
            if (plan.one_tile && out.out_off) out.out_off[p] = c0v;  // every pair lies in the one tile
            if (out.counts && (!direct || plan.one_tile)) {  // else the placement writes them
                if ((f & 3u) == 3u) out.counts[p] = c;
                else if (c) atomicAdd(&out.counts[p], c);
            }
        }
    }
}

} // namespace setops
