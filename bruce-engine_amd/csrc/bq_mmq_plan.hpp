// bq_mmq_plan.hpp -- which launch a prefill GEMM takes (token-tile height, K
// split, leftover-tile split), the workspace that choice can use, and which
// tile and K slice each block of the launch computes.  Arithmetic on the shape
// alone, without HIP: tests/test_mmq_plan.py builds it with the host compiler.
#pragma once
#include <stddef.h>

#include <algorithm>
#include <cmath>

namespace bq {

constexpr int kTN = 128;   // weight rows per tile
constexpr int kXcds = 8;

#ifdef __HIPCC__
#define BQ_HD __host__ __device__ __forceinline__
#else
#define BQ_HD inline
#endif

// Leftover-tile K split.  A launch of T tiles on C CUs runs for as long as its
// busiest CU, which gets ceil(T / C) tiles; with T = q * C + L (0 < L < C)
// every CU but L of them idles for the last tile's duration.  The tail split
// runs the first q * C tiles whole and cuts each of the L leftover tiles into
// k K slices, so the leftover work spreads over L * k pieces; the slices'
// partial tiles go to the caller's workspace [slice][leftover tile][TM][128]
// and k_sum_tail adds them in slice order.  k == 1: no tail split (the
// uniform K split or no split at all).
struct TailSplit {
    int k = 1;        // slices per leftover tile
    int nfull = 0;    // tiles run whole (tile indices 0 .. nfull-1)
    int gridfull = 0; // blocks of the whole tiles (a multiple of the XCD count)
    int nleft = 0;    // leftover tiles (indices nfull .. nfull+nleft-1)
};

// K split.  A launch with fewer tiles than the workgroup slots (two per CU
// for the 128-token tiles, three for the 32-token tiles; 512 / 768 on
// MI355X's 256 CUs) leaves CUs idle (one token tile of a 9216-row matrix: 72
// tiles), so it may be split over K into up to kMaxKSplit slices of whole K
// units (stage pairs for the DMA-staged kernels, stages for the raw tier) when
// the caller's workspace holds the slices' partial outputs
// [slice][part][rows][N[part]]; one more launch sums them in a fixed order.  The
// choice depends only on the shape and the workspace size, so equal calls take
// equal paths (eager or captured in a graph) and give equal bits.
//
// Leftover-tile split: k = 2 .. kMaxTailSplit slices per leftover tile, if that
// takes at least half a tile off the busiest CU's ceil(tiles / CUs).  Measured
// (9216 x 3072 W144, eager launches, us, unsplit -> split): 2048 rows (k = 2,
// 0.5 tile) 181.5 -> 168.5; smaller gains did not pay for the shorter slices and
// the summing launch (2560 rows, k = 3 for 0.33 tile: 216 -> 218), nor did more
// than 4 slices (2304 rows, k = 8: 220 -> 227).  With one whole tile per CU each
// runs alone on its CU and the leftover slices lose (512 x 9216 W144, 128-token
// tiles: 62 -> 67 us).
constexpr int kMaxKSplit = 8, kMaxTailSplit = 4;

// Cost of one 128-value stage of a tile, us per workgroup and CU of a full GPU
// (c128, c32: by tile height), and the W144 tier's min term, which is part of an
// unsplit tile's cost and all in the first slice of a split one: w less per
// stage there, and min_us per stage of the whole K.
struct TileCost {
    float c128, c32;
    float w128, w32, min_us;
    bool stage_units;  // slices at 128-value stages (else at stage pairs)
    bool tail;         // the kernel takes the leftover-tile split
    constexpr int units(int K) const { return stage_units ? K >> 7 : K >> 8; }
};
constexpr TileCost kCostW144 = {1.27f, 0.415f, 0.21f, 0.076f, 0.108f, false, true};
constexpr TileCost kCostRaw = {1.60f, 0.623f, 0.f, 0.f, 0.f, true, true};
constexpr TileCost kCostQ6 = {2.02f, 0.60f, 0.f, 0.f, 0.f, false, false};

// A tile height: the workgroups a CU holds at once, us before the first stage
// and after the last, and what a CU's last round costs, by its workgroups.
struct TileHeight {
    int tm, round;
    float start, last[3];
};
constexpr TileHeight kTileHeights[2] = {{128, 2, 5.2f, {1.55f, 2.06f}}, {32, 3, 4.0f, {1.61f, 2.21f, 3.01f}}};
constexpr float kSumUs = 2.3f, kSumTailUs = 4.4f, kPartialUs = 0.42e-6f;  // sum launches; per byte of partials

// One launch a GEMM may take, what it writes to the workspace, and the
// estimate of its time:
//   start + stages per slice x c x load + (sum launch + its partials if split),
// load = the workgroups of the busiest CU (as the XCDs are dealt) in whole rounds,
// plus the last round's cost; with the leftover split its whole tiles + slices / k.
// Fitted to the times of every height and split of 1512 shapes (9 .. 4096 rows, K
// 768 .. 9216, N 512 .. 18432, all tiers; from 45 us on each launch repeated for
// 12 ms, because the clock falls), minimising the time of the launch chosen: 0.8%
// (W144), 0.4% (raw), 0.2% (Q6_K) over the fastest launch in the geometric mean.
// The estimate it replaces, fitted to 9 shapes without a price on partials and
// leftover sums, was 2.0 / 1.1 / 1.2% over it, and up to 15% slower than the one
// before that: 9216 x 3072 W144 at 1279 rows 119.6 us (now 110.8), Q6_K 3200 x 8960
// at 253 rows 57.0 (49.3), raw 6912 x 2048 at 247 rows 31.8 (26.5).  Over 640 other
// shapes in turn W144 1.9, raw 3.2, Q6_K 2.6% faster (one 6%, four 3-4% slower).
struct TilePick {
    int tm = 128, ks = 1;
    TailSplit ts;
    size_t ws_floats = 0;
    float us = 0.f;
};

// Calls f with every launch `rows` x ntot x K may take: both heights, every count
// of slices with a longest slice of its own, every leftover split that saves more
// than one of fewer slices.
// `cus`: the CU count of the device the launch runs on (MI355X: 256).
template <typename F>
inline void mmq_launches(int rows, int K, int ntot, const TileCost& tc, int cus, F&& f) {
    const int units = tc.units(K);
    const float per_unit = tc.stage_units ? 1.f : 2.f;  // stages
    for (const TileHeight& h : kTileHeights) {
        const int tm = h.tm, ntiles = ((rows + tm - 1) / tm) * (ntot / kTN);
        const float c = per_unit * (tm == 128 ? tc.c128 : tc.c32), w = per_unit * (tm == 128 ? tc.w128 : tc.w32);
        const int ksmax = std::min({kMaxKSplit, units, h.round * cus / std::max(ntiles, 1)});
        for (int k = 1; k <= std::max(ksmax, 1); ++k) {
            const int per = (units + k - 1) / k;
            if (k > 1 && (units + per - 1) / per != k) continue;  // fewer slices have the same longest one
            const float l = (float)((ntiles * k + kXcds - 1) / kXcds) * (float)kXcds / (float)cus;
            const int full = std::max((int)std::ceil(l) - 1, 0);
            const float load = (float)(full / h.round * h.round) + h.last[full % h.round];
            TilePick p;
            p.tm = tm;
            p.ks = k;
            p.ws_floats = k > 1 ? (size_t)k * rows * ntot : 0;
            p.us = h.start + c * (float)per * load;
            if (k > 1)
                p.us += kSumUs + kPartialUs * 4.f * (float)p.ws_floats + per_unit * (float)units * tc.min_us -
                        w * (float)per * load;
            f(p);
        }
        const int q = ntiles / cus, nleft = ntiles % cus;
        if (!tc.tail || q < 2 || nleft == 0) continue;
        float least = 0.5f;  // of the leftover tile's time, on the busiest CU
        for (int k = 2; k <= std::min(kMaxTailSplit, units); ++k) {
            const float left = (float)((nleft * k + cus - 1) / cus) / (float)k;
            if (k > 2 ? left >= least : left > least) continue;  // no more than fewer slices save
            least = left;
            TilePick p;
            p.tm = tm;
            p.ts.k = k;
            p.ts.nleft = nleft;
            p.ts.nfull = ntiles - nleft;
            p.ts.gridfull = (p.ts.nfull + kXcds - 1) / kXcds * kXcds;
            p.ws_floats = (size_t)nleft * k * kTN * tm;
            p.us = h.start + c * (float)units * ((float)q + left) + kSumTailUs + kPartialUs * 4.f * (float)p.ws_floats;
            f(p);
        }
    }
}

// The launch with the smallest estimate whose partial outputs fit the workspace.
inline TilePick mmq_pick(int rows, int K, int ntot, size_t ws_floats, const TileCost& tc, int cus) {
    TilePick best;
    bool any = false;
    mmq_launches(rows, K, ntot, tc, cus, [&](const TilePick& p) {
        if (p.ws_floats > ws_floats || (any && p.us >= best.us)) return;
        best = p;
        any = true;
    });
    return best;
}

// Workspace floats of the largest launch any tier may take for this shape, so
// that every launch under it is the one it takes under any larger workspace (a
// caller sizes one workspace per shape before it knows which tier a call takes).
inline size_t mmq_ws_floats(int rows, int K, int ntot, int cus) {
    size_t need = 0;
    for (const TileCost& tc : {kCostW144, kCostRaw, kCostQ6})
        mmq_launches(rows, K, ntot, tc, cus, [&](const TilePick& p) { need = std::max(need, p.ws_floats); });
    return need;
}

// ---------------------------------------------------------------------------
// Block -> tile and K slice.
// ---------------------------------------------------------------------------
struct TileMap {
    int mt, nt;  // token tile, weight-row tile (over concatenated parts)
};

// v / d for v, d >= 0 and v + d < 2^21 (SMALL), without the ~40 dependent
// instructions of the integer division: (v + 0.5) / d is at least 0.5 / d from
// the next integer, and the float error is at most (v / d + 1) * 2^-22.
template <bool SMALL>
BQ_HD int tile_div(int v, int d) {
    if (!SMALL) return v / d;
#ifdef __HIP_DEVICE_COMPILE__
    return (int)(((float)v + 0.5f) * __builtin_amdgcn_rcpf((float)d));
#else
    return (int)(((float)v + 0.5f) * (1.f / (float)d));
#endif
}

// Order of the tiles: an XCD's resident workgroups (64 of the 128-token tiles,
// 96 of the 32-token ones) run consecutive indices at about the same K stage,
// so the fewer bytes of weight panels and token tiles those cover, the more of
// every stage its 4 MB L2 serves.  With more token tiles than one such round
// wants, the order walks G panels per token tile instead of all token tiles of
// one panel: G = 8 at 128 tokens (64 indices = 8 panels x 8 token tiles of 18 +
// 16 KB a stage; panel-major 8192 rows: 1 x 64, 1 MB of tokens a stage from
// beyond the L2), G = 4 at 32 tokens (18 and 4 KB: 4 x 24).  Up to kRound token
// tiles the panel-major order is already as compact (512 rows as 32-token tiles,
// 14336 x 2560: 66.4 us, in groups of 8 70.1).  9216 x 3072 W144: 8192 rows
// 635.9 -> 600.6 us, 2048 rows 164.7 -> 161.6 (G = 4 / 16 1-2% behind at 8192
// rows); bytes from beyond the L2s 2262 -> 741 MB and 202 -> 162 MB.
template <int TM, bool SMALL = false>
BQ_HD void tile_at(int idx, int ntm, int ntn, TileMap& t) {
    constexpr int G = TM == 32 ? 4 : 8, kRound = TM == 32 ? 24 : 8;
    if (ntm <= kRound) {
        t.nt = tile_div<SMALL>(idx, ntm);
        t.mt = idx - t.nt * ntm;
        return;
    }
    const int grp = tile_div<SMALL>(idx, G * ntm), first = grp * G;
    const int width = ntn - first < G ? ntn - first : G, r = idx - first * ntm;
    t.mt = tile_div<SMALL>(r, width);
    t.nt = first + r - t.mt * width;
}

// Block b of a launch of ntm x ntn tiles in ks K slices -> (tile, slice kc).
// The n = ntiles * ks pieces, a tile's slices next to each other, are dealt to
// the XCDs in contiguous ranges of ceil(n / 8) (block b runs on XCD b % 8; the
// last range is what is left).  Inside an XCD the blocks go slice by slice, so
// that the first slices, which hold the W144 min term, start first and
// on a CU each (two of them on one CU: 7040 x 5120 at 41 rows 21.9 -> 28.5 us).
// (With the slices on blockIdx.y each XCD took ceil(ntiles / 8) tiles times
// ks: Q6_K 2560 x 7168 at 640 rows, 100 tiles x 5 slices, put 65 workgroups on an
// XCD's 64 slots: 97 us, now 67.  With 7 empty blocks in front of 63 the same
// call took 93.)
// Every workgroup computes this before its first load, so it is closed-form: a
// loop over the slices with an integer division each took 0.4-1 us of every
// split launch (raw 7168 x 2560 at 24 rows 13.4 us, now 12.3; Q6_K 2560 x 4096 at
// 12 rows 11.1, now 10.5).
template <int TM>
BQ_HD bool map_tile(int b, int ntm, int ntn, int ks, TileMap& t, int& kc) {
    const unsigned n = ntm * ntn * ks, x = (unsigned)b % kXcds;
    const int j = (unsigned)b / kXcds;
    const int per = (n + kXcds - 1) / kXcds, p0 = x * per, p1 = p0 + per < (int)n ? p0 + per : (int)n;
    kc = 0;
    if (j >= p1 - p0) return false;
    if (ks == 1) {
        tile_at<TM>(p0 + j, ntm, ntn, t);
        return true;
    }
    // The range starts at slice `lead` of tile t0 and holds q or q + 1 pieces of
    // each slice (q + 1: the r slices from `lead` on, cyclically).  i: the j-th
    // piece in the order of (slice, tile), counted from slice `lead`; it is the
    // m-th piece of slice lead + c.  (A split launch has at most 3 pieces per CU.)
    const int len = p1 - p0, t0 = tile_div<true>(p0, ks), lead = p0 - t0 * ks;
    const int q = tile_div<true>(len, ks), r = len - q * ks;
    const int c0 = lead ? ks - lead : 0;  // slice 0
    int i = j + c0 * q + (c0 < r ? c0 : r);
    if (i >= len) i -= len;
    const bool longer = i < r * (q + 1);
    const int rest = longer ? i : i - r * (q + 1), d = longer ? q + 1 : q;
    const int g = tile_div<true>(rest, d), c = longer ? g : r + g, m = rest - g * d;
    const bool next = lead + c >= ks;  // the piece is in the tile after its slice's first one
    kc = next ? lead + c - ks : lead + c;
    tile_at<TM, true>(t0 + m + (next ? 1 : 0), ntm, ntn, t);
    return true;
}

// Block -> (tile, slice, slices).  Returns false for a block with no work.
// XCD-major over the whole tiles as map_tile; a leftover tile's k slices are
// consecutive blocks.
template <int TM>
BQ_HD bool map_tile_tail(int b, int ntm, int ntn, const TailSplit& ts, TileMap& t, int& kc, int& ks, int& left) {
    left = -1;
    if (ts.k <= 1) return map_tile<TM>(b, ntm, ntn, ks, t, kc);
    if (b < ts.gridfull) {
        const int per = ts.gridfull / kXcds;
        const int idx = (b % kXcds) * per + b / kXcds;
        if (idx >= ts.nfull) return false;
        tile_at<TM>(idx, ntm, ntn, t);
        kc = 0;
        ks = 1;
        return true;
    }
    const int j = b - ts.gridfull;
    if (j >= ts.nleft * ts.k) return false;
    left = j / ts.k;
    kc = j % ts.k;
    ks = ts.k;
    const int idx = ts.nfull + left;
    tile_at<TM>(idx, ntm, ntn, t);
    return true;
}

}  // namespace bq
