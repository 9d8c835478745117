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
// MI355X's 256 CUs) leaves CUs idle (one
// token tile of a 9216-row matrix: 72 tiles), so it
// is split over K into up to kMaxKSplit slices of whole K units (stage pairs
// for the DMA-staged kernels, stages for the raw tier) when the caller's
// workspace holds the slices' partial outputs [slice][part][rows][N[part]];
// one more launch sums them in a fixed order.  The choice depends only on the
// shape and the workspace size, so equal calls take equal paths (eager or
// captured in a graph) and give equal bits.
constexpr int kMaxKSplit = 8;

// `units`: the launch's slice units (TileCost::units).  `cus` below: the CU
// count of the device the launch runs on (MI355X: 256), which sets the workgroup slots every split and tile-height choice counts.
inline int mmq_ksplit(int rows, int ntot, int units, size_t ws_floats, int tm, int cus) {
    const int ntiles = ((rows + tm - 1) / tm) * (ntot / kTN);
    if (ntiles <= 0) return 1;
    const int slots = (tm == 32 ? 3 : 2) * cus;  // workgroups resident at once (3 or 2 per CU)
    int ks = std::min(kMaxKSplit, std::max(1, slots / ntiles));
    while (ks > 1 && ((size_t)ks * rows * ntot > ws_floats || units < ks)) --ks;
    // the fewest slices with the same longest slice (fewer partial outputs)
    const int per = (units + ks - 1) / ks;
    return (units + per - 1) / per;
}

// The leftover-tile split for `ntiles` tiles of `tm` tokens whose K has
// `units` slice units: the k (2..4) that minimises the busiest CU's work,
// floor(ntiles / CUs) + ceil(nleft * k / CUs) / k tiles, if that beats the
// unsplit ceil(ntiles / CUs) by at least half a tile and the slices fit the
// workspace; else k = 1.  Measured (9216 x 3072 W144, eager launches, µs,
// unsplit -> split): 2048 rows (k = 2, 0.5 tile) 181.5 -> 168.5; smaller
// gains did not pay for the shorter slices and the summing launch (2560 rows,
// k = 3 for 0.33 tile: 216 -> 218), nor did more than 4 slices (2304 rows,
// k = 8: 220 -> 227).
// It must also save at least kTailMinSaving tile-token-units (tm x K units x
// e, e = the tile height's relative cost per output) on the busiest CU, about
// half of what the summing launch and the partial tiles cost.
constexpr int kMaxTailSplit = 4;
constexpr float kTailMinSaving = 192.f;
inline TailSplit mmq_tail_split(int ntiles, int units, size_t ws_floats, int tm, float e, int cus) {
    TailSplit ts;
    const int q = ntiles / cus, nleft = ntiles % cus;
    // with one whole tile per CU each runs alone on its CU and the leftover
    // slices lose (512 x 9216 W144, 128-token tiles: 62 -> 67 us)
    if (q < 2 || nleft == 0) return ts;
    float best = (float)(q + 1);
    int bk = 1;
    for (int k = 2; k <= std::min(kMaxTailSplit, units); ++k) {
        if ((size_t)nleft * k * kTN * tm > ws_floats) break;
        const float load = (float)q + (float)((nleft * k + cus - 1) / cus) / (float)k;
        if (load < best - 1e-6f) {
            best = load;
            bk = k;
        }
    }
    if (bk == 1 || best > (float)(q + 1) - 0.5f) return ts;
    if (((float)(q + 1) - best) * (float)tm * (float)units * e < kTailMinSaving) return ts;
    ts.k = bk;
    ts.nleft = nleft;
    ts.nfull = ntiles - nleft;
    ts.gridfull = (ts.nfull + kXcds - 1) / kXcds * kXcds;
    return ts;
}

// Token-tile height (128 or 32) and K split of a launch: the pair with the
// smallest estimated time
//   start[tm] + stages per slice x c[tm] x load + 2.5 us if a sum launch follows,
// c = us per 128-value stage and workgroup per CU of a full GPU.  load: the
// workgroups of the busiest CU (per XCD, as they are dealt), with two corrections.
// A CU that holds a single 128-token tile takes `lone` (1.05: one wave per SIMD
// keeps it nearly as busy as two; 1.22 for the raw tier, whose two barriers and
// unpacking per stage a second workgroup covers), one that holds two no less
// than `pair` = 1.7 (W144, unsplit) to 1.9 loads' time; the 32-token tile 1.3
// and 1.9.  With the
// leftover-tile split the load is the split one.  Fitted to both heights at
// every split, 9 shapes x 11 row counts (9216 / 14336 / 8704 x 2560 / 3072 and
// 2560 x 4096 W144, raw 3072 x 4096, Q6_K 3072 x 9216 and 2560 x 7168; 16..2048
// rows).  Against the estimate this replaces (tile height weighted by 1.06 ..
// 1.33, always the largest split): 14336 x 2560 at 512 rows 68.1 -> 59.7 us
// (128 tokens instead of 32), 9216 x 3072 at 768 rows 78.8 -> 69.2, 8704 x 2560 at 768 /
// 128 rows 66.3 -> 57.8 / 27.6 -> 24.5, 2560 x 4096 at 1536 rows 66.6 -> 58.1,
// raw 3072 x 4096 at 300 rows 37.1 -> 32.9.
struct TileCost {
    float c128, c32, lone, pair;
    bool stage_units;  // slices at 128-value stages (else at stage pairs)
    bool tail;         // the kernel takes the leftover-tile split
    float e32;         // its 32-token tile's cost per output over the 128-token one's
    constexpr int units(int K) const { return stage_units ? K >> 7 : K >> 8; }
};
constexpr TileCost kCostW144 = {1.40f, 0.385f, 1.05f, 1.70f, false, true, 1.03f};
constexpr TileCost kCostRaw = {1.74f, 0.61f, 1.22f, 1.78f, true, true, 1.38f};
constexpr TileCost kCostQ6 = {2.4f, 0.64f, 1.05f, 1.9f, false, false, 1.f};
constexpr float kSplitUs = 2.5f, kStartUs128 = 11.5f, kStartUs32 = 9.f;

struct TilePick {
    int tm, ks;
    TailSplit ts;
};

inline TilePick mmq_pick(int rows, int K, int ntot, size_t ws_floats, const TileCost& tc, int cus) {
    TilePick best = {128, 1, {}};
    float best_us = -1.f;
    const int units = tc.units(K);
    for (const int tm : {128, 32}) {
        const int ntiles = ((rows + tm - 1) / tm) * (ntot / kTN);
        const int ksmax = mmq_ksplit(rows, ntot, units, ws_floats, tm, cus);
        const float lone = tm == 128 ? tc.lone : 1.3f;
        for (int k = 1; k <= ksmax; ++k) {
            const int per = (units + k - 1) / k;
            if ((units + per - 1) / per != k) continue;  // fewer slices have the same longest one
            const float l = (float)((ntiles * k + kXcds - 1) / kXcds) * (float)kXcds / (float)cus;
            const float pair = tm == 128 && k == 1 ? tc.pair : 1.9f;
            float load;
            if (l <= 1.f)
                load = lone;
            else if (l <= 2.f)
                load = std::max(l, pair);
            else if (tm == 32)  // up to three at once, then one after another as slots free up
                load = l <= 3.f ? 2.45f + 0.35f * (l - 2.f) : l + 0.3f;
            else  // two at once: nearly whole rounds
                load = std::min(std::ceil(l) + 0.05f, l + 0.6f);
            TailSplit ts;
            if (tc.tail && k == 1) ts = mmq_tail_split(ntiles, units, ws_floats, tm, tm == 32 ? tc.e32 : 1.f, cus);
            if (ts.k > 1) load = (float)(ntiles / cus) + (float)((ts.nleft * ts.k + cus - 1) / cus) / (float)ts.k;
            const float stage = (float)(tc.stage_units ? per : 2 * per) * (tm == 128 ? tc.c128 : tc.c32);
            const float extra = k > 1 ? kSplitUs : 0.f;
            const float us = (tm == 128 ? kStartUs128 : kStartUs32) + stage * load + extra;
            if (best_us < 0.f || us < best_us) {
                best_us = us;
                best = {tm, k, ts};
            }
        }
    }
    return best;
}

// Workspace floats the leftover-tile split of either Q5_K tier takes for this
// shape (the larger of the two tile heights), from the constants the launches
// use, so that a launch under the reserved workspace is the one it takes under
// any larger one.
inline size_t mmq_tail_ws_floats(int rows, int K, int ntot, int cus) {
    size_t need = 0;
    for (const int tm : {128, 32}) {
        const int ntiles = ((rows + tm - 1) / tm) * (ntot / kTN);
        for (const TileCost& tc : {kCostW144, kCostRaw}) {
            const TailSplit ts = mmq_tail_split(ntiles, tc.units(K), (size_t)-1, tm, tm == 32 ? tc.e32 : 1.f, cus);
            if (ts.k > 1) need = std::max(need, (size_t)ts.nleft * ts.k * kTN * tm);
        }
    }
    return need;
}

// Workspace floats that allow the largest split any tier or tile height takes
// for this shape: a caller sizes one workspace per shape before it knows which
// tier a call takes (the raw tier, which splits at 128-value stages, can take
// more slices than the W144 and Q6_K kernels, which split at 256).
inline size_t mmq_ws_floats(int rows, int K, int ntot, int cus) {
    const int ks = std::max(mmq_ksplit(rows, ntot, kCostRaw.units(K), (size_t)-1, 128, cus),
                            mmq_ksplit(rows, ntot, kCostRaw.units(K), (size_t)-1, 32, cus));
    const size_t split = ks > 1 ? (size_t)ks * rows * ntot : 0;
    return std::max(split, mmq_tail_ws_floats(rows, K, ntot, cus));
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
// 642 -> 606 us, 2048 rows 166.6 -> 162.2 (G = 4 / 16 1-2% behind at 8192 rows).
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
