// bq_mmq_plan.hpp -- which launch a prefill GEMM takes (token-tile height, K
// split, leftover-tile split) and the workspace that choice can use.  Host
// arithmetic on the shape alone, without HIP: tests/test_mmq_plan.py builds it
// with the host compiler.
#pragma once
#include <stddef.h>

#include <algorithm>
#include <cmath>

namespace bq {

constexpr int kTN = 128;   // weight rows per tile
constexpr int kXcds = 8;

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

}  // namespace bq
