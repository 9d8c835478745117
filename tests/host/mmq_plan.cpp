// The prefill GEMMs' launch choice and deal (bq_mmq_plan.hpp) for tests/test_mmq_plan.py,
// built with the host compiler.  tier: 0 W144, 1 raw Q5_K, 2 Q6_K.
#include <vector>

#include "bq_mmq_plan.hpp"

using namespace bq;

static TilePick pick(int tier, int rows, int K, int ntot, size_t ws, int cus) {
    const TileCost& tc = tier == 0 ? kCostW144 : tier == 1 ? kCostRaw : kCostQ6;
    return mmq_pick(rows, K, ntot, ws, tc, cus);
}

extern "C" {

// out: token-tile height, K slices, slices per leftover tile, leftover tiles
void t_pick(int tier, int rows, int K, int ntot, size_t ws_floats, int cus, int* out) {
    const TilePick p = pick(tier, rows, K, ntot, ws_floats, cus);
    out[0] = p.tm;
    out[1] = p.ks;
    out[2] = p.ts.k;
    out[3] = p.ts.nleft;
}

size_t t_ws_floats(int rows, int K, int ntot, int cus) { return mmq_ws_floats(rows, K, ntot, cus); }

// Over K, N and rows in steps: the shapes whose launch under the reserved
// workspace is not the one an unlimited workspace gives (count; the first one's
// tier, rows, K and N in first[4]).
long t_reserved_differs(int tier, int cus, int k_step, int n_step, int max_rows, int* first) {
    long bad = 0;
    for (int K = k_step; K <= 9216; K += k_step)
        for (int N = n_step; N <= 18432; N += n_step)
            for (int rows = 9; rows <= max_rows; rows += rows < 128 ? 7 : rows < 1024 ? 61 : 97) {
                const TilePick a = pick(tier, rows, K, N, mmq_ws_floats(rows, K, N, cus), cus);
                const TilePick b = pick(tier, rows, K, N, (size_t)-1, cus);
                if (a.tm == b.tm && a.ks == b.ks && a.ts.k == b.ts.k && a.ts.nleft == b.ts.nleft) continue;
                if (bad++ == 0) first[0] = tier, first[1] = rows, first[2] = K, first[3] = N;
            }
    return bad;
}

// The blocks of a launch of ntm x ntn tiles in ks K slices (tail_k <= 1) or
// with its last `left` tiles in tail_k slices: 0 if every piece is computed
// exactly once, by a tile of its own, and no XCD (blocks b, b + 8, ...) starts a
// slice before an earlier one or has an empty block before a piece (not looked at
// with a leftover split); else the number of the check that failed.
int t_deal(int tm, int ntm, int ntn, int ks, int tail_k, int left) {
    const int ntiles = ntm * ntn;
    TailSplit ts;
    if (tail_k > 1) {
        ts.k = tail_k;
        ts.nleft = left;
        ts.nfull = ntiles - left;
        ts.gridfull = (ts.nfull + kXcds - 1) / kXcds * kXcds;
    }
    const int grid = tail_k > 1 ? ts.gridfull + ts.nleft * ts.k : (ntiles * ks + kXcds - 1) / kXcds * kXcds;
    std::vector<int> seen((size_t)ntiles * 8, 0), last(kXcds, 0), empty(kXcds, 0);
    for (int b = 0; b < grid; ++b) {
        TileMap t;
        int kc, k = ks, lf;
        const bool ok = tm == 32 ? map_tile_tail<32>(b, ntm, ntn, ts, t, kc, k, lf)
                                 : map_tile_tail<128>(b, ntm, ntn, ts, t, kc, k, lf);
        const int x = b % kXcds;
        if (!ok) {
            empty[x]++;
            continue;
        }
        if (t.mt < 0 || t.mt >= ntm || t.nt < 0 || t.nt >= ntn || kc < 0 || kc >= k || k > 8) return 1;
        if (k != (lf >= 0 ? tail_k : tail_k > 1 ? 1 : ks)) return 2;
        if (seen[((size_t)t.nt * ntm + t.mt) * 8 + kc]++) return 3;
        if (tail_k > 1) continue;
        if (empty[x]) return 4;
        if (kc < last[x]) return 5;
        last[x] = kc;
    }
    long pieces = 0;
    for (int v : seen) pieces += v;
    if (pieces != (tail_k > 1 ? (long)ts.nfull + (long)ts.nleft * ts.k : (long)ntiles * ks)) return 6;
    if (tail_k > 1) {  // a leftover tile has all its slices, a whole one just its own
        for (int t = 0; t < ntiles; ++t) {
            int c = 0;
            while (c < 8 && seen[(size_t)t * 8 + c]) ++c;
            for (int d = c; d < 8; ++d)
                if (seen[(size_t)t * 8 + d]) return 7;
            if (c != 1 && c != tail_k) return 8;
        }
        return 0;
    }
    return 0;
}

// first[2]: the first v, d with another quotient than v / d (-1: none) over v < max_v, d < max_d
void t_div(int max_v, int max_d, int* first) {
    first[0] = -1;
    for (int v = 0; v < max_v; ++v)
        for (int d = 1; d < max_d; ++d)
            if (tile_div<true>(v, d) != v / d) {
                first[0] = v;
                first[1] = d;
                return;
            }
}
}
