// The prefill GEMMs' launch choice (bq_mmq_plan.hpp) for tests/test_mmq_plan.py,
// built with the host compiler.  tier: 0 W144, 1 raw Q5_K, 2 Q6_K.
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
}
