// Host-only check of the tile gridding's work construction (tn_worklist.h):
// the pieces of a footprint along one axis cover each of its cells exactly
// once, in the right tile and with the right tap, for every origin, width up
// to 6, tile of 4 and 8 and grid length from the width on (footprints that
// wrap, grids of one ragged tile); bricks list every tile once; and the deal
// over the XCDs keeps every item once, whole workgroups of shared tiles first,
// each XCD's share in list order, within its part of the work. Prints
// "ok <cases>" or the first failure.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "tn_worklist.h"

static int fail(const char *what, long a, long b) {
    std::printf("FAIL %s (%ld, %ld)\n", what, a, b);
    return 1;
}

int main() {
    int cases = 0;
    for (int T : {4, 8})
        for (int W = 1; W <= 6; ++W)
            for (int G = W; G <= 40; ++G)
                for (int base = 0; base < G; ++base, ++cases) {
                    int tile[tn::kMaxPieces], local[tn::kMaxPieces];
                    const int n = tn::axis_pieces(base, W, G, T, tile, local);
                    std::vector<int> seen(W, 0);
                    for (int q = 0; q < n; ++q) {
                        if (local[q] < -(W - 1) || local[q] > T - 1) return fail("origin out of range", base, local[q]);
                        if (tile[q] < 0 || tile[q] >= (G + T - 1) / T) return fail("tile out of range", base, tile[q]);
                        for (int c = 0; c < T; ++c) {
                            const int tap = c - local[q], cell = tile[q] * T + c;
                            if (tap < 0 || tap >= W || cell >= G) continue;  // outside the footprint or the grid
                            if (cell != (base + tap) % G) return fail("cell holds the wrong tap", base, cell);
                            ++seen[tap];
                        }
                    }
                    for (int k = 0; k < W; ++k)
                        if (seen[k] != 1) return fail("tap not covered once", base, k);
                }
    std::mt19937 rng(5);
    for (int cs = 0; cs < 200; ++cs, ++cases) {
        const int ndim = 2 + cs % 2;
        const int32_t nt[3] = {1 + (int32_t)(rng() % 30), 1 + (int32_t)(rng() % 30), ndim == 3 ? 1 + (int32_t)(rng() % 12) : 1};
        const std::vector<int32_t> order = tn::brick_order(nt, ndim);
        std::vector<int> hit((size_t)nt[0] * nt[1] * nt[2], 0);
        for (int32_t t : order) ++hit.at(t);
        for (int h : hit)
            if (h != 1 || order.size() != hit.size()) return fail("brick order", cs, h);

        std::vector<tn::Item> joined, grid;
        const int ngroups = rng() % 20, nrest = cs % 10 == 0 ? 0 : rng() % 3000;
        int id = 0;
        for (int q = 0; q < 4 * ngroups; ++q) joined.push_back(tn::Item{0, id++ | tn::kTilesJoin, 0, 1, 0, 16, 0, -1});
        const bool skew = cs % 3 == 0;
        int64_t total = 0, most = 0;
        for (int q = 0; q < nrest; ++q) {
            const int n = skew && q < nrest / 8 ? 300 : rng() % 20;
            total += n + tn::kTilesBase;
            most = std::max<int64_t>(most, n + tn::kTilesBase);
            grid.push_back(tn::Item{0, id++, 0, 1, 0, n, 0, -1});
        }
        tn::tiles_deal(joined, grid);
        if (nrest && grid.size() % tn::kTilesGroup) return fail("whole workgroups", cs, (long)grid.size());
        std::vector<int> got(id, 0);
        int64_t work[tn::kDealXcds] = {0};
        int last[tn::kDealXcds];
        for (int &l : last) l = -1;
        for (size_t w = 0; w < grid.size(); ++w) {
            const tn::Item &it = grid[w];
            if (it.job < 0) continue;
            const int x = (int)(w / tn::kTilesGroup % tn::kDealXcds), u = it.unit & ~tn::kTilesJoin;
            ++got.at(u);
            if ((it.unit & tn::kTilesJoin) != 0) {
                if (u != (int)w) return fail("shared tiles first", cs, u);
                continue;
            }
            if (u <= last[x]) return fail("an XCD's items out of order", cs, u);
            last[x] = u;
            work[x] += it.e1 - it.e0 + tn::kTilesBase;
        }
        for (int g : got)
            if (g != 1) return fail("item not dealt once", cs, g);
        for (int64_t x : work)
            if (x > total / tn::kDealXcds + 2 * tn::kTilesGroup * most) return fail("unequal work", cs, (long)x);
    }
    std::printf("ok %d\n", cases);
    return 0;
}
