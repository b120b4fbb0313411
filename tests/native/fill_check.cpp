// Host-only check of the tile gridding's runs of empty tiles (tn_worklist.h):
// every tile without entries lies in exactly one run, tiles with entries in
// none, a run stays in its row and is at most as long as asked, and only the
// length limit or a tile with entries ends one. Prints "ok <cases>" or the
// first failure.
#include <cstdio>
#include <random>
#include <vector>

#include "tn_worklist.h"

int main() {
    std::mt19937 rng(3);
    int cases = 0;
    for (; cases < 400; ++cases) {
        const int32_t nt[3] = {1 + (int32_t)(rng() % 70), 1 + (int32_t)(rng() % 9), 1 + (int32_t)(rng() % 5)};
        const int longest = cases % 2 ? 8 : 16, n = nt[0] * nt[1] * nt[2];
        const unsigned full = rng() % 5;  // 0: every tile empty, 4: none
        std::vector<int32_t> off(n + 1, 100);
        for (int t = 0; t < n; ++t) off[t + 1] = off[t] + (rng() % 4 < full ? 1 + (int32_t)(rng() % 9) : 0);
        const std::vector<int32_t> run = tn::empty_runs(off.data(), nt, longest);
        std::vector<int> covered(n, 0);
        for (int t = 0; t < n; ++t) {
            if (run[t] < 0 || run[t] > longest || t % nt[0] + run[t] > nt[0]) return std::printf("FAIL length\n"), 1;
            for (int k = 0; k < run[t]; ++k) ++covered[t + k];
            const int next = t + run[t];
            if (run[t] > 0 && run[t] < longest && next % nt[0] != 0 && off[next] == off[next + 1])
                return std::printf("FAIL run ends early\n"), 1;
        }
        for (int t = 0; t < n; ++t)
            if (covered[t] != (off[t] == off[t + 1])) return std::printf("FAIL tile %d covered %d times\n", t, covered[t]), 1;
    }
    std::printf("ok %d\n", cases);
    return 0;
}
