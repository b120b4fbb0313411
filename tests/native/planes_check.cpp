// Host-only check of the planes per sample of a launch (tn_worklist.h): those
// of equal jobs exactly, with little weight on a job of few samples, none for
// a launch without samples, and no overflow at large jobs. Prints "ok".
#include <cstdint>
#include <cstdio>
#include <vector>

#include "tn_worklist.h"

struct Job {
    int64_t npts;
    int32_t nbatch;
};

int main() {
    struct {
        std::vector<Job> jobs;
        int planes;
    } cases[] = {
        {{}, 0},
        {{{0, 8}}, 0},
        {{{1000, 1}}, 1},
        {{{1000, 8}, {10, 8}, {0, 1}}, 8},
        {{{1000000, 8}, {1000, 1}}, 8},
        {{{1000000, 16}, {1, 1}, {1000000, 16}}, 16},
        {{{1000000, 1}, {1000, 64}}, 1},
        {{{1000, 2}, {1000, 6}}, 4},
        {{{1000, 2}, {1000, 5}}, 4},
        {{{1000, 8}, {800, 1}}, 5},
        {{{1ll << 40, 1 << 20}, {1ll << 40, 1 << 20}}, 1 << 20},
    };
    for (const auto &c : cases)
        if (const int got = tn::mean_planes(c.jobs); got != c.planes)
            return std::printf("FAIL %zu jobs: %d, not %d\n", c.jobs.size(), got, c.planes), 1;
    std::printf("ok\n");
    return 0;
}
