// Host-only check of the chirp transforms' convolution lengths
// (tn_worklist.h): the shortest length that holds N + L - 1, none beyond the
// longest one, also where that sum passes 32 bits. Prints "ok".
#include <climits>
#include <cstdio>
#include <initializer_list>

#include "tn_worklist.h"

int main() {
    for (int L = 1; L <= 1600; ++L)
        for (int N = 1; N <= L; N += 1 + L / 50) {
            const int M = tn::chirp_length(N, L), need = N + L - 1;
            if ((L < 2 || need > 1536) != (M == 0) || (M != 0 && M < need)) return std::printf("FAIL %d %d: %d\n", N, L, M), 1;
            for (int shorter : tn::kChirpLengths)
                if (M != 0 && shorter < M && shorter >= need) return std::printf("FAIL %d %d: %d\n", N, L, M), 1;
        }
    for (int L : {1 << 20, 1 << 30, (1 << 30) + 1, INT_MAX - 1, INT_MAX})
        for (int N : {L, L / 2, L - 7})
            if (tn::chirp_length(N, L) != 0) return std::printf("FAIL %d %d\n", N, L), 1;
    std::printf("ok\n");
    return 0;
}
