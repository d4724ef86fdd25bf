// Walks the records of one thread of the dense build's scatter
// (pyrit_amd/csrc/dense_walk.h) for tests/test_dense_walk.py:
//   <count> <threads of the grid> <records per round> <thread>
// prints the rounds, the records taken, the first and the last of them and
// whether each lay one grid below the one before; gives up, with status 1,
// after more rounds than the records need.
#include <stdio.h>
#include <stdlib.h>

#define __host__
#define __device__
#include "dense_walk.h"

int main(int argc, char** argv) {
    if (argc != 5) return 2;
    const uint32_t n = (uint32_t)strtoull(argv[1], nullptr, 10), threads = (uint32_t)strtoull(argv[2], nullptr, 10);
    const uint32_t unroll = (uint32_t)strtoull(argv[3], nullptr, 10), thread = (uint32_t)strtoull(argv[4], nullptr, 10);
    const uint64_t most = (uint64_t)n / ((uint64_t)threads * unroll) + 2;
    uint64_t rounds = 0, taken = 0;
    uint32_t first = 0, last = 0;
    bool regular = true;
    for (pyr::DenseWalk w(thread, threads, n); w.more(); w.next(unroll)) {
        if (++rounds > most) return 1;
        for (uint32_t u = 0; u < unroll; u++) {
            if (!w.has(u)) continue;
            const uint32_t i = w.record(u);
            if (taken == 0) first = i;
            else regular = regular && last - i == threads && last > i;
            last = i;
            taken++;
        }
    }
    printf("%llu %llu %u %u %d\n", (unsigned long long)rounds, (unsigned long long)taken, first, last, regular ? 1 : 0);
    return 0;
}
