/*
 * Host check of mdz_host_parallel: every element of the range is visited
 * once wherever starting a thread fails (no memory for its state), and an
 * exception of a chunk comes back to the caller after every chunk has ended.
 */
#include <stdio.h>
#include <stdlib.h>

#include <atomic>
#include <new>

#include "../mdoodz6.0_amd/csrc/mdz_host_parallel.h"

static std::atomic<int> left{-1}; /* allocations until they fail (-1: never) */

void *operator new(std::size_t n) {
    if (left.load() >= 0 && left.fetch_sub(1) <= 0) {
        left = 0;
        throw std::bad_alloc();
    }
    if (void *p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, std::size_t) noexcept { free(p); }

int main() {
    const int n = 1000;
    static std::atomic<int> seen[n];
    int bad = 0;
    /* the first allocation is the threads' vector */
    for (int fail = -1; fail <= 9; fail++) {
        for (auto &s : seen) s = 0;
        bool thrown = false;
        left = fail;
        try {
            mdz_host_parallel(n, 10, [&](long long a, long long b) {
                for (long long i = a; i < b; i++) seen[i]++;
            });
        } catch (const std::bad_alloc &) {
            thrown = true;
        }
        left = -1;
        int wrong = 0;
        for (auto &s : seen) wrong += s != (thrown ? 0 : 1);
        if (wrong || thrown != (fail == 0)) bad++;
        printf("allocation %d fails: %s, %d elements wrong\n", fail, thrown ? "thrown" : "done", wrong);
    }
    std::atomic<int> ended{0};
    bool thrown = false;
    try {
        mdz_host_parallel(n, 10, [&](long long a, long long) {
            ended++;
            if (a == 0) throw 7;
        });
    } catch (int) {
        thrown = true;
    }
    if (!thrown || ended < 1) bad++;
    printf("%d failed\n", bad);
    return bad;
}
