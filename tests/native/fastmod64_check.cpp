// Randomized and edge check of qs_fastmod64 (bucket and mask index of 64-bit
// keys) against the % operator, on the host.
#include "../../qsketch_amd/csrc/qs_internal.h"
#include <cstdio>

static uint64_t y = 0x9E3779B97F4A7C15ull;
static uint64_t rnd()
{
    y ^= y << 13;
    y ^= y >> 7;
    y ^= y << 17;
    return y;
}

static unsigned long long check(uint32_t d, int reps)
{
    const qs_fastdiv64 f = qs_fastdiv64_make(d);
    unsigned long long bad = 0;
    const uint64_t top = ~0ull / d * d; // the largest multiple of d
    const uint64_t edges[] = {0, 1, d - 1ull, d, d + 1ull, 0x7fffffffffffffffull, 1ull << 63, ~0ull - 1, ~0ull,
                              top - 1, top, top + (d > 1), 0xffffffffull * d, 0x100000000ull * (d >> 1) + 1};
    for (uint64_t h : edges)
        bad += qs_fastmod64(h, f) != (uint32_t)(h % d);
    for (int r = 0; r < reps; ++r) {
        uint64_t h = rnd();
        bad += qs_fastmod64(h, f) != (uint32_t)(h % d);
        h = rnd() / d * d; // multiples of d and their left neighbours
        bad += qs_fastmod64(h, f) != 0u;
        bad += qs_fastmod64(h - 1, f) != (uint32_t)((h - 1) % d);
    }
    return bad;
}

int main()
{
    const uint32_t ds[] = {1u,         2u,         3u,          4u,          7u,          256u,        1021u,
                           4096u,      12582893u,  100663291u,  201326557u,  536870909u,  2147483647u, 2147483648u,
                           4294967291u, 4294967295u};
    unsigned long long bad = 0;
    for (uint32_t d : ds)
        bad += check(d, 1000000);
    for (int k = 0; k < 200000; ++k) {
        uint32_t d = (uint32_t)(rnd() >> 32) >> (rnd() & 31);
        bad += check(d ? d : 1u, 16);
    }
    printf("fastmod64 mismatches: %llu\n", bad);
    return bad ? 1 : 0;
}
