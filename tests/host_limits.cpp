// Size limits that the library checks on the host (mripy_amd/csrc/gn_host_plan.h), at sizes
// too large to run: the pair total of set_points.  Built and run by
// tests/test_host_limits.py with the undefined-behaviour sanitizer; prints "OK".
#include <stdio.h>
#include <stdlib.h>

#include "gn_host_plan.h"

using namespace gn::host;

#define CHECK(c)                                                                                                       \
    do {                                                                                                               \
        if (!(c)) {                                                                                                    \
            fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c);                                         \
            exit(1);                                                                                                   \
        }                                                                                                              \
    } while (0)

// The last block of the pair scan: tiles of 2048 samples with `pairs` pairs each, their
// totals added 256 at a time modulo 2^32 and carried by scan_carry.
static int64_t scanned_total(int64_t samples, int64_t pairs)
{
    int64_t carry = 0;
    for (int64_t s = 0; s < samples;) {
        uint32_t all = 0;
        for (int b = 0; b < 256 && s < samples; ++b) {
            const int64_t n = std::min<int64_t>(2048, samples - s);
            all += (uint32_t)(n * pairs);
            s += n;
        }
        carry = scan_carry(carry, (int)all);
    }
    return scan_total((int)(uint32_t)carry, (int)(carry >> 32));
}

static void check_pair_total()
{
    // 4096: nspread 8 with one-cell tiles, the most a window touches; 22: 4 x 4 x 8 tiles, nspread 5
    for (int64_t pairs : {1, 8, 22, 4096})
        for (int64_t samples : {(int64_t)0, (int64_t)1, (int64_t)2049, (int64_t)524287, (int64_t)524288, (int64_t)1048576,
                                (int64_t)1048677, (int64_t)200000000, (int64_t)INT32_MAX})
            CHECK(scanned_total(samples, pairs) == samples * pairs);
}

int main()
{
    check_pair_total();
    printf("OK\n");
    return 0;
}
