// Size limits that the library checks on the host (mripy_amd/csrc/gn_host_plan.h), at sizes
// too large to run: the pair total of set_points, launches of the Cartesian FFT passes.  Built and run by
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

// Long strided axes of the Cartesian FFT: the lengths that were measured.
static void check_strided()
{
    for (int L : {2, 16, 17, 34, 1000, 1024, 1088, 1820, 1834, 1850, 1860, 1444 /* 4 19^2 */}) CHECK(axis_strided_ok(L));
    for (int L : {1156, 1224, 1360, 1530, 1700, 1836, 1862, 1875, 1904, 1912, 2000, 2048}) CHECK(!axis_strided_ok(L));
}

// Which grids with primes above 5 use the pruned passes: the measured ones, and every grid
// of the primes 2, 3, 5.
static void check_passes()
{
    auto pay2 = [](int64_t a, int64_t b, int64_t nc) { const int64_t nf[3] = {a, b, 1}; return pruned_passes_pay(2, nf, nc); };
    auto pay3 = [](int64_t a, int64_t b, int64_t c, int64_t nc) { const int64_t nf[3] = {a, b, c}; return pruned_passes_pay(3, nf, nc); };
    for (int L = 2; L <= 2048; ++L) {
        CHECK(largest_prime(L) == 2 || L % largest_prime(L) == 0);
        if (!fft_radices(L).empty()) CHECK(largest_prime(L) <= 5 && pay2(L, L, 8) && pay3(L, 32, 32, 1));
    }
    CHECK(largest_prime(2008) == 251 && largest_prime(289) == 17 && largest_prime(2) == 2 && largest_prime(1) == 1);
    for (int L : {14, 254, 502, 770, 844, 890, 1010, 1038, 1834}) CHECK(pay2(L, L, 8));
    for (int L : {784, 858, 952, 1300, 916, 1002, 1904, 1912, 2002, 2008}) CHECK(!pay2(L, L, 8));
    CHECK(pay2(256, 1910, 1) && !pay2(1910, 256, 1) && pay2(256, 770, 1) && !pay2(256, 910, 1));
    CHECK(pay3(182, 218, 150, 3) && pay3(220, 32, 32, 8) && !pay3(220, 32, 32, 4) && pay3(32, 32, 220, 1));
    CHECK(!pay3(22, 52, 220, 28) && !pay3(14, 24, 306, 16) && !pay3(12, 220, 312, 10) && !pay3(18, 104, 250, 21));
    CHECK(pay3(22, 44, 48, 22) && pay3(26, 110, 32, 24) && pay3(20, 44, 272, 9) && pay3(18, 126, 172, 21) && pay3(18, 100, 250, 21));
    CHECK(!pay2(984, 502, 20) && !pay2(950, 796, 20) && !pay2(920, 660, 24) && pay2(948, 728, 7) && pay2(856, 728, 24) && pay2(1000, 484, 31));
    CHECK(pay3(530, 32, 32, 1) && !pay3(502, 32, 32, 1) && !pay3(942, 32, 32, 1) && pay3(940, 64, 128, 1));
}

// A launch has fewer than 2^32 threads; a split covers every line once.
static void check_launches()
{
    for (int L = 1; L <= 2048; ++L) {
        const std::vector<int> r = fft_radices_prime(L);
        if (!r.empty()) CHECK(fft_direct_sums(L) == (*std::max_element(r.begin(), r.end()) > kFFTRadixMax));
    }
    for (int threads : {64, 256, 512, 1000, 1024}) {
        const int64_t last = (((int64_t)1 << 32) - 1) / threads;
        CHECK(launch_fits(last, threads) && !launch_fits(last + 1, threads));
    }
    for (int lines : {1, 2, 16})
        for (int64_t slabs : {(int64_t)1, (int64_t)3, (int64_t)513, (int64_t)1 << 22, (int64_t)1 << 29})
            for (int64_t ncols : {(int64_t)1, (int64_t)2, (int64_t)15, (int64_t)17, (int64_t)4096, ((int64_t)1 << 27) - 1, (int64_t)1 << 27}) {
                const AxisSplit s = axis_split(slabs, ncols, lines, 512);
                CHECK(s.C >= 1 && s.S >= 1 && (int64_t)s.C * s.S <= lines && (s.S == 1 || s.C == ncols));
                CHECK(s.ncb * s.C >= ncols && (s.ncb - 1) * s.C < ncols && s.blocks % s.ncb == 0);
                CHECK(s.blocks / s.ncb * s.S >= slabs && (s.blocks / s.ncb - 1) * s.S < slabs);
            }
    // 2 points x 2^28 and 16 x 512 x 512 x 512, 16 lines per block: too many blocks for a launch
    CHECK(!launch_fits(axis_split(1, (int64_t)1 << 28, 16, 512).blocks, 512));
    CHECK(!launch_fits(axis_split(1, (int64_t)512 * 512 * 512, 16, 512).blocks, 512));
    CHECK(launch_fits(axis_split(1, ((int64_t)1 << 27) - 16, 16, 512).blocks, 512));
}

int main()
{
    check_pair_total();
    check_launches();
    check_strided();
    check_passes();
    printf("OK\n");
    return 0;
}
