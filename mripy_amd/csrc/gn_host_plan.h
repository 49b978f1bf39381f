// Host-side planning of the NUFFT library in plain C++ (no HIP calls), shared by the
// library and by the address/undefined-behaviour-sanitized host test
// (tests/host_asan.cpp): default tile shapes, the radix plan, digit-reversal map and
// twiddles of the pruned FFT passes, and the spread / gather work items and tile
// occupancy masks built from the bin offsets that set_points computes on the device.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

namespace gn {
namespace host {

constexpr int kGatherCellBytesHost = 16; // a staged gather cell: one coil pair, complex64

// {a, b, c, d} with the layout of HIP's int4 (copied to the device as is)
struct Item {
    int x, y, z, w;
};
static_assert(sizeof(Item) == 16, "work items are int4");

// The device scans' grand total: block totals (or sums of them) modulo 2^32 added in 64
// bits, and the same number from the two ints that return it to the host.
constexpr int64_t scan_carry(int64_t carry, int total) { return carry + (int64_t)(uint32_t)total; }
constexpr int64_t scan_total(int lo, int hi) { return (int64_t)((uint64_t)(uint32_t)hi << 32 | (uint32_t)lo); }

// Default spread (output) and gather (home) tile shapes.  Wide windows shrink the
// gather tile, largest axis first, until tile + halo of a coil pair fits 160 KiB.
inline void default_tiles(int dim, int ns, const int64_t *nf, int *tile, int *gtile)
{
    if (dim == 3) {
        tile[0] = 4;
        tile[1] = 4;
        tile[2] = 8;
        gtile[0] = 10;
        gtile[1] = 10;
        gtile[2] = 16;
    } else {
        tile[0] = 8;
        tile[1] = 16;
        tile[2] = 1;
        gtile[0] = 24;
        gtile[1] = 24;
        gtile[2] = 1;
    }
    auto staged = [&]() {
        int64_t r = kGatherCellBytesHost;
        for (int a = 0; a < dim; ++a) r *= std::min<int64_t>(gtile[a] + 2 * ns - 1, nf[a]);
        return r;
    };
    while (staged() > 160 * 1024) {
        int a = 0;
        for (int b = 1; b < dim; ++b)
            if (gtile[b] > gtile[a]) a = b;
        if (gtile[a] == 1) break;
        --gtile[a];
    }
}

// Radix sequence (8, 4, 2, then 3, 5) of a length-L FFT, applied in reverse order of
// extraction; empty when L has another prime factor.
inline std::vector<int> fft_radices(int L)
{
    std::vector<int> r;
    if (L < 1) return r;
    int n = L;
    while (n % 8 == 0 && n > 1) {
        r.push_back(8);
        n /= 8;
    }
    while (n % 4 == 0 && n > 1) {
        r.push_back(4);
        n /= 4;
    }
    while (n % 2 == 0 && n > 1) {
        r.push_back(2);
        n /= 2;
    }
    for (int p : {3, 5})
        while (n % p == 0 && n > 1) {
            r.push_back(p);
            n /= p;
        }
    if (n != 1) return {};
    std::reverse(r.begin(), r.end());
    return r;
}

// The same with primes from 7 up to kFFTPrimeMax, which come first (the first stage
// needs no twiddles); empty when L has a larger prime factor.  Primes up to
// kFFTRadixMax are register butterflies, larger ones the direct-sum stage.
constexpr int kFFTRadixMax = 13;
constexpr int kFFTPrimeMax = 256;
inline std::vector<int> fft_radices_prime(int L)
{
    std::vector<int> big;
    int n = L;
    if (L < 1) return {};
    while (n % 2 == 0) n /= 2;
    for (int p : {3, 5})
        while (n % p == 0) n /= p;
    int smooth = L / n;
    for (int p = 7; p <= kFFTPrimeMax && n > 1; p += 2)
        while (n % p == 0) {
            big.push_back(p);
            n /= p;
        }
    if (n != 1) return {};
    std::reverse(big.begin(), big.end());
    const std::vector<int> r = fft_radices(smooth);
    big.insert(big.end(), r.begin(), r.end());
    return big;
}

// Whether a length has a prime factor above kFFTRadixMax (its lines need a second buffer).
inline bool fft_direct_sums(int L)
{
    for (int p : {2, 3, 5, 7, 11, 13})
        while (L % p == 0) L /= p;
    return L > 1;
}

inline int largest_prime(int64_t L)
{
    int64_t big = 1;
    for (int64_t p = 2; p * p <= L; ++p)
        while (L % p == 0) {
            big = p;
            L /= p;
        }
    return (int)std::max(big, L);
}

// Whether the pruned FFT passes of a plan are to be used on grids whose lengths they cover:
// always for the primes 2, 3, 5.  rocFFT has radices up to 17 as well and takes other lengths
// as Bluestein transforms, which double where 2 L passes a power of two (1024); a column pass
// slows down as its blocks hold fewer columns (LDS: 8, 4, 2 of them up to 780, 1260, 1820
// points, or 525, 890, 1365 with a second buffer).  Type 2, pad + rocFFT / passes, as a
// ratio (type 1 gains more or loses less):
//   primes up to 17, n x n x 8 coils: 770 0.88, 784 1.01, 858 1.07, 952 1.50, 1300 1.81;
//     last axis, 256 x n x 1: 448 0.89, 910 1.08, 1260 1.03, 1750 1.09
//   others, n x n x 8: 844 (211) 0.84, 892 (223) 1.04, 916 (229) 1.16, 1002 (167) 1.14, 1010
//     (101) 0.94, 1038 (173) 0.66, 1834 (131) 0.79, 1912 (239) 1.31; last axis, 256 x 1910 0.70
//   a 3-D grid with few columns beside a long first axis, where rocFFT has more blocks:
//     154 x 32 x 32 1.18, 112 x 32 x 32 x 4 coils 1.13, 220 x 32 x 32 x 8 0.79; 530 x 32 x 32 (53)
//     0.74, 502 x 32 x 32 (251) 0.92 and 1.03 in type 1, 942 x 32 x 32 (157) 0.94 and 1.13
//   3-D with a short first axis, whose column blocks hold few elements, primes up to 17 and
//     many coils: 22 x 52 x 220 x 28 coils 1.23 (type 1 1.30), 22 x 96 x 80 x 23 1.09 (1.22), 12 x
//     220 x 312 x 10 1.02 (1.13), 14 x 196 x 264 x 27 0.98 (1.08); 22 x 44 x 48 x 22 0.78, 24 x 128 x
//     306 x 3 0.89, 26 x 110 x 32 x 24 0.85 (0.90)
//   columns of 891 to 1024 points with two line buffers, large 2-D grids: 984 x 502 x 20 (41)
//     1.29, 950 x 796 x 20 (19) 1.16, 920 x 660 x 24 (23) 1.10; 948 x 728 x 7 (79) 0.98, 1010 x
//     1010 x 8 (101) 0.94
inline bool pruned_passes_pay(int dim, const int64_t *nf, int64_t ncoils)
{
    const int64_t cells = nf[0] * nf[1] * (dim == 3 ? nf[2] : 1) * ncoils;
    int most = 1;
    for (int a = 0; a < dim; ++a) most = std::max(most, largest_prime(nf[a]));
    if (dim == 3 && nf[0] <= 22 && most > 5 && most <= 17 && ncoils >= 10 && cells >= 1500000) return false;
    for (int a = 0; a < dim; ++a) {
        const int64_t L = nf[a];
        const int p = largest_prime(L);
        if (p <= 5) continue;
        const bool rows = a == dim - 1; // contiguous lines
        if (p <= 17 ? L > 780 : !rows && (L > 1860 || (L > 890 && L <= 1024 && p > 128))) return false;
        if (dim == 2 && !rows && L > 890 && L <= 1024 && p > 17 && cells > 9000000) return false;
        if (dim == 3 && a == 0 && nf[1] * nf[2] * ncoils <= 4096 && (p <= 17 || p > 180 || L > 890)) return false;
    }
    return true;
}

// Whether a strided axis of this length (several columns) is left to the Cartesian axis
// passes: not where a block's LDS holds one column, so that a row segment is 8 bytes.
// Microseconds, rocFFT with its shift passes / axis passes, n x n x 2: 1834 (prime 131) 352 /
// 295, 1820 206 / 150, 1875 218 / 233, 2000 228 / 272, 2048 230 / 286, 1912 (prime 239) 361 / 522; rocFFT has radix 17:
// 1088 105 / 79, 1156 121 / 132, 1360 135 / 159, 1530 162 / 210, 1700 184 / 235.
inline bool axis_strided_ok(int L)
{
    int n = L;
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    const bool direct = n > 1;
    while (n % 17 == 0) n /= 17;
    return L <= 1860 && !(direct && n == 1 && L > 1100);
}

// HIP takes launches of fewer than 2^32 threads per grid axis.
constexpr bool launch_fits(int64_t blocks, int threads) { return blocks < (((int64_t)1 << 32) + threads - 1) / threads; }

// Blocks of a Cartesian FFT pass over (slabs, L, ncols): C columns of one slab, or S slabs of
// all C = ncols columns where they are fewer than the lines a block may hold; fewer of either
// while the launch has less than `want` blocks.
struct AxisSplit {
    int C, S;
    int64_t ncb, blocks;
};
inline AxisSplit axis_split(int64_t slabs, int64_t ncols, int lines, int64_t want)
{
    AxisSplit s;
    if (ncols >= lines) {
        s.C = lines;
        s.S = 1;
        while (s.C > 4 && (ncols + s.C - 1) / s.C * slabs < want) s.C /= 2;
    } else {
        s.C = (int)ncols;
        s.S = (int)std::min<int64_t>(lines / s.C, slabs);
        while (s.S > 1 && (slabs + s.S - 1) / s.S < want) s.S = (s.S + 1) / 2;
    }
    s.ncb = (ncols + s.C - 1) / s.C;
    s.blocks = (slabs + s.S - 1) / s.S * s.ncb;
    return s;
}

// Digit-reversal map (pinv[position] = LDS slot) and twiddles e^{-2 pi i k/L}
// (tw[2k], tw[2k+1]) of a length-L transform with radices r.
inline void fft_tables(int L, const std::vector<int> &r, std::vector<int> &pinv, std::vector<float> &tw)
{
    pinv.assign((size_t)L, 0);
    for (int i = 0; i < L; ++i) {
        int rem = i, rev = 0, scale = L;
        for (int rr : r) {
            const int dgt = rem % rr;
            rem /= rr;
            scale /= rr;
            rev += dgt * scale;
        }
        pinv.at((size_t)rev) = i;
    }
    tw.assign(2 * (size_t)L, 0.f);
    const double two_pi = 6.283185307179586476925286766559;
    for (int k = 0; k < L; ++k) {
        const double ang = -two_pi * (double)k / (double)L;
        tw[2 * (size_t)k] = (float)std::cos(ang);
        tw[2 * (size_t)k + 1] = (float)std::sin(ang);
    }
}

struct WorkItems {
    std::vector<Item> spread;  // {tile, pbeg, pend, slot or -1}: tiles with pairs, then empty tiles
    int full = 0;              // spread items of tiles with pairs (the first part)
    std::vector<Item> reduce;  // {tile, slot0, nslots, 0}
    std::vector<Item> gather;  // {gather tile, sbeg, send, 0}
    std::vector<unsigned long long> occ; // per column of spread tiles: leading-axis tile groups with pairs
    int slots = 0;
    int mask_k = 1;
};

// Gather work items {tile, sbeg, send, 0}: each gather tile's samples (bin offsets
// h_home[Kg + 1]) in slices of at most chunk, in tile order.
inline void build_gather_items(int64_t Kg, const int *h_home, int chunk, std::vector<Item> &items)
{
    items.clear();
    for (int64_t k = 0; k < Kg; ++k) {
        const int hb = h_home[k], he = h_home[k + 1];
        for (int s0 = hb; s0 < he; s0 += chunk) items.push_back({(int)k, s0, std::min(he, s0 + chunk), 0});
    }
}

// Work items from the bin offsets: h_pair[K + 1] (pairs of each spread tile) and
// h_home[Kg + 1] (samples of each gather tile).  Every spread tile gets at least one
// item; tiles with more than spread_chunk pairs are split into slices written to
// partial slots and combined by a reduce item.  The items of tiles with pairs come
// first (w.full of them), in tile order, then one item per empty tile, in tile order.
// ntiles: spread tiles per axis (1 for absent axes).
inline void build_work_items(int64_t K, int64_t Kg, const int *ntiles, const int *h_pair, const int *h_home,
                             int spread_chunk, int gather_chunk, WorkItems &w)
{
    w = WorkItems();
    std::vector<Item> empty;
    for (int64_t k = 0; k < K; ++k) {
        const int b = h_pair[k], e = h_pair[k + 1];
        const int n = e - b;
        if (n == 0) {
            empty.push_back({(int)k, b, e, -1});
        } else if (n <= spread_chunk) {
            w.spread.push_back({(int)k, b, e, -1});
        } else {
            const int nch = (n + spread_chunk - 1) / spread_chunk;
            w.reduce.push_back({(int)k, w.slots, nch, 0});
            for (int c = 0; c < nch; ++c)
                w.spread.push_back({(int)k, b + c * spread_chunk, std::min(e, b + (c + 1) * spread_chunk), w.slots + c});
            w.slots += nch;
        }
    }
    w.full = (int)w.spread.size();
    w.spread.insert(w.spread.end(), empty.begin(), empty.end());
    build_gather_items(Kg, h_home, gather_chunk, w.gather);
    // one mask word per column of spread tiles; bit b: leading-axis tiles [b k, (b + 1) k)
    const int64_t ncolt = (int64_t)ntiles[1] * ntiles[2];
    w.mask_k = (ntiles[0] + 63) / 64;
    w.occ.assign((size_t)ncolt, 0ull);
    for (const Item &it : w.spread)
        if (it.z > it.y) {
            const int64_t t0 = it.x / ncolt;
            w.occ.at((size_t)(it.x - t0 * ncolt)) |= 1ull << (t0 / w.mask_k);
        }
}

} // namespace host
} // namespace gn
