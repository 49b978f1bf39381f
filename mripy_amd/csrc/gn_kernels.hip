// HIP kernels of the Gaussian-gridding NUFFT for CDNA4 (gfx950).
//
// Data layout in HBM (per plan):
//   grid    : nc oversampled grids, coil-major, C order (nf0, nf1[, nf2]), complex64
//   records : samples sorted by home tile (the tile holding the window start cell)
//             cell = {s0,s1,s2,orig}, frac = {t0,t1,t2,dcf}; bin_start[K+1]
//   pairs   : (output tile, sample) pairs grouped by tile, samples in sorted order
//   items   : spread/gather work items (a tile and a bounded slice of its list)
//   image / samples at the boundary: coil-last (reference) or coil-major.
//
// Window convention (fft/nufft_func.py:293-295, 536-546): xi = x mod 2pi,
// m = 1 + xi // h, taps g = m - ns + j (j = 0..2ns-1) wrapped mod nf, weight
// exp(-(xi - h g)^2/(4 tau)) = exp2(-coef (t + ns - j)^2) with t = xi/h - m.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <type_traits>
#include <vector>

#include <map>
#include <mutex>

#include "gn_internal.h"
#include "gn_host_plan.h"

namespace gn {

namespace {

constexpr double kTwoPi = 6.283185307179586; // 2*np.pi in float64
constexpr int kXCDs = 8;                      // MI355X: 8 XCDs, each with its own L2

// Workgroups are dispatched to the XCDs round-robin by linear block id.  Give each
// XCD runs of kXCDRun consecutive work items (neighbouring tiles: shared halo cells
// and sample values stay in one L2) while the runs still rotate over the XCDs, so a
// dense region of the trajectory is shared out evenly.  Blocks past the last whole
// round of runs keep their order; the map is a bijection on [0, n).
#ifndef GN_XCD_RUN
#define GN_XCD_RUN 32
#endif
constexpr int64_t kXCDRun = GN_XCD_RUN;
constexpr int kStageUnroll = 8; // global loads in flight per thread while staging

__device__ inline uint32_t xcd_swizzle(uint32_t lin, uint32_t n)
{
    // 32-bit: every launch of these kernels has fewer than 2^31 blocks (checked on the host)
    constexpr uint32_t run = (uint32_t)kXCDRun, round = (uint32_t)kXCDs * run;
    if (lin >= (n / round) * round) return lin;
    const uint32_t x = lin % kXCDs, k = lin / kXCDs;
    return ((k / run) * kXCDs + x) * run + k % run;
}

// ---------------------------------------------------------------------------
// set_points: window start cell, offset and home tile of every sample (FP64)
// ---------------------------------------------------------------------------

// CPython float divmod (fmod based), the semantics of numba's x % y and x // y.
__device__ inline double py_divmod(double vx, double wx, double *modp)
{
    double mod = fmod(vx, wx);
    double div = (vx - mod) / wx;
    if (mod != 0.0) {
        if ((wx < 0) != (mod < 0)) {
            mod += wx;
            div -= 1.0;
        }
    } else {
        mod = copysign(0.0, wx);
    }
    double fl;
    if (div != 0.0) {
        fl = floor(div);
        if (div - fl > 0.5) fl += 1.0;
    } else {
        fl = copysign(0.0, vx / wx);
    }
    *modp = mod;
    return fl;
}

struct PrepArgs {
    int64_t M;
    const void *x[3];
    int coord_f64;
    double df;
    int dim;
    int64_t nf[3];
    int ns;
    int tile[3];
    int ntiles[3];
    int4 *cell;
    float4 *frac;
    int *err; // set to seq, this call's number, on a non-finite coordinate
    int seq;
};

__global__ __launch_bounds__(256) void k_prep(PrepArgs a)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.M) return;
    int s[3] = {0, 0, 0};
    float t[3] = {0.f, 0.f, 0.f};
    int key = 0;
    for (int ax = 0; ax < a.dim; ++ax) {
        double x = a.coord_f64 ? ((const double *)a.x[ax])[i] : (double)((const float *)a.x[ax])[i];
        x = x * a.df;
        if (!isfinite(x)) {
            *a.err = a.seq; // every such thread stores the same value
            x = 0.0;
        }
        double xi, dummy;
        py_divmod(x, kTwoPi, &xi);                         // xi = x % (2 pi)
        const double h = kTwoPi / (double)a.nf[ax];
        int64_t m = 1 + (int64_t)py_divmod(xi, h, &dummy); // m = 1 + int(xi // h)
        double delta = xi - h * (double)m;
        t[ax] = (float)(delta / h);
        int64_t st = (m - a.ns) % a.nf[ax];
        if (st < 0) st += a.nf[ax];
        s[ax] = (int)st;
        key = key * a.ntiles[ax] + s[ax] / a.tile[ax];
    }
    a.cell[i] = make_int4(s[0], s[1], s[2], key);
    a.frac[i] = make_float4(t[0], t[1], t[2], 0.f);
}

// ---------------------------------------------------------------------------
// Device exclusive scans in one launch: every block scans its tile in place and publishes
// its total; the block that takes the last ticket scans the totals (bsum[nb] = the grand
// total) and may return values to the host through mapped pinned memory.  Consumers add
// the block's offset themselves: offset of i = data[i] + bsum[i / kScanTile].  No block
// waits for another.  A scan was three launches (local, totals, add) and each returned
// value a copy: 13056 samples in 2-D took 41 launches and 8 copies, 294 us; now 17 launches,
// 140 us (1,048,576 samples in 3-D at nspread 3: 950 -> 641 us).
// ---------------------------------------------------------------------------

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;
constexpr int kItemTile = kScanThreads * 4; // tiles per block of the work-item scan

// Exclusive scan of N ints per thread over the 256 threads of the block (all threads call
// it); total is the block's, modulo 2^32.
template <int N>
__device__ inline void block_exclusive_scan(int (&x)[N], int (&total)[N])
{
    __shared__ int s_wave[N][kScanThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc[N];
#pragma unroll
    for (int c = 0; c < N; ++c) {
        int v = x[c];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(v, o, 64);
            if (lane >= o) v += u;
        }
        inc[c] = v;
        if (lane == 63) s_wave[c][wave] = v;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < N; ++c) {
        uint32_t before = 0, all = 0;
        for (int w = 0; w < kScanThreads / 64; ++w) {
            const uint32_t t = (uint32_t)s_wave[c][w];
            before += w < wave ? t : 0;
            all += t;
        }
        x[c] = (int)((uint32_t)(inc[c] - x[c]) + before);
        total[c] = (int)all;
    }
    __syncthreads(); // s_wave may be written again
}

// Publish this block's totals and, in the block that finishes last, turn all of them into
// exclusive offsets; bsum holds (gridDim.x + 1) * N ints.  True in the last block, with the
// grand totals in grand (thread 0).  The ticket is left at zero for the next scan.
// The grand totals are 64-bit, so that a caller can refuse one that does not fit an int
// (the offsets past it are modulo 2^32): a sample has at most 16^3 (tile, sample) pairs, so
// a tile of the scan totals at most 2^23 and 256 of them at most 2^31, which scan_carry adds
// as an unsigned number.
template <int N>
__device__ inline bool scan_block_totals(int *bsum, int *ticket, const int (&total)[N], int64_t (&grand)[N])
{
    __shared__ int s_last;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < N; ++c)
            __hip_atomic_store(bsum + (int64_t)blockIdx.x * N + c, total[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        s_last = t == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!s_last) return false;
    int64_t carry[N] = {};
    const int64_t nb = gridDim.x;
    for (int64_t b0 = 0; b0 < nb; b0 += kScanThreads) {
        const int64_t i = b0 + threadIdx.x;
        int x[N], all[N];
#pragma unroll
        for (int c = 0; c < N; ++c)
            x[c] = i < nb ? __hip_atomic_load(bsum + i * N + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
        block_exclusive_scan<N>(x, all);
#pragma unroll
        for (int c = 0; c < N; ++c) {
            if (i < nb) bsum[i * N + c] = (int)((uint32_t)x[c] + (uint32_t)carry[c]);
            carry[c] = host::scan_carry(carry[c], all[c]);
        }
    }
    if (threadIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < N; ++c) {
            bsum[nb * N + c] = (int)carry[c];
            grand[c] = carry[c];
        }
        *ticket = 0;
    }
    return true;
}

// data[i] = exclusive scan within the tile of load(i), i < n.  ret (null: none): ret[0],
// ret[1] = the grand total's low and high half, ret[2] = *err.
template <typename F>
__device__ inline void scan_tile(F load, int *__restrict__ data, int64_t n, int *bsum, int *ticket, int *ret, int *err)
{
    // values pass through LDS, so that a wave reads and writes consecutive entries while
    // each thread sums kScanItems consecutive ones
    __shared__ int4 s_v[kScanTile / 4];
    int *sv = (int *)s_v;
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = k * kScanThreads + threadIdx.x;
        sv[i] = base + i < n ? load(base + i) : 0;
    }
    __syncthreads();
    int v[kScanItems];
    int sum[1] = {0}, total[1];
#pragma unroll
    for (int k = 0; k < kScanItems; k += 4) {
        const int4 t = s_v[(threadIdx.x * kScanItems + k) / 4];
        v[k] = t.x;
        v[k + 1] = t.y;
        v[k + 2] = t.z;
        v[k + 3] = t.w;
        sum[0] += t.x + t.y + t.z + t.w;
    }
    block_exclusive_scan<1>(sum, total);
    int run = sum[0];
#pragma unroll
    for (int k = 0; k < kScanItems; k += 4) {
        const int4 t = make_int4(run, run + v[k], run + v[k] + v[k + 1], run + v[k] + v[k + 1] + v[k + 2]);
        run = t.w + v[k + 3];
        s_v[(threadIdx.x * kScanItems + k) / 4] = t;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = k * kScanThreads + threadIdx.x;
        if (base + i < n) data[base + i] = sv[i];
    }
    int64_t grand[1];
    if (scan_block_totals<1>(bsum, ticket, total, grand) && ret && threadIdx.x == 0) {
        ret[0] = (int)(uint32_t)grand[0];
        ret[1] = (int)(grand[0] >> 32);
        ret[2] = *err;
    }
}

__global__ __launch_bounds__(kScanThreads) void k_scan(int *__restrict__ data, int64_t n, int *bsum, int *ticket)
{
    scan_tile([&](int64_t i) { return data[i]; }, data, n, bsum, ticket, nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// Digit passes of the stable counting sort.  A key in [0, K) is sorted by
// ceil(log2 K / kRadixBits) stable counting sorts on successive digits, least significant
// first.  Each workgroup owns one chunk of consecutive items, each of its waves a quarter:
//   k_radix_count   : per-chunk digit histogram (LDS), written digit-major
//                     cnt[digit * C + chunk]
//   exclusive scan  : cnt -> global start of every (digit, chunk) run; digit-major
//                     order keeps chunks, hence items, in index order
//   k_radix_scatter : the waves count their quarters again (the chunk is in cache) and take
//                     their starts within the chunk's runs in wave order; then a wave walks
//                     its quarter 64 items at a time: the lanes holding the same digit find
//                     each other with one ballot per digit bit (match mask), rank themselves
//                     by lane, and the lowest lane of each group advances that digit's
//                     running offset in LDS.
// Every pass is stable, so the result is the stable order by key.  A count per workgroup
// instead of per wave makes the count array, whose digit-major writes and reads touch a
// cache line each, a quarter as long: set_points of 1048576 samples on a 256^3 grid
// 645 -> 546 us (nspread 3) and 1390 -> 1143 us (5), of 13056 on 384^2 142 -> 120 us.
// ---------------------------------------------------------------------------

// Digits are of equal width, at most kRadixBits: fewer bins mean shorter count arrays to
// scan (17-bit keys as 9 + 8 instead of 10 + 7 bits).
constexpr int kRadixBits = 11;
constexpr int kRadixWaves = 4;
constexpr int kRadixUnroll = 4; // steps of 64 items whose loads are in flight together

__global__ __launch_bounds__(64 * kRadixWaves) void k_radix_count(int64_t n, const int *__restrict__ keys, int stride,
                                                                  int shift, int bins, int64_t chunk_len, int C,
                                                                  int *__restrict__ cnt)
{
    extern __shared__ int lds_radix[]; // [bins]
    for (int d = threadIdx.x; d < bins; d += blockDim.x) lds_radix[d] = 0;
    __syncthreads();
    const int64_t beg = (int64_t)blockIdx.x * chunk_len;
    const int64_t end = min(n, beg + chunk_len);
    for (int64_t i0 = beg + threadIdx.x; i0 < end; i0 += kRadixUnroll * blockDim.x) {
        int key[kRadixUnroll];
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u) {
            const int64_t i = i0 + u * blockDim.x;
            key[u] = i < end ? keys[i * stride] : 0;
        }
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u)
            if (i0 + u * blockDim.x < end) atomicAdd(&lds_radix[(key[u] >> shift) & (bins - 1)], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < bins; d += blockDim.x) cnt[(int64_t)d * C + blockIdx.x] = lds_radix[d];
}

// vals_in == nullptr: the values are the item indices
__global__ __launch_bounds__(64 * kRadixWaves) void k_radix_scatter(int64_t n, const int *__restrict__ keys_in,
                                                                    int stride, const int *__restrict__ vals_in,
                                                                    int shift, int bits, int64_t chunk_len, int C,
                                                                    const int *__restrict__ offs,
                                                                    const int *__restrict__ bsum,
                                                                    int *__restrict__ keys_out,
                                                                    int *__restrict__ vals_out)
{
    extern __shared__ int lds_radix[]; // [kRadixWaves][bins]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int bins = 1 << bits;
    int *base = lds_radix + wave * bins;
    for (int d = threadIdx.x; d < kRadixWaves * bins; d += blockDim.x) lds_radix[d] = 0;
    __syncthreads();
    const int64_t part = chunk_len / kRadixWaves;
    const int64_t beg = (int64_t)blockIdx.x * chunk_len + wave * part;
    const int64_t end = min(n, beg + part);
    for (int64_t g = beg; g < end; g += kRadixUnroll * 64) {
        int key[kRadixUnroll];
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u) {
            const int64_t i = g + u * 64 + lane;
            key[u] = i < end ? keys_in[i * stride] : 0;
        }
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u)
            if (g + u * 64 + lane < end) atomicAdd(&base[(key[u] >> shift) & (bins - 1)], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < bins; d += blockDim.x) {
        const int64_t i = (int64_t)d * C + blockIdx.x;
        int run = offs[i] + bsum[i / kScanTile];
#pragma unroll
        for (int w = 0; w < kRadixWaves; ++w) {
            const int c = lds_radix[w * bins + d];
            lds_radix[w * bins + d] = run;
            run += c;
        }
    }
    __syncthreads();
    const unsigned long long lt = (1ull << lane) - 1ull;
    for (int64_t g0 = beg; g0 < end; g0 += kRadixUnroll * 64) {
        int keys[kRadixUnroll], vals[kRadixUnroll];
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u) {
            const int64_t i = g0 + u * 64 + lane;
            keys[u] = i < end ? keys_in[i * stride] : 0;
            vals[u] = i < end ? (vals_in ? vals_in[i] : (int)i) : 0;
        }
#pragma unroll
        for (int u = 0; u < kRadixUnroll; ++u) {
            if (g0 + u * 64 >= end) break; // uniform over the wave
            const bool valid = g0 + u * 64 + lane < end;
            const int d = (keys[u] >> shift) & (bins - 1);
            unsigned long long m = __ballot(valid);
            for (int b = 0; b < bits; ++b) {
                const bool on = (d >> b) & 1;
                const unsigned long long bb = __ballot(on);
                m &= on ? bb : ~bb;
            }
            const int rank = __popcll(m & lt);
            const int b0 = base[d];
            __builtin_amdgcn_wave_barrier();
            if (valid && rank == 0) base[d] = b0 + __popcll(m);
            __builtin_amdgcn_wave_barrier();
            if (valid) {
                keys_out[b0 + rank] = keys[u];
                vals_out[b0 + rank] = vals[u];
            }
        }
    }
}

// bin_start[k] = first position of key k in the sorted keys (n where none), k = 0..K;
// thread i = 0..n
__device__ inline void bin_starts(int64_t i, int64_t n, const int *__restrict__ skeys, int64_t K,
                                  int *__restrict__ bin_start)
{
    const int64_t kprev = i == 0 ? -1 : skeys[i - 1];
    const int64_t knext = i == n ? K : skeys[i];
    for (int64_t k = kprev + 1; k <= knext; ++k) bin_start[k] = (int)i;
}

__global__ __launch_bounds__(256) void k_make_records(int64_t M, const int *__restrict__ sorted,
                                                      const int4 *__restrict__ cell, const float4 *__restrict__ frac,
                                                      const float *__restrict__ dcf, const int *__restrict__ skeys,
                                                      int64_t K, int *__restrict__ bin_start,
                                                      int4 *__restrict__ rec_cell, float4 *__restrict__ rec_frac)
{
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p > M) return;
    bin_starts(p, M, skeys, K, bin_start);
    if (p == M) return;
    const int i = sorted[p];
    const int4 c = cell[i];
    const float4 f = frac[i];
    rec_cell[p] = make_int4(c.x, c.y, c.z, i);
    rec_frac[p] = make_float4(f.x, f.y, f.z, dcf ? dcf[i] : 1.0f);
}

// ---------------------------------------------------------------------------
// (tile, sample) pair records for the output-stationary spread
// ---------------------------------------------------------------------------

struct TileGeom {
    int dim;
    int64_t nf[3];
    int tile[3];
    int ntiles[3];
    int W; // window taps per axis (2 nspread)
};

// Tiles touched by the window [s, s+W) mod nf along one axis, in tap order: the
// consecutive tiles q0, q0 + 1, ... (mod the tile count), n of them.  Tiles are
// chosen so that a window never re-enters a tile it left (T + W - 1 <= nf or T = nf).
__device__ inline void axis_tile_span(int s, int W, int nf, int T, int &q0, int &n)
{
    if (T == nf) {
        q0 = 0;
        n = 1;
        return;
    }
    q0 = s / T;
    const int e = s + W - 1; // last cell, unwrapped
    n = e < nf ? e / T - q0 + 1 : ((nf + T - 1) / T - q0) + (e - nf) / T + 1;
}

// window taps [jlo, jlo+cnt) of a window starting at s that fall in tile q, and the
// tile-local cell of tap jlo
__device__ inline void tap_box(int s, int q, int T, int nf, int W, int &jlo, int &cnt, int &lstart)
{
    const int org = q * T;
    const int teff = min(T, nf - org);
    if (T == nf) {
        jlo = 0;
        cnt = W;
        lstart = s;
        return;
    }
    int v = org - s;
    if (v < 0) v += nf;
    if (v < W) {
        jlo = v;
        cnt = min(W - v, teff);
        lstart = 0;
    } else {
        jlo = 0;
        cnt = min(W, teff - (s - org));
        lstart = s - org;
    }
}

// offs[p] = pairs of the records before p within its scan tile; ret: the pair total and the
// coordinate error flag
__global__ __launch_bounds__(kScanThreads) void k_pair_scan(int64_t M, const int4 *__restrict__ rec_cell, TileGeom g,
                                                            int *__restrict__ offs, int *bsum, int *ticket, int *ret,
                                                            int *err)
{
    scan_tile(
        [&](int64_t p) {
            const int4 rc = rec_cell[p];
            const int s[3] = {rc.x, rc.y, rc.z};
            int n = 1;
            for (int ax = 0; ax < g.dim; ++ax) {
                int q0, na;
                axis_tile_span(s[ax], g.W, (int)g.nf[ax], g.tile[ax], q0, na);
                n *= na;
            }
            return n;
        },
        offs, M, bsum, ticket, ret, err);
}

// The pairs of sample record p are offs[p] .. offs[p] + n - 1 with n = the product of
// its per-axis tile spans, enumerated leading axis outermost: local index
// (i * n1 + k) * n2 + m is tile (q0[0] + i, q0[1] + k, q0[2] + m), each wrapped.
// k_pair_keys writes each pair's spread tile (the sort key) and its record position;
// after the stable sort by tile, k_pair_records rebuilds every record in sorted order
// from its sample record, so only 8 bytes per pair are written in sample order.
__global__ __launch_bounds__(256) void k_pair_keys(int64_t M, const int4 *__restrict__ rec_cell, TileGeom g,
                                                   const int *__restrict__ offs, const int *__restrict__ bsum,
                                                   int *__restrict__ pkey, int *__restrict__ psamp)
{
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= M) return;
    const int4 rc = rec_cell[p];
    int q0[3] = {0, 0, 0}, n[3] = {1, 1, 1};
    axis_tile_span(rc.x, g.W, (int)g.nf[0], g.tile[0], q0[0], n[0]);
    axis_tile_span(rc.y, g.W, (int)g.nf[1], g.tile[1], q0[1], n[1]);
    if (g.dim == 3) axis_tile_span(rc.z, g.W, (int)g.nf[2], g.tile[2], q0[2], n[2]);
    int o = offs[p] + bsum[p / kScanTile];
    int t0 = q0[0];
    for (int i = 0; i < n[0]; ++i) {
        int t1 = q0[1];
        for (int k = 0; k < n[1]; ++k) {
            int t2 = q0[2];
            for (int m = 0; m < n[2]; ++m) {
                int key = t0 * g.ntiles[1] + t1;
                if (g.dim == 3) key = key * g.ntiles[2] + t2;
                pkey[o] = key;
                psamp[o] = (int)p;
                ++o;
                if (++t2 == g.ntiles[2]) t2 = 0;
            }
            if (++t1 == g.ntiles[1]) t1 = 0;
        }
        if (++t0 == g.ntiles[0]) t0 = 0;
    }
}

// Pair q of the tile-sorted order: its sample record is p = sorted[q] (the sort carries the
// sample indices as values), its tile the sorted key (148 -> 113 us for 2.7 M pairs against
// finding the tile from the pair's original index); the record is
//   a = {orig, j0 | j1<<8 | j2<<16, c0 | c1<<8 | c2<<16, l0 | l1<<10 | l2<<20}
//   b = {t0, t1, t2, dcf} (float bits)
// (j = first window tap inside the tile, c = taps inside, l = tile-local cell of tap j).
__global__ __launch_bounds__(256) void k_pair_records(int64_t P, const int *__restrict__ sorted,
                                                      const int *__restrict__ skeys, int64_t K,
                                                      int *__restrict__ bin_start, const int4 *__restrict__ rec_cell,
                                                      const float4 *__restrict__ rec_frac, TileGeom g,
                                                      int4 *__restrict__ pa, int4 *__restrict__ pb)
{
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q > P) return;
    bin_starts(q, P, skeys, K, bin_start);
    if (q == P) return;
    const int p = sorted[q];
    const int4 rc = rec_cell[p];
    const float4 rf = rec_frac[p];
    uint32_t key = (uint32_t)skeys[q];
    int t2 = 0;
    if (g.dim == 3) {
        t2 = (int)(key % (uint32_t)g.ntiles[2]);
        key /= (uint32_t)g.ntiles[2];
    }
    const int t1 = (int)(key % (uint32_t)g.ntiles[1]), t0 = (int)(key / (uint32_t)g.ntiles[1]);
    int j0, c0, l0, j1, c1, l1, j2 = 0, c2 = 1, l2 = 0;
    tap_box(rc.x, t0, g.tile[0], (int)g.nf[0], g.W, j0, c0, l0);
    tap_box(rc.y, t1, g.tile[1], (int)g.nf[1], g.W, j1, c1, l1);
    if (g.dim == 3) tap_box(rc.z, t2, g.tile[2], (int)g.nf[2], g.W, j2, c2, l2);
    pa[q] = make_int4(rc.w, j0 | (j1 << 8) | (j2 << 16), c0 | (c1 << 8) | (c2 << 16), l0 | (l1 << 10) | (l2 << 20));
    pb[q] = make_int4(__float_as_int(rf.x), __float_as_int(rf.y), __float_as_int(rf.z), __float_as_int(rf.w));
}

// Spread work items, built on the device from the tile offsets pstart[K + 1] (the
// rule of the host planner's build_work_items): tile k with n pairs gets one item
// {k, pbeg, pend, -1}, or, when n > chunk, ceil(n / chunk) slices {k, ..., slot} that
// write consecutive partial slots and one reduce item {k, slot0, slices, 0}.  The
// items of tiles with pairs come first, in tile order, then one item per empty tile,
// in tile order (a launch that need not write empty tiles takes only the first
// part).  Items, empty-tile items, slots and reduce items are numbered by exclusive
// scans of the per-tile counts (k_item_scan).  The gather's items are numbered the same
// way from the gather tiles' sample offsets.
__global__ __launch_bounds__(kScanThreads) void k_item_scan(int64_t K, const int *__restrict__ pstart, int chunk,
                                                            int4 *__restrict__ off, int *bsum, int *ticket, int *ret)
{
    const int64_t base = (int64_t)blockIdx.x * kItemTile + (int64_t)threadIdx.x * 4;
    int c[4][4], sum[4] = {0, 0, 0, 0}, total[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t k = base + i;
        const int n = k < K ? pstart[k + 1] - pstart[k] : 0;
        const int nch = (n + chunk - 1) / chunk;
        c[i][0] = nch;                             // work items
        c[i][1] = k < K && n == 0 ? 1 : 0;         // items of empty tiles
        c[i][2] = n > chunk ? nch : 0;             // partial slots
        c[i][3] = n > chunk ? 1 : 0;               // reduce items
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] += c[i][j];
    }
    block_exclusive_scan<4>(sum, total);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (base + i < K) off[base + i] = make_int4(sum[0], sum[1], sum[2], sum[3]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] += c[i][j];
    }
    int64_t grand[4];
    if (scan_block_totals<4>(bsum, ticket, total, grand) && threadIdx.x == 0)
        for (int j = 0; j < 4; ++j) ret[j] = (int)grand[j]; // at most tiles + pairs / chunk
}

// reduce null: gather items (none for empty tiles).  bsum: the block offsets of
// k_item_scan, then the grand totals.
__global__ __launch_bounds__(256) void k_item_write(int64_t K, const int *__restrict__ pstart, int chunk,
                                                    const int4 *__restrict__ off, const int4 *__restrict__ bsum,
                                                    int64_t nb, int4 *__restrict__ items, int4 *__restrict__ reduce)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    const int b = pstart[k], e = pstart[k + 1];
    const int4 o = off[k], s = bsum[k / kItemTile];
    if (e == b) {
        if (reduce) items[bsum[nb].x + o.y + s.y] = make_int4((int)k, b, e, -1);
        return;
    }
    const int i0 = o.x + s.x;
    if (!reduce) {
        for (int c = 0, x = b; x < e; ++c, x += chunk) items[i0 + c] = make_int4((int)k, x, min(e, x + chunk), 0);
        return;
    }
    if (e - b <= chunk) {
        items[i0] = make_int4((int)k, b, e, -1);
        return;
    }
    const int nch = (e - b + chunk - 1) / chunk, s0 = o.z + s.z;
    reduce[o.w + s.w] = make_int4((int)k, s0, nch, 0);
    for (int c = 0; c < nch; ++c) items[i0 + c] = make_int4((int)k, b + c * chunk, min(e, b + (c + 1) * chunk), s0 + c);
}

// Occupancy row masks: one word per column of spread tiles (ncolt = ntiles[1] *
// ntiles[2] columns), bit b set when one of the leading-axis tiles [b mask_k,
// (b + 1) mask_k) of the column holds pairs; one wave per column, a bit per lane.
__global__ __launch_bounds__(256) void k_occ_masks(int64_t ncolt, int nt0, int mask_k, const int *__restrict__ pstart,
                                                   unsigned long long *__restrict__ occ)
{
    const int lane = threadIdx.x & 63;
    for (int64_t c = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); c < ncolt; c += (int64_t)gridDim.x * 4) {
        bool on = false;
        for (int i = 0; i < mask_k; ++i) {
            const int t0 = lane * mask_k + i;
            if (t0 >= nt0) break;
            const int64_t k = t0 * ncolt + c;
            on = on || pstart[k + 1] > pstart[k];
        }
        const unsigned long long m = __ballot(on);
        if (lane == 0) occ[c] = m;
    }
}

// ---------------------------------------------------------------------------
// Adjoint spread: output-stationary tiles accumulated in registers.
//
// A work item is a tile and a slice of at most kSpreadChunk of the (tile,
// sample) pair records whose windows touch it.  The workgroup splits the tile
// into blocks of 64 cells (4x4x4 in 3-D, 8x8 in 2-D), one block per wave and
// one cell per lane; every lane keeps its cell's value for up to 8 coils in
// registers.  Pair records are staged in LDS 64 at a time: the sample's coil
// values (times dcf) and, per axis, a table of the separable kernel weight at
// every tile-local cell, zero outside the window.  A wave then visits the
// staged pairs whose windows reach its block; each lane forms its weight from
// three table reads and accumulates all coils with FMAs.  Nothing is written
// to shared memory by more than one wave, there are no atomics, and every
// lane adds its contributions in the fixed pair order: the result is
// deterministic.  After each batch the plain FP32 batch sums (at most 64
// terms) are folded into Kahan-compensated (sum, compensation) registers.
// The tile is then written to HBM once, coalesced through LDS; slices of a
// split tile go to partial buffers combined by k_spread_reduce.
// ---------------------------------------------------------------------------



#ifndef GN_SPREAD_BATCH
#define GN_SPREAD_BATCH 64
#endif
constexpr int kSpreadBatch = GN_SPREAD_BATCH; // pairs staged in LDS per step (at most one per lane)
constexpr int kSpreadWavesMax = 8;

// Spread tile t has no pairs and no later pass reads it: its cells need not be written.
__device__ inline bool tile_skippable(const SpreadArgs &a, const int4 item)
{
    if (item.y < item.z || !a.occ) return false;
    const uint32_t nt12 = (uint32_t)a.ntiles[1] * (uint32_t)a.ntiles[2];
    const uint32_t t0 = (uint32_t)item.x / nt12, rest = (uint32_t)item.x - t0 * nt12;
    return ((a.occ[rest] >> (t0 / (uint32_t)a.occ_k)) & 1ull) == 0;
}

template <int D, int NCG>
__device__ __forceinline__ void spread_body(const SpreadArgs &a, const int4 item, const int cgi, const int bz)
{
    extern __shared__ float lds_sp[];
    // LDS: weight tables [batch][TT] | coil values [batch][NCG] float2 | masks [batch][3]
    float *s_tab = lds_sp;
    float2 *s_val = (float2 *)(lds_sp + kSpreadBatch * a.TT);
    int *s_msk = (int *)(s_val + kSpreadBatch * NCG);
    int4 *s_pa = (int4 *)(s_msk + kSpreadBatch * 4);
    float4 *s_pb = (float4 *)(s_pa + kSpreadBatch);

    if (tile_skippable(a, item)) return; // uniform over the workgroup
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int nwaves = blockDim.x >> 6;
    const int cg0 = cgi * NCG;
    const int ncg = (int)min((int64_t)NCG, a.nc - cg0);
    const int T0 = a.tile[0], T1 = a.tile[1], T2 = (D == 3) ? a.tile[2] : 1;

    // this wave's block (block index = blockIdx.z * waves + wave) and this lane's cell
    const int nb = a.nblk[0] * a.nblk[1] * (D == 3 ? a.nblk[2] : 1);
    const int bidx = bz * nwaves + wave;
    const bool has_block = bidx < nb;
    int bq0, bq1, bq2 = 0;
    if (D == 3) {
        bq2 = bidx % a.nblk[2];
        bq1 = (bidx / a.nblk[2]) % a.nblk[1];
        bq0 = bidx / (a.nblk[2] * a.nblk[1]);
    } else {
        bq1 = bidx % a.nblk[1];
        bq0 = bidx / a.nblk[1];
    }
    int L0, L1, L2 = 0;
    if (D == 3) {
        L2 = bq2 * a.blk[2] + (lane % a.blk[2]);
        L1 = bq1 * a.blk[1] + (lane / a.blk[2]) % a.blk[1];
        L0 = bq0 * a.blk[0] + lane / (a.blk[2] * a.blk[1]);
    } else {
        L1 = bq1 * a.blk[1] + (lane % a.blk[1]);
        L0 = bq0 * a.blk[0] + lane / a.blk[1];
    }
    const bool in_tile = has_block && L0 < T0 && L1 < T1 && L2 < T2;
    // lanes of a partial block read a valid table entry; their result is never stored
    L0 = min(L0, T0 - 1);
    L1 = min(L1, T1 - 1);
    L2 = min(L2, T2 - 1);
    // bit masks of the block's cells per axis (tile extents <= 32)
    uint32_t bm0 = 0, bm1 = 0, bm2 = 1;
    if (has_block) {
        for (int i = 0; i < a.blk[0]; ++i) bm0 |= (bq0 * a.blk[0] + i < T0) ? (1u << (bq0 * a.blk[0] + i)) : 0u;
        for (int i = 0; i < a.blk[1]; ++i) bm1 |= (bq1 * a.blk[1] + i < T1) ? (1u << (bq1 * a.blk[1] + i)) : 0u;
        if (D == 3) {
            bm2 = 0;
            for (int i = 0; i < a.blk[2]; ++i) bm2 |= (bq2 * a.blk[2] + i < T2) ? (1u << (bq2 * a.blk[2] + i)) : 0u;
        }
    }
    const int to1 = T0, to2 = T0 + T1; // table offsets of axes 1 and 2

    float sr[NCG], si[NCG], kr[NCG], ki[NCG];
#pragma unroll
    for (int c = 0; c < NCG; ++c) sr[c] = si[c] = kr[c] = ki[c] = 0.f;

    for (int base = item.y; base < item.z; base += kSpreadBatch) {
        const int n = min(kSpreadBatch, item.z - base);
        __syncthreads(); // previous batch fully consumed
        // phase 1: one thread per pair loads its record and coil values, builds the masks
        if (tid < n) {
            const int q = base + tid;
            const int4 pa = a.pair_a[q];
            const int4 pbi = a.pair_b[q];
            const float4 pb = make_float4(__int_as_float(pbi.x), __int_as_float(pbi.y), __int_as_float(pbi.z),
                                          __int_as_float(pbi.w));
            s_pa[tid] = pa;
            s_pb[tid] = pb;
            const float scale = a.use_dcf ? pb.w : 1.0f;
#pragma unroll
            for (int c = 0; c < NCG; ++c) {
                float2 v = make_float2(0.f, 0.f);
                if (c < ncg) {
                    const int64_t coil = cg0 + c;
                    v = (a.layout == GN_COIL_LAST) ? a.in[(int64_t)pa.x * a.nc + coil] : a.in[coil * a.M + pa.x];
                }
                s_val[tid * NCG + c] = make_float2(v.x * scale, v.y * scale);
            }
            // valid tile-local cells of the window per axis: (L - l) mod T < c
            const int Ts[3] = {T0, T1, T2};
            for (int ax = 0; ax < D; ++ax) {
                const int l = (ax == 0 ? pa.w : ax == 1 ? (pa.w >> 10) : (pa.w >> 20)) & 0x3ff;
                const int c = (pa.z >> (8 * ax)) & 0xff;
                uint32_t m = 0;
                for (int r = 0; r < c; ++r) {
                    int L = l + r;
                    if (L >= Ts[ax]) L -= Ts[ax];
                    m |= 1u << L;
                }
                s_msk[tid * 4 + ax] = (int)m;
            }
        }
        __syncthreads();
        // phase 2: weight tables, one entry per (pair, axis, tile-local cell)
        for (int e = tid; e < n * a.TT; e += blockDim.x) {
            const int k = e / a.TT;
            const int i = e - k * a.TT;
            const int ax = i < to1 ? 0 : (i < to2 ? 1 : 2);
            const int L = i - (ax == 0 ? 0 : (ax == 1 ? to1 : to2));
            const int4 pa = s_pa[k];
            const float4 pb = s_pb[k];
            const int Tax = ax == 0 ? T0 : (ax == 1 ? T1 : T2);
            const int l = (ax == 0 ? pa.w : ax == 1 ? (pa.w >> 10) : (pa.w >> 20)) & 0x3ff;
            const int c = (pa.z >> (8 * ax)) & 0xff;
            const int j = (pa.y >> (8 * ax)) & 0xff;
            int rel = L - l;
            if (rel < 0) rel += Tax;
            float w = 0.f;
            if (rel < c) {
                const float t = ax == 0 ? pb.x : (ax == 1 ? pb.y : pb.z);
                const float u = t + (float)(a.ns - j - rel);
                w = exp2f(-a.coef[ax] * u * u);
            }
            s_tab[e] = w;
        }
        __syncthreads();
        // phase 3: each wave visits the pairs that reach its block
        bool hit = false;
        if (lane < n && has_block) {
            const int m0 = s_msk[lane * 4], m1 = s_msk[lane * 4 + 1];
            const int m2 = D == 3 ? s_msk[lane * 4 + 2] : 1;
            hit = ((uint32_t)m0 & bm0) && ((uint32_t)m1 & bm1) && ((uint32_t)m2 & bm2);
        }
        unsigned long long todo = __ballot(hit);
        float ar[NCG], ai[NCG];
#pragma unroll
        for (int c = 0; c < NCG; ++c) ar[c] = ai[c] = 0.f;
        // visits in groups of up to 4 so their LDS reads are in flight together; a
        // missing visit reuses pair 0 with weight 0 (adds exact zeros)
        while (todo) {
            int kk[4];
            float wz[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool some = todo != 0;
                kk[u] = some ? __ffsll((long long)todo) - 1 : 0;
                wz[u] = some ? 1.f : 0.f;
                todo &= todo - 1;
            }
            float w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float *tab = s_tab + kk[u] * a.TT;
                float ww = tab[L0] * tab[to1 + L1];
                if (D == 3) ww *= tab[to2 + L2];
                w[u] = ww * wz[u];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float2 *v = s_val + kk[u] * NCG;
#pragma unroll
                for (int c = 0; c < NCG; ++c) {
                    const float2 vc = v[c];
                    ar[c] = fmaf(w[u], vc.x, ar[c]);
                    ai[c] = fmaf(w[u], vc.y, ai[c]);
                }
            }
        }
        // Kahan fold of this batch's partial sums
#pragma unroll
        for (int c = 0; c < NCG; ++c) {
            const float yr = ar[c] - kr[c], yi = ai[c] - ki[c];
            const float tr = sr[c] + yr, ti = si[c] + yi;
            kr[c] = (tr - sr[c]) - yr;
            ki[c] = (ti - si[c]) - yi;
            sr[c] = tr;
            si[c] = ti;
        }
    }

    // write the tile once, straight from registers
    if (!in_tile) return;
    const int TC = a.TC;
    const int cidx = (L0 * T1 + L1) * T2 + L2;
    if (item.w >= 0) {
        float2 *dst = a.partial + ((int64_t)item.w * a.nc + cg0) * TC + cidx;
#pragma unroll
        for (int c = 0; c < NCG; ++c)
            if (c < ncg) dst[(int64_t)c * TC] = make_float2(sr[c] - kr[c], si[c] - ki[c]);
        return;
    }
    int org[3] = {0, 0, 0}, teff[3] = {1, 1, 1};
    {
        uint32_t r = (uint32_t)item.x; // tile index < 2^31
        for (int ax = D - 1; ax >= 0; --ax) {
            const int qq = (int)(r % (uint32_t)a.ntiles[ax]);
            r /= (uint32_t)a.ntiles[ax];
            org[ax] = qq * a.tile[ax];
            teff[ax] = (int)min((int64_t)a.tile[ax], a.nf[ax] - org[ax]);
        }
    }
    if (L0 >= teff[0] || L1 >= teff[1] || (D == 3 && L2 >= teff[2])) return;
    int64_t gi = (int64_t)(org[0] + L0) * a.nf[1] + (org[1] + L1);
    if (D == 3) gi = gi * a.nf[2] + (org[2] + L2);
#pragma unroll
    for (int c = 0; c < NCG; ++c)
        if (c < ncg) a.grid[(int64_t)(cg0 + c) * a.G + gi] = make_float2(sr[c] - kr[c], si[c] - ki[c]);
}

template <int D, int NCG>
__global__ __launch_bounds__(64 * kSpreadWavesMax) void k_spread(SpreadArgs a)
{
    const uint32_t n = gridDim.x * gridDim.y * gridDim.z;
    const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const uint32_t w = xcd_swizzle(lin, n);
    const int bx = (int)(w % gridDim.x);
    const uint32_t yz = w / gridDim.x;
    spread_body<D, NCG>(a, a.items[bx], (int)(yz % gridDim.y), (int)(yz / gridDim.y));
}

// Batched launch over many plans: bitems[b] = {instance, work item, coil group, 0},
// taken in the XCD-aware order of the plain launch.
template <int D, int NCG>
__global__ __launch_bounds__(64 * kSpreadWavesMax) void k_spread_batch(const SpreadArgs *__restrict__ args,
                                                                        const int4 *__restrict__ bitems)
{
    const uint32_t n = gridDim.x * gridDim.y;
    const uint32_t w = xcd_swizzle(blockIdx.x + gridDim.x * blockIdx.y, n);
    const int4 bi = bitems[w % gridDim.x];
    const SpreadArgs &a = args[bi.x]; // read in place: uniform scalar loads
    spread_body<D, NCG>(a, a.items[bi.y], bi.z, (int)(w / gridDim.x));
}

// ---------------------------------------------------------------------------
// Adjoint spread on the matrix cores (v_mfma_f32_16x16x4_f32).
//
// Same work items, pair staging and weight tables as spread_body; the per-wave
// visit loop becomes small dense products.  A wave's 64-cell block (4x4x4 in 3-D,
// 8x8 in 2-D) is split into four slices of 16 cells (in 3-D the 4x4 x-y cells of
// each of the block's 4 z planes; in 2-D pairs of x rows of 8 cells) and
// accumulates
//     D[cell i][real j] += sum over 4 listed pairs k of  w_k(cell i) * v_k[j]
// with one MFMA per slice and 4 pairs: rows are the slice's cells, columns the
// 2*NCG reals (re, im per coil; zero columns beyond), K the pairs.  Per batch the
// wave lists the staged pairs that reach its block (padded to a multiple of 4 with
// an all-zero pair); each step a lane forms the weight factor its row shares across
// the slices once (3-D: the x-y weight; 2-D: the y weight) and multiplies it by the
// per-slice factor.  The FMAs run on the matrix pipe.  The products are summed in a fixed order,
// so the result is deterministic; batch sums are folded into Kahan-compensated
// registers as in spread_body.  Lane layout of the 16x16x4 f32 operation:
// A[i][k] and B[k][j] in lane i + 16k and j + 16k, D[4g + v][j] in register v of
// lane j + 16g.  Each lane writes its cells of the finished tile straight from its
// registers (16-byte stores of two cells along the last axis).  Needs block-aligned
// tiles (multiples of 4 per axis in 3-D, of 8 in 2-D) of at most kSpreadWavesMax
// blocks: one workgroup per tile and coil group.
// ---------------------------------------------------------------------------

typedef float f32x4 __attribute__((ext_vector_type(4)));

inline size_t spread_mfma_lds_bytes(const SpreadArgs &a, int waves)
{
    const int ttp = a.TT <= 16 ? 16 : a.TT <= 32 ? 32 : a.TT <= 64 ? 64 : 128; // table row stride
    return (size_t)(kSpreadBatch + 1) * ttp * 4 * 2 + (size_t)kSpreadBatch * 16 + (size_t)kSpreadBatch * 64 +
           (size_t)waves * kSpreadBatch * 4;
}

template <int D, int NCG>
__device__ __forceinline__ void spread_mfma_body(const SpreadArgs &a, const int4 item, const int cgi, const int bz)
{
    constexpr int B = kSpreadBatch;
    extern __shared__ float lds_sp[];
    if (tile_skippable(a, item)) return; // uniform over the workgroup
    // LDS: weight tables [B + 1][ttp] | reals [B + 1][ttp] (16 used) | masks [4][B] |
    //      per-axis window parameters [4][B] {l, c, ns - j, t} | per-wave pair lists
    //      [waves][B]; row B of the tables and reals is the all-zero pair.  Table and
    //      value rows have the same stride, so a list entry is the byte offset of a
    //      pair's rows in both.  Masks and parameters are axis-major, so that a wave's
    //      lanes touch consecutive entries.
    const int TT = a.TT;
    // table rows padded to a power of two: a pair's row starts at kk << lgt
    const int ttp = TT <= 16 ? 16 : TT <= 32 ? 32 : TT <= 64 ? 64 : 128;
    const int lgt = __builtin_ctz(ttp);
    float *s_tab = lds_sp;
    float *s_val = s_tab + (B + 1) * ttp;
    int *s_msk = (int *)(s_val + (B + 1) * ttp);
    int4 *s_par = (int4 *)(s_msk + B * 4);
    int *s_list = (int *)(s_par + B * 4);

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // uniform: block set-up on the scalar unit
    const int lane = tid & 63;
    const int nwaves = blockDim.x >> 6;
    const bool split = nwaves >= 2; // phase 1 spread over two waves
    static_assert(kSpreadBatch <= 64, "a batch's pairs are one wave's lanes");
    const int cg0 = cgi * NCG;
    const int ncg = (int)min((int64_t)NCG, a.nc - cg0);
    const int T0 = a.tile[0], T1 = a.tile[1], T2 = (D == 3) ? a.tile[2] : 1;
    const int to1 = T0, to2 = T0 + T1; // table offsets of axes 1 and 2

    const int nb = a.nblk[0] * a.nblk[1] * (D == 3 ? a.nblk[2] : 1);
    const int bidx = bz * nwaves + wave;
    const bool has_block = bidx < nb;
    // block coordinates (wave-uniform integer arithmetic)
    int bq0, bq1, bq2 = 0;
    if (D == 3) {
        const int q2 = bidx / a.nblk[2];
        bq2 = bidx - q2 * a.nblk[2];
        bq0 = q2 / a.nblk[1];
        bq1 = q2 - bq0 * a.nblk[1];
    } else {
        bq0 = bidx / a.nblk[1];
        bq1 = bidx - bq0 * a.nblk[1];
    }
    // this lane's MFMA row ri (a cell of a slice) and its pair slot k = lane / 16
    const int ri = lane & 15, kg = lane >> 4;
    // the wave's block: 4x4x4 cells in 3-D, 8x8 in 2-D, as bit masks per axis
    const uint32_t bm0 = D == 3 ? (0xfu << (bq0 * 4)) : (0xffu << (bq0 * 8));
    const uint32_t bm1 = D == 3 ? (0xfu << (bq1 * 4)) : (0xffu << (bq1 * 8));
    const uint32_t bm2 = D == 3 ? (0xfu << (bq2 * 4)) : 1u;
    // this lane's table columns and value in the rows of pair 0; a list entry (byte
    // offset of a pair's rows) added to them addresses the pair's entries.
    // 3-D: row ri is x-y cell (ri >> 2, ri & 3) of the block, slice s its z plane s:
    //   qx, qy the row's x and y columns, qz the block's 4 z columns (16-byte aligned:
    //   the z table starts at T0 + T1, a multiple of 4).
    // 2-D: row ri is cell (ri >> 3, ri & 7) of a 2 x 8 slice, slice s x rows 2s, 2s + 1:
    //   qx the row's x column in slice 0 (slice s: + 2s), qy its y column.
    const char *pv = (const char *)(s_val + ri);
    const char *qx = (const char *)(s_tab + (D == 3 ? bq0 * 4 + (ri >> 2) : bq0 * 8 + (ri >> 3)));
    const char *qy = (const char *)(s_tab + to1 + (D == 3 ? bq1 * 4 + (ri & 3) : bq1 * 8 + (ri & 7)));
    const char *qz = (const char *)(s_tab + to2 + bq2 * 4);

    if (tid < ttp) s_tab[B * ttp + tid] = 0.f;
    if (tid < 16) s_val[B * ttp + tid] = 0.f;

    // Kahan sums and compensations: set by the first batch (S = batch sums, K = 0), or to
    // zero after the loop when the item has no pairs
    float S[4][4], K[4][4];

    // phase-2 entry of this thread: the 4 consecutive table columns e_i .. e_i + 3 (one
    // axis e_ax, cells e_L .. e_L + 3: the tile extents are multiples of 4) of pairs
    // e_k0, e_k0 + e_kstep, ...; a row holds ttp / 4 column quads (ttp <= 128, so a
    // workgroup of at least 64 threads covers at least two pairs per step)
    const int lgq = lgt - 2;
    const int e_i = (tid & ((ttp >> 2) - 1)) << 2;
    const int e_k0 = tid >> lgq;
    const int e_kstep = (int)blockDim.x >> lgq;
    const int e_ax = e_i < to1 ? 0 : (e_i < to2 ? 1 : 2);
    const int e_L = e_i - (e_ax == 0 ? 0 : (e_ax == 1 ? to1 : to2));
    const int e_T = e_ax == 0 ? T0 : (e_ax == 1 ? T1 : T2);
    const float e_coef = a.coef[e_ax];
    for (int base = item.y; base < item.z; base += B) {
        const int n = min(B, item.z - base);
        if (base != item.y) __syncthreads(); // previous batch fully consumed (uniform)
        // phase 1: per pair, a thread of the first wave loads the coil values and a
        // thread of the second wave (the same thread with one wave) builds the masks and
        // window parameters; each loads the pair's record
        const int pt = split ? (tid & 63) : tid;
        const bool do_vals = tid < n;
        const bool do_msk = split ? (tid >= 64 && pt < n) : tid < n;
        if (do_vals || do_msk) {
            const int q = base + pt;
            const int4 pa = a.pair_a[q];
            const int4 pbi = a.pair_b[q];
            const float4 pb = make_float4(__int_as_float(pbi.x), __int_as_float(pbi.y), __int_as_float(pbi.z),
                                          __int_as_float(pbi.w));
            if (do_vals) {
            const float scale = a.use_dcf ? pb.w : 1.0f;
            float2 v[NCG];
            // coil-last with an even coil count: the pair's coils are contiguous 16-byte pairs
            const bool v4 = NCG >= 2 && a.layout == GN_COIL_LAST && ((a.nc | cg0) & 1) == 0 &&
                            (reinterpret_cast<uintptr_t>(a.in) & 15) == 0;
            if (v4) {
                const float4 *src = reinterpret_cast<const float4 *>(a.in + (int64_t)pa.x * a.nc + cg0);
#pragma unroll
                for (int c2 = 0; c2 < (NCG + 1) / 2; ++c2) {
                    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (2 * c2 < ncg) t = src[c2];
                    v[2 * c2] = make_float2(t.x, t.y);
                    if (2 * c2 + 1 < NCG) v[2 * c2 + 1] = make_float2(t.z, t.w);
                }
            } else {
#pragma unroll
                for (int c = 0; c < NCG; ++c) {
                    v[c] = make_float2(0.f, 0.f);
                    if (c < ncg) {
                        const int64_t coil = cg0 + c;
                        v[c] = (a.layout == GN_COIL_LAST) ? a.in[(int64_t)pa.x * a.nc + coil] : a.in[coil * a.M + pa.x];
                    }
                }
            }
            float4 *dv = (float4 *)(s_val + pt * ttp);
#pragma unroll
            for (int c2 = 0; c2 < 4; ++c2) {
                float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
                if (2 * c2 < NCG) o = make_float4(v[2 * c2].x * scale, v[2 * c2].y * scale, 0.f, 0.f);
                if (2 * c2 + 1 < NCG) {
                    o.z = v[2 * c2 + 1].x * scale;
                    o.w = v[2 * c2 + 1].y * scale;
                }
                dv[c2] = o;
            }
            }
            if (do_msk) {
            // per axis: the window's tile-local cells (L - l) mod T < c as a bit mask,
            // and the parameters of its weights
            const int Ts[3] = {T0, T1, T2};
            const float ts[3] = {pb.x, pb.y, pb.z};
#pragma unroll
            for (int ax = 0; ax < D; ++ax) {
                const int l = (ax == 0 ? pa.w : ax == 1 ? (pa.w >> 10) : (pa.w >> 20)) & 0x3ff;
                const int c = (pa.z >> (8 * ax)) & 0xff;
                const int j = (pa.y >> (8 * ax)) & 0xff;
                uint64_t m = ((1ull << c) - 1) << l;
                m = (m | (m >> Ts[ax])) & ((1ull << Ts[ax]) - 1);
                s_msk[ax * B + pt] = (int)(uint32_t)m;
                s_par[ax * B + pt] = make_int4(l, c, a.ns - j, __float_as_int(ts[ax]));
            }
            }
        }
        __syncthreads();
        // phase 2: weight tables, one entry per (pair, axis, tile-local cell); a thread
        // keeps one column quad (its axis and 4 cells) and steps over the pairs
        if (e_i < TT) {
            for (int k = e_k0; k < n; k += e_kstep) {
                const int4 par = s_par[e_ax * B + k];
                int rel0 = e_L - par.x; // (L - l) mod T of the quad's first column
                if (rel0 < 0) rel0 += e_T;
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int rel = rel0 + i;
                    if (i > 0 && rel >= e_T) rel -= e_T;
                    const float u = __int_as_float(par.w) + (float)(par.z - rel);
                    const float g = __builtin_amdgcn_exp2f(-e_coef * u * u);
                    w[i] = rel < par.y ? g : 0.f;
                }
                *(float4 *)(s_tab + (k << lgt) + e_i) = make_float4(w[0], w[1], w[2], w[3]);
            }
        }
        __syncthreads();
        if (!has_block) continue;
        uint32_t m0 = 0, m1 = 0, m2 = 0;
        if (lane < n) {
            m0 = (uint32_t)s_msk[lane];
            m1 = (uint32_t)s_msk[B + lane];
            m2 = D == 3 ? (uint32_t)s_msk[2 * B + lane] : 1u;
        }
        f32x4 acc[4];
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) acc[sb] = f32x4{0.f, 0.f, 0.f, 0.f};
        // phase 3: one list of the pairs whose windows reach the wave's block; per 4
        // listed pairs a lane forms its weight factors once and feeds the block's four
        // slice MFMAs (a pair that misses a slice adds exact zeros there)
        const bool hit = (m0 & bm0) && (m1 & bm1) && (m2 & bm2);
        const unsigned long long hm = __ballot(hit);
        const int cnt = __popcll(hm);
        const int cpad = (cnt + 3) & ~3;
        int *lst = s_list + wave * B;
        const int pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(hm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hm, 0));
        if (hit) lst[pos] = lane << (lgt + 2);
        if (lane >= cnt && lane < cpad) lst[lane] = B << (lgt + 2);
        // the list was written by this wave's own lanes: order the LDS accesses
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int *lst0 = lst + kg;
        for (int t = 0; t < cpad; t += 4) {
            const int off = lst0[t]; // byte offset of the pair's rows
            const float v = *(const float *)(pv + off);
            float w[4];
            if (D == 3) {
                const float wxy = *(const float *)(qx + off) * *(const float *)(qy + off);
                const float4 wz = *(const float4 *)(qz + off);
                w[0] = wxy * wz.x;
                w[1] = wxy * wz.y;
                w[2] = wxy * wz.z;
                w[3] = wxy * wz.w;
            } else {
                const float wy = *(const float *)(qy + off);
#pragma unroll
                for (int sl = 0; sl < 4; ++sl) w[sl] = *(const float *)(qx + off + 8 * sl) * wy;
            }
#pragma unroll
            for (int sl = 0; sl < 4; ++sl) acc[sl] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[sl], v, acc[sl], 0, 0, 0);
        }
        if (base == item.y) {
            // first batch: the Kahan step from zero sums is exact (S = acc, K = 0)
#pragma unroll
            for (int sb = 0; sb < 4; ++sb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    S[sb][v] = acc[sb][v];
                    K[sb][v] = 0.f;
                }
        } else {
#pragma unroll
            for (int sb = 0; sb < 4; ++sb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float y = acc[sb][v] - K[sb][v];
                    const float tsum = S[sb][v] + y;
                    K[sb][v] = (tsum - S[sb][v]) - y;
                    S[sb][v] = tsum;
                }
        }
    }
    // Write-out straight from the registers.  Lane (ri, kg) holds re (ri even) or im
    // (ri odd) of coil ri >> 1 for 16 cells; for each of 4 outer steps i its 4 values
    // o[z] are consecutive cells along the last axis (3-D: z planes sb of x-y cell
    // (kg, i); 2-D: y cells v of slice i).  Neighbouring lanes swap halves (DPP) so
    // that the even lane holds cells z = 0, 1 and the odd lane cells z = 2, 3 as
    // (re, im) pairs: one 16-byte store per lane and step.  An item without pairs (a
    // tile no window reaches, when empty tiles are written) stores the zero sums.
    const int TC = a.TC;
    const int c = ri >> 1;         // coil within the group
    const bool odd = (ri & 1) != 0;
    const bool writer = c < ncg;
    int org[3] = {0, 0, 0}, teff[3] = {1, 1, 1};
    if (item.w < 0) {
        int r = item.x;
        for (int ax = D - 1; ax >= 0; --ax) {
            const int nt = a.ntiles[ax];
            const int qq = r % nt;
            r /= nt;
            org[ax] = qq * a.tile[ax];
            teff[ax] = (int)min((int64_t)a.tile[ax], a.nf[ax] - org[ax]);
        }
    }
    if (item.y >= item.z || !has_block) { // no pairs: the tile's sums are zero
#pragma unroll
        for (int sb = 0; sb < 4; ++sb)
#pragma unroll
            for (int v = 0; v < 4; ++v) S[sb][v] = K[sb][v] = 0.f;
    }
    const bool wide = ((a.G | a.nf[D - 1]) & 1) == 0;
    const int tl = teff[D - 1];
    // this lane's cells of step i: 3-D (L0b, L1b + i, L2), 2-D (L0b + 2 i, L1b); the
    // addresses of step 0 plus i times the step's stride
    const int L0b = D == 3 ? bq0 * 4 + kg : bq0 * 8 + (kg >> 1);
    const int L1b = D == 3 ? bq1 * 4 : bq1 * 8 + 4 * (kg & 1) + (odd ? 2 : 0);
    const int L2 = D == 3 ? bq2 * 4 + (odd ? 2 : 0) : 0;
    const int Ll = D == 3 ? L2 : L1b; // the pair's cell along the last axis
    const bool slot = item.w >= 0;
    float2 *dst0;
    int64_t step;
    bool lane_ok = writer;
    if (slot) {
        dst0 = a.partial + ((int64_t)item.w * a.nc + cg0 + c) * TC + (D == 3 ? (L0b * T1 + L1b) * T2 + L2 : L0b * T1 + L1b);
        step = D == 3 ? T2 : 2 * T1;
    } else {
        lane_ok = lane_ok && Ll < tl && (D == 2 || L0b < teff[0]);
        int64_t gi = (int64_t)(org[0] + L0b) * a.nf[1] + (org[1] + L1b);
        if (D == 3) gi = gi * a.nf[2] + (org[2] + L2);
        dst0 = a.grid + (int64_t)(cg0 + c) * a.G + gi;
        step = D == 3 ? a.nf[2] : 2 * a.nf[1];
    }
    const bool pairw = slot || (wide && Ll + 1 < tl);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float o[4];
#pragma unroll
        for (int z = 0; z < 4; ++z) o[z] = D == 3 ? S[z][i] - K[z][i] : S[i][z] - K[i][z];
        // quad_perm [1, 0, 3, 2]: the value of lane ^ 1
        const float r0 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? o[0] : o[2]), 0xb1, 0xf, 0xf, false));
        const float r1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? o[1] : o[3]), 0xb1, 0xf, 0xf, false));
        const float4 w = odd ? make_float4(r0, o[2], r1, o[3]) : make_float4(o[0], r0, o[1], r1);
        if (!lane_ok) continue;
        if (!slot && (D == 3 ? L1b + i >= teff[1] : L0b + 2 * i >= teff[0])) continue;
        float2 *dst = dst0 + i * step;
        if (pairw) {
            *(float4 *)dst = w;
        } else {
            dst[0] = make_float2(w.x, w.y);
            if (Ll + 1 < tl) dst[1] = make_float2(w.z, w.w);
        }
    }
}


template <int D, int NCG>
__global__ __launch_bounds__(64 * kSpreadWavesMax) void k_spread_mfma(SpreadArgs a)
{
    const uint32_t n = gridDim.x * gridDim.y * gridDim.z;
    const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const uint32_t w = xcd_swizzle(lin, n);
    const int bx = (int)(w % gridDim.x);
    const uint32_t yz = w / gridDim.x;
    spread_mfma_body<D, NCG>(a, a.items[bx], (int)(yz % gridDim.y), (int)(yz / gridDim.y));
}

template <int D, int NCG>
__global__ __launch_bounds__(64 * kSpreadWavesMax) void k_spread_mfma_batch(const SpreadArgs *__restrict__ args,
                                                                             const int4 *__restrict__ bitems)
{
    const uint32_t n = gridDim.x * gridDim.y;
    const uint32_t w = xcd_swizzle(blockIdx.x + gridDim.x * blockIdx.y, n);
    const int4 bi = bitems[w % gridDim.x];
    const SpreadArgs &a = args[bi.x]; // read in place: uniform scalar loads
    spread_mfma_body<D, NCG>(a, a.items[bi.y], bi.z, (int)(w / gridDim.x));
}

// ---------------------------------------------------------------------------
// Adjoint spread of few coils, one wave per tile (v_mfma_f32_16x16x4_f32).
//
// For the default tiles (4 x 4 x 8 cells in 3-D, 8 x 16 in 2-D), whose 128 cells are 16
// "row" cells (the x-y cells, or the 16 y cells) times 8 "slices" (the z planes, or the x
// rows).  A pair's weight is w_row(i) w_slice(s) and its value v[real], so with
//     A[i][k] = w_row of pair k,     B[k][(s, real)] = w_slice(s) v[real] of pair k
// one product accumulates 16 / R slices of R reals (R / 2 coils) for 4 pairs, and M = R / 2
// products per 4 pairs cover the tile (slice (j / R) M + m in column j of product m):
// where k_spread_mfma leaves 16 - R columns empty, these are full.  Every pair of a tile
// reaches it, so there are no lists or masks, and a one-wave workgroup has no barriers to
// wait at.  Batches of 64 pairs are folded with a Kahan step, as in k_spread_mfma.
// Bound by the batches' table fills and load latency.  128^3, 1,048,576 samples, 1 coil:
// nspread 3 486 -> 231 us, nspread 5 1172 -> 491 us; 4 coils, nspread 3 499 -> 459 us.
// LDS per batch: row weights [B][8 (x, y) or 16], slice weights [B][8], values [B][R]; the
// 4 pairs of a product fall on distinct banks.
// ---------------------------------------------------------------------------
inline size_t spread_tile_lds(int dim, int R)
{
    return (size_t)kSpreadBatch * ((dim == 3 ? 8 : 16) + 8 + R) * sizeof(float);
}

template <int D, int R>
__device__ __forceinline__ void spread_tile_body(const SpreadArgs &a, const int4 item, const int cgi)
{
    constexpr int B = kSpreadBatch, M = R / 2, NC = R / 2; // products per step, coils per wave
    constexpr int RW = D == 3 ? 8 : 16;                    // row-weight stride
    constexpr int T0 = D == 3 ? 4 : 8, T1 = D == 3 ? 4 : 16, T2 = D == 3 ? 8 : 1, TC = 128;
    constexpr int QP = D == 3 ? 4 : 6;                     // table quads per pair
    extern __shared__ float lds_sp[];
    if (tile_skippable(a, item)) return; // uniform over the workgroup
    const int lane = threadIdx.x;
    float *s_row = lds_sp, *s_sl = s_row + B * RW, *s_v = s_sl + B * 8;
    const int cg0 = cgi * NC;
    const int ncg = (int)min((int64_t)NC, a.nc - cg0);
    const int ri = lane & 15, kg = lane >> 4;
    const float *pa0 = s_row + (D == 3 ? (ri >> 2) : ri) + kg * RW, *pa1 = s_row + 4 + (ri & 3) + kg * RW;
    const float *ps = s_sl + (ri / R) * M + kg * 8, *pv = s_v + (ri % R) + kg * R;
    // coil-last with an even coil count: a pair's coils are 16-byte pairs
    const bool v4 = NC >= 2 && a.layout == GN_COIL_LAST && ((a.nc | cg0) & 1) == 0 &&
                    (reinterpret_cast<uintptr_t>(a.in) & 15) == 0;
    float S[M][4], K[M][4];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) S[m][v] = K[m][v] = 0.f;
    for (int base = item.y; base < item.z; base += B) {
        const int n = min(B, item.z - base), np = (n + 3) & ~3;
        if (base != item.y) __syncthreads(); // previous batch fully consumed (uniform)
        // values, one pair per lane (pairs n .. np - 1 are zeros)
        if (lane < np) {
            float2 v[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) v[c] = make_float2(0.f, 0.f);
            float scale = 1.0f;
            if (lane < n) {
                const int orig = a.pair_a[base + lane].x;
                if (a.use_dcf) scale = __int_as_float(a.pair_b[base + lane].w);
                if (v4) {
                    const float4 *src = reinterpret_cast<const float4 *>(a.in + (int64_t)orig * a.nc + cg0);
#pragma unroll
                    for (int c2 = 0; c2 < NC / 2; ++c2)
                        if (2 * c2 < ncg) {
                            const float4 t = src[c2];
                            v[2 * c2] = make_float2(t.x, t.y);
                            v[2 * c2 + 1] = make_float2(t.z, t.w);
                        }
                } else {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        if (c < ncg)
                            v[c] = a.layout == GN_COIL_LAST ? a.in[(int64_t)orig * a.nc + cg0 + c]
                                                            : a.in[(int64_t)(cg0 + c) * a.M + orig];
                }
            }
            if constexpr (NC == 1) {
                *(float2 *)(s_v + lane * R) = make_float2(v[0].x * scale, v[0].y * scale);
            } else {
#pragma unroll
                for (int c2 = 0; c2 < NC / 2; ++c2)
                    *(float4 *)(s_v + lane * R + 4 * c2) =
                        make_float4(v[2 * c2].x * scale, v[2 * c2].y * scale, v[2 * c2 + 1].x * scale,
                                    v[2 * c2 + 1].y * scale);
            }
        }
        // weight tables: 4 consecutive tile-local cells of one axis per step
        for (int q = lane; q < np * QP; q += 64) {
            const int k = q / QP, e = q - k * QP;
            const int ax = D == 3 ? min(e, 2) : (e < 2 ? 0 : 1);
            const int L0 = D == 3 ? (e == 3 ? 4 : 0) : (e < 2 ? 4 * e : 4 * (e - 2));
            const int T = D == 3 ? (ax == 2 ? T2 : T0) : (ax == 0 ? T0 : T1);
            float w[4] = {0.f, 0.f, 0.f, 0.f};
            if (k < n) {
                const int4 pa = a.pair_a[base + k], pb = a.pair_b[base + k];
                const int l = (pa.w >> (10 * ax)) & 0x3ff, c = (pa.z >> (8 * ax)) & 0xff;
                const int j = a.ns - ((pa.y >> (8 * ax)) & 0xff);
                const float t = __int_as_float(ax == 0 ? pb.x : ax == 1 ? pb.y : pb.z);
                const float coef = ax == 0 ? a.coef[0] : ax == 1 ? a.coef[1] : a.coef[2];
                int rel0 = L0 - l; // (L - l) mod T of the quad's first cell
                if (rel0 < 0) rel0 += T;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int rel = rel0 + i;
                    if (i > 0 && rel >= T) rel -= T;
                    const float u = t + (float)(j - rel);
                    const float g = __builtin_amdgcn_exp2f(-coef * u * u);
                    w[i] = rel < c ? g : 0.f;
                }
            }
            float *dst = D == 3 ? (e < 2 ? s_row + k * RW + 4 * e : s_sl + k * 8 + L0)
                                : (e < 2 ? s_sl + k * 8 + L0 : s_row + k * RW + L0);
            *(float4 *)dst = make_float4(w[0], w[1], w[2], w[3]);
        }
        __syncthreads();
        f32x4 acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int t = 0; t < np; t += 4) {
            float w = pa0[t * RW];
            if (D == 3) w *= pa1[t * RW];
            const float v = pv[t * R];
            float b[M];
            if constexpr (M == 4) {
                const float4 x = *(const float4 *)(ps + t * 8);
                b[0] = x.x * v;
                b[1] = x.y * v;
                b[2] = x.z * v;
                b[3] = x.w * v;
            } else if constexpr (M == 2) {
                const float2 x = *(const float2 *)(ps + t * 8);
                b[0] = x.x * v;
                b[1] = x.y * v;
            } else {
                b[0] = ps[t * 8] * v;
            }
#pragma unroll
            for (int m = 0; m < M; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, b[m], acc[m], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float y = acc[m][v] - K[m][v];
                const float ts = S[m][v] + y;
                K[m][v] = (ts - S[m][v]) - y;
                S[m][v] = ts;
            }
    }
    // Write-out.  Lane (ri, kg) holds re (ri even) or im (ri odd) of coil (ri % R) / 2 for
    // slices (ri / R) M + m and row cells 4 kg + v.  Neighbouring lanes swap halves (DPP):
    // the even lane gets row cells v = 0, 1 and the odd lane v = 2, 3 as (re, im) pairs.
    const int c = (ri % R) >> 1;
    const bool odd = (ri & 1) != 0;
    const bool slot = item.w >= 0;
    float2 o[M][2];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        float x[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) x[v] = S[m][v] - K[m][v];
        // quad_perm [1, 0, 3, 2]: the value of lane ^ 1
        const float r0 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? x[0] : x[2]), 0xb1, 0xf, 0xf, false));
        const float r1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? x[1] : x[3]), 0xb1, 0xf, 0xf, false));
        o[m][0] = odd ? make_float2(r0, x[2]) : make_float2(x[0], r0);
        o[m][1] = odd ? make_float2(r1, x[3]) : make_float2(x[1], r1);
    }
    if (c >= ncg) return;
    int org[3] = {0, 0, 0}, te[3] = {T0, T1, T2};
    if (!slot) {
        uint32_t r = (uint32_t)item.x;
#pragma unroll
        for (int ax = D - 1; ax >= 0; --ax) {
            const uint32_t nt = (uint32_t)a.ntiles[ax], qq = r % nt;
            r /= nt;
            org[ax] = (int)qq * (ax == 0 ? T0 : ax == 1 ? T1 : T2);
            te[ax] = (int)min((int64_t)te[ax], a.nf[ax] - org[ax]);
        }
    }
    float2 *dst = slot ? a.partial + ((int64_t)item.w * a.nc + cg0 + c) * TC : a.grid + (int64_t)(cg0 + c) * a.G;
    const bool wide = slot || ((a.G | a.nf[D - 1]) & 1) == 0; // 16-byte pairs along the last axis
    const int s0 = (ri / R) * M;
    if (D == 3) {
        // x = kg, y = 2 odd + i, z = s0 + m
        const int64_t n1 = slot ? T1 : a.nf[1], n2 = slot ? T2 : a.nf[2];
        if (kg >= te[0]) return;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int y = (odd ? 2 : 0) + i;
            if (y >= te[1]) continue;
            float2 *p = dst + ((org[0] + kg) * n1 + (org[1] + y)) * n2 + org[2] + s0;
            if constexpr (M == 1) {
                if (s0 < te[2]) p[0] = o[0][i];
            } else {
#pragma unroll
                for (int m = 0; m < M; m += 2) {
                    if (wide && s0 + m + 1 < te[2]) {
                        *(float4 *)(p + m) = make_float4(o[m][i].x, o[m][i].y, o[m + 1][i].x, o[m + 1][i].y);
                    } else {
                        if (s0 + m < te[2]) p[m] = o[m][i];
                        if (s0 + m + 1 < te[2]) p[m + 1] = o[m + 1][i];
                    }
                }
            }
        }
    } else {
        // x = s0 + m, y = 4 kg + 2 odd + i
        const int64_t n1 = slot ? T1 : a.nf[1];
        const int y = 4 * kg + (odd ? 2 : 0);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (s0 + m >= te[0]) continue;
            float2 *p = dst + (org[0] + s0 + m) * n1 + org[1] + y;
            if (wide && y + 1 < te[1]) {
                *(float4 *)p = make_float4(o[m][0].x, o[m][0].y, o[m][1].x, o[m][1].y);
            } else {
                if (y < te[1]) p[0] = o[m][0];
                if (y + 1 < te[1]) p[1] = o[m][1];
            }
        }
    }
}

template <int D, int R>
__global__ __launch_bounds__(64) void k_spread_tile(SpreadArgs a)
{
    const uint32_t n = gridDim.x * gridDim.y;
    const uint32_t w = xcd_swizzle(blockIdx.x + gridDim.x * blockIdx.y, n);
    spread_tile_body<D, R>(a, a.items[w % gridDim.x], (int)(w / gridDim.x));
}

template <int D, int R>
__global__ __launch_bounds__(64) void k_spread_tile_batch(const SpreadArgs *__restrict__ args,
                                                                            const int4 *__restrict__ bitems)
{
    const int4 bi = bitems[xcd_swizzle(blockIdx.x, gridDim.x)];
    const SpreadArgs &a = args[bi.x]; // read in place: uniform scalar loads
    spread_tile_body<D, R>(a, a.items[bi.y], bi.z);
}

// ---------------------------------------------------------------------------
// Adjoint spread in 2-D on 4 x 4 sub-blocks (v_mfma_f32_16x16x4_f32).
//
// Default 8 x 16 tiles, four waves: wave q takes y cells 4 q .. 4 q + 3, as two 4 x 4
// sub-blocks, and 8 NG coils.  Per batch of 64 pairs a wave lists the pairs whose windows
// reach each sub-block; 4 listed pairs take one weight product wx wy per lane (row = cell)
// and NG matrix products whose columns are the reals of 8 coils.  A window of 6 cells
// fills 0.44 of a 4 x 4 block it reaches, against 0.22 of an 8 x 8 block, so the products
// are half of k_spread_mfma's; the tables and records serve up to 16 coils.
// Bound by the batches' vector instructions and latency (matrix cores about 0.4 busy), so a
// batch's records are held a pair per lane: a wave forms one quad of weights of every pair
// without divisions, tests its own sub-blocks, and takes values' sample indices by lane
// exchange; two list steps' LDS reads are in flight together; 6 waves per SIMD.  256^2,
// 98304 spiral samples, nspread 3 (spread and reduction): 32 coils 112 (8 x 8 blocks) -> 65
// -> 60 us, 8 coils 34 -> 30 us; 16 instances of 128 to 320 with up to 32 coils, forward and
// adjoint, 1579 -> 1485 us.
// LDS rows, one per pair: weights x[8] y[16] | reals [16 NG]; row B is zero (list padding).
// ---------------------------------------------------------------------------
constexpr int kSpreadSubWaves = 4;
constexpr int spread_sub_row(int NG) { return 28 + 16 * NG; } // 4 floats of padding: 16 banks of 16 bytes

inline size_t spread_sub_lds(int NG)
{
    return (size_t)(kSpreadBatch + 1) * spread_sub_row(NG) * 4 + (size_t)kSpreadSubWaves * 2 * kSpreadBatch * 4;
}

template <int NG>
__device__ __forceinline__ void spread_sub_body(const SpreadArgs &a, const int4 item, const int cgi)
{
    constexpr int B = kSpreadBatch, ROW = spread_sub_row(NG), NC = 8 * NG, NT = 64 * kSpreadSubWaves;
    constexpr int T0 = 8, T1 = 16, TC = 128;
    extern __shared__ float lds_sp[];
    if (tile_skippable(a, item)) return; // uniform over the workgroup
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int *s_list = (int *)(lds_sp + (B + 1) * ROW) + wave * 2 * B;
    const int cg0 = cgi * NC;
    const int ncg = (int)min((int64_t)NC, a.nc - cg0);
    const int ri = lane & 15, kg = lane >> 4;
    // coil-last with an even coil count: a pair's coils are 16-byte pairs
    const bool v4 = a.layout == GN_COIL_LAST && ((a.nc | cg0) & 1) == 0 && (reinterpret_cast<uintptr_t>(a.in) & 15) == 0;
    const char *qx = (const char *)(lds_sp + (ri >> 2)), *qy = (const char *)(lds_sp + 8 + 4 * wave + (ri & 3));
    const char *qv = (const char *)(lds_sp + 24 + ri);
    for (int i = tid; i < ROW; i += NT) lds_sp[B * ROW + i] = 0.f;
    float S[2][NG][4], K[2][NG][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) S[s][g][v] = K[s][g][v] = 0.f;
    for (int base = item.y; base < item.z; base += B) {
        const int n = min(B, item.z - base);
        // every wave holds the batch's records, a pair per lane
        int4 pa = make_int4(0, 0, 0, 0), pb = pa;
        if (lane < n) {
            pa = a.pair_a[base + lane];
            pb = a.pair_b[base + lane];
        }
        // values: one 16-byte coil pair per step, loaded before the weights are formed
        constexpr int NV = B * (NC / 2) / NT;
        float4 val[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int q = tid + v * NT, k = q / (NC / 2), c = 2 * (q - k * (NC / 2));
            const int orig = __shfl(pa.x, k);
            float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
            if (k < n) {
                if (v4) {
                    if (c < ncg) t = *reinterpret_cast<const float4 *>(a.in + (int64_t)orig * a.nc + cg0 + c);
                } else {
                    float2 x = make_float2(0.f, 0.f), y = x;
                    if (c < ncg) x = a.layout == GN_COIL_LAST ? a.in[(int64_t)orig * a.nc + cg0 + c] : a.in[(int64_t)(cg0 + c) * a.M + orig];
                    if (c + 1 < ncg) y = a.layout == GN_COIL_LAST ? a.in[(int64_t)orig * a.nc + cg0 + c + 1] : a.in[(int64_t)(cg0 + c + 1) * a.M + orig];
                    t = make_float4(x.x, x.y, y.x, y.y);
                }
            }
            val[v] = t;
        }
        if (base != item.y) __syncthreads(); // previous batch fully consumed (uniform)
        // weight tables: wave w forms quads e = w, w + 4 of 4 consecutive tile-local cells of
        // one axis (two along x, four along y) for the pair of each lane
#pragma unroll
        for (int e = wave; e < 6; e += kSpreadSubWaves) {
            const int ax = e < 2 ? 0 : 1;
            const int L0 = 4 * (ax ? e - 2 : e), T = ax ? T1 : T0;
            const int l = (pa.w >> (10 * ax)) & 0x3ff, c = (pa.z >> (8 * ax)) & 0xff;
            const int j = a.ns - ((pa.y >> (8 * ax)) & 0xff);
            const float t = __int_as_float(ax ? pb.y : pb.x), coef = ax ? a.coef[1] : a.coef[0];
            const int rel0 = (L0 - l) & (T - 1); // (L - l) mod T of the quad's first cell
            float w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int rel = (rel0 + i) & (T - 1);
                const float u = t + (float)(j - rel);
                const float g = __builtin_amdgcn_exp2f(-coef * u * u);
                w[i] = rel < c ? g : 0.f;
            }
            if (lane < n) *(float4 *)(lds_sp + lane * ROW + 4 * e) = make_float4(w[0], w[1], w[2], w[3]);
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int q = tid + v * NT, k = q / (NC / 2), c = 2 * (q - k * (NC / 2));
            const float scale = a.use_dcf ? __int_as_float(__shfl(pb.w, k)) : 1.0f;
            if (k < n)
                *(float4 *)(lds_sp + k * ROW + 24 + 2 * c) =
                    make_float4(val[v].x * scale, val[v].y * scale, val[v].z * scale, val[v].w * scale);
        }
        // pairs that reach this wave's sub-blocks: window cells are (l + i) mod T, i < c, so a
        // block at b is reached when (b - l) mod T is below c or its 4 cells pass T
        const int ly = (4 * wave - (pa.w >> 10)) & (T1 - 1);
        const bool hy = lane < n && (ly < ((pa.z >> 8) & 0xff) || ly > T1 - 4);
        int cnt[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int lx = (4 * s - pa.w) & (T0 - 1);
            const bool hit = hy && (lx < (pa.z & 0xff) || lx > T0 - 4);
            const unsigned long long hm = __ballot(hit);
            cnt[s] = __popcll(hm);
            const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(hm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hm, 0));
            // listed pairs first, then the zero row; entry i of the list is the row of step
            // i / 4 and k group i % 4, kept as 16 steps per k group
            const int i = hit ? rank : cnt[s] + lane - rank;
            s_list[s * B + (i & 3) * (B / 4) + (i >> 2)] = (hit ? lane : B) * (ROW * 4);
        }
        __syncthreads();
        // the lists were written by this wave's own lanes: order the LDS accesses
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            f32x4 acc[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
            // two steps of 4 pairs together: their LDS reads are in flight at once
            const int *lst = s_list + s * B + kg * (B / 4);
            for (int t = 0; t < cnt[s]; t += 8) {
                const int2 off = *(const int2 *)(lst + (t >> 2)); // byte offsets of the pairs' rows
                const float w0 = *(const float *)(qx + 16 * s + off.x) * *(const float *)(qy + off.x);
                const float w1 = *(const float *)(qx + 16 * s + off.y) * *(const float *)(qy + off.y);
                float v0[NG], v1[NG];
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    v0[g] = *(const float *)(qv + 64 * g + off.x);
                    v1[g] = *(const float *)(qv + 64 * g + off.y);
                }
#pragma unroll
                for (int g = 0; g < NG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0, v0[g], acc[g], 0, 0, 0);
#pragma unroll
                for (int g = 0; g < NG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1, v1[g], acc[g], 0, 0, 0);
            }
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float y = acc[g][v] - K[s][g][v];
                    const float ts = S[s][g][v] + y;
                    K[s][g][v] = (ts - S[s][g][v]) - y;
                    S[s][g][v] = ts;
                }
        }
    }
    // Write-out.  Lane (ri, kg) holds re (ri even) or im (ri odd) of coil 8 g + ri / 2 for
    // the cells x = 4 s + kg, y = 4 wave + v.  Neighbouring lanes swap halves (DPP): the
    // even lane gets cells v = 0, 1 and the odd lane v = 2, 3 as (re, im) pairs.
    const bool odd = (ri & 1) != 0;
    const bool slot = item.w >= 0;
    int org0 = 0, org1 = 0, te0 = T0, te1 = T1;
    if (!slot) {
        const uint32_t t1 = (uint32_t)item.x % (uint32_t)a.ntiles[1], t0 = (uint32_t)item.x / (uint32_t)a.ntiles[1];
        org0 = (int)t0 * T0;
        org1 = (int)t1 * T1;
        te0 = (int)min((int64_t)T0, a.nf[0] - org0);
        te1 = (int)min((int64_t)T1, a.nf[1] - org1);
    }
    const bool wide = slot || ((a.G | a.nf[1]) & 1) == 0; // 16-byte pairs of cells
    const int64_t n1 = slot ? T1 : a.nf[1];
    const int y = 4 * wave + (odd ? 2 : 0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int x = 4 * s + kg;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) o[v] = S[s][g][v] - K[s][g][v];
            // quad_perm [1, 0, 3, 2]: the value of lane ^ 1
            const float r0 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? o[0] : o[2]), 0xb1, 0xf, 0xf, false));
            const float r1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(odd ? o[1] : o[3]), 0xb1, 0xf, 0xf, false));
            const float4 w = odd ? make_float4(r0, o[2], r1, o[3]) : make_float4(o[0], r0, o[1], r1);
            const int c = 8 * g + (ri >> 1);
            if (c >= ncg || x >= te0) continue;
            float2 *p = (slot ? a.partial + ((int64_t)item.w * a.nc + cg0 + c) * TC : a.grid + (int64_t)(cg0 + c) * a.G) +
                        (org0 + x) * n1 + org1 + y;
            if (wide && y + 1 < te1) {
                *(float4 *)p = w;
            } else {
                if (y < te1) p[0] = make_float2(w.x, w.y);
                if (y + 1 < te1) p[1] = make_float2(w.z, w.w);
            }
        }
    }
}

template <int NG>
__global__ __launch_bounds__(64 * kSpreadSubWaves, 6) void k_spread_sub(SpreadArgs a)
{
    const uint32_t n = gridDim.x * gridDim.y;
    const uint32_t w = xcd_swizzle(blockIdx.x + gridDim.x * blockIdx.y, n);
    spread_sub_body<NG>(a, a.items[w % gridDim.x], (int)(w / gridDim.x));
}

template <int NG>
__global__ __launch_bounds__(64 * kSpreadSubWaves) void k_spread_sub_batch(const SpreadArgs *__restrict__ args,
                                                                           const int4 *__restrict__ bitems)
{
    const int4 bi = bitems[xcd_swizzle(blockIdx.x, gridDim.x)];
    const SpreadArgs &a = args[bi.x]; // read in place: uniform scalar loads
    spread_sub_body<NG>(a, a.items[bi.y], bi.z);
}

// Kahan-compensated sum of the partial tiles of each split tile, in slice order; one
// thread per (coil, cell) of a tile, blockIdx.y over its cells of every coil (as one block
// of 1024 threads per tile: 27 instead of 11 us at 32 coils and 256^2).
constexpr int kReduceThreads = 256;
constexpr int kReduceBlocks = 16; // blocks per tile at most
template <int D>
__device__ __forceinline__ void spread_reduce_body(const SpreadArgs &a, const int4 it)
{
    // it = {tile, slot0, nslots}
    int org[3] = {0, 0, 0}, teff[3] = {1, 1, 1};
    {
        uint32_t r = (uint32_t)it.x; // tile index < 2^31
        for (int ax = D - 1; ax >= 0; --ax) {
            const int q = (int)(r % (uint32_t)a.ntiles[ax]);
            r /= (uint32_t)a.ntiles[ax];
            org[ax] = q * a.tile[ax];
            teff[ax] = (int)min((int64_t)a.tile[ax], a.nf[ax] - org[ax]);
        }
    }
    const int TC = a.TC;
    const int T1 = a.tile[1], T2 = (D == 3) ? a.tile[2] : 1;
    const int ne = (int)(TC * a.nc); // a tile's cells of every coil (< 2^31)
    for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < ne; e += blockDim.x * gridDim.y) {
        const int64_t coil = e / TC;
        const int cidx = e - (int)coil * TC;
        int x0, x1, x2 = 0;
        if (D == 3) {
            x2 = cidx % T2;
            x1 = (cidx / T2) % T1;
            x0 = cidx / (T2 * T1);
        } else {
            x1 = cidx % T1;
            x0 = cidx / T1;
        }
        if (x0 >= teff[0] || x1 >= teff[1] || (D == 3 && x2 >= teff[2])) continue;
        float sr = 0.f, si = 0.f, cr = 0.f, ci = 0.f;
        const float2 *src = a.partial + (int64_t)it.y * a.nc * TC + coil * TC + cidx;
        const int64_t sstride = a.nc * TC;
        // slices in groups of kStageUnroll: the loads are issued together, the
        // compensated sum still runs in slice order
        for (int s0 = 0; s0 < it.z; s0 += kStageUnroll) {
            float2 v[kStageUnroll];
#pragma unroll
            for (int u = 0; u < kStageUnroll; ++u)
                v[u] = s0 + u < it.z ? src[(int64_t)(s0 + u) * sstride] : make_float2(0.f, 0.f);
#pragma unroll
            for (int u = 0; u < kStageUnroll; ++u) {
                if (s0 + u >= it.z) break;
                const float yr = v[u].x - cr, yi = v[u].y - ci;
                const float tr = sr + yr, ti = si + yi;
                cr = (tr - sr) - yr;
                ci = (ti - si) - yi;
                sr = tr;
                si = ti;
            }
        }
        int64_t gi = (int64_t)(org[0] + x0) * a.nf[1] + (org[1] + x1);
        if (D == 3) gi = gi * a.nf[2] + (org[2] + x2);
        a.grid[coil * a.G + gi] = make_float2(sr - cr, si - ci);
    }
}

template <int D>
__global__ __launch_bounds__(kReduceThreads) void k_spread_reduce(SpreadArgs a, const int4 *__restrict__ ritems)
{
    spread_reduce_body<D>(a, ritems[blockIdx.x]);
}

// bitems[b] = {instance, reduce item}
template <int D>
__global__ __launch_bounds__(kReduceThreads) void k_spread_reduce_batch(const SpreadArgs *__restrict__ args,
                                                             const int4 *__restrict__ bitems)
{
    const int4 bi = bitems[blockIdx.x];
    const SpreadArgs &a = args[bi.x]; // read in place: uniform scalar loads
    spread_reduce_body<D>(a, a.reduce_items[bi.y]);
}

// ---------------------------------------------------------------------------
// Forward gather: one workgroup per (work item, coil pair).  A work item is a
// gather tile and up to kGatherChunk of its samples.  The tile plus its window
// halo is staged in LDS as 16-byte cells holding both coils of the pair, with
// coalesced loads; every thread then interpolates one sample of both coils from
// LDS, one 16-byte LDS read per tap, forming the separable 1-D weights in
// registers.  With an odd coil count the last pair's second coil is zero and
// not written.
// ---------------------------------------------------------------------------

static_assert(kGatherCoils == 2, "the gather stages coil pairs");

// A staged cell: coils g0 and g1 (zeros for a missing second coil), or g0 alone.
template <typename Cell>
__device__ inline Cell load_cell(const float2 *__restrict__ g0, const float2 *__restrict__ g1, bool two, int64_t i)
{
    if constexpr (sizeof(Cell) == sizeof(float4)) {
        const float2 x0 = g0[i], x1 = two ? g1[i] : make_float2(0.f, 0.f);
        return make_float4(x0.x, x0.y, x1.x, x1.y);
    } else {
        return g0[i];
    }
}

template <int D, typename Cell>
__device__ inline void stage_region_flat(Cell *lds, const float2 *__restrict__ g0, const float2 *__restrict__ g1,
                                         bool two, const int64_t *nf, const int *org, int R1, int R2, int RC)
{
    // A thread takes cells rr = tid, tid + NT, ... of the region, rr = (r0 * R1 + r1) * R2 + r2
    // (R2 = 1 in 2-D), and steps its (r0, r1, r2) by NT = (d0 * R1 + d1) * R2 + d2 with
    // carries instead of dividing for every cell.
    const int NT = blockDim.x;
    const int R12 = R1 * R2;
    const int d0 = NT / R12, dr = NT - d0 * R12, d1 = dr / R2, d2 = dr - d1 * R2;
    const int tid = threadIdx.x;
    int r0 = tid / R12;
    int r1 = (tid - r0 * R12) / R2;
    int r2 = tid - r0 * R12 - r1 * R2;
    const int nf0 = (int)nf[0], nf1 = (int)nf[1], nf2 = D == 3 ? (int)nf[2] : 1;
    for (int base = tid; base < RC; base += kStageUnroll * NT) {
        Cell v[kStageUnroll];
#pragma unroll
        for (int u = 0; u < kStageUnroll; ++u) {
            const int rr = base + u * NT;
            if (rr < RC) {
                int q0 = org[0] + r0;
                if (q0 >= nf0) q0 -= nf0;
                int q1 = org[1] + r1;
                if (q1 >= nf1) q1 -= nf1;
                int64_t gi = (int64_t)q0 * nf1 + q1;
                if (D == 3) {
                    int q2 = org[2] + r2;
                    if (q2 >= nf2) q2 -= nf2;
                    gi = gi * nf2 + q2;
                }
                v[u] = load_cell<Cell>(g0, g1, two, gi);
            }
            r2 += d2;
            int c = r2 >= R2 ? 1 : 0;
            r2 -= c * R2;
            r1 += d1 + c;
            c = r1 >= R1 ? 1 : 0;
            r1 -= c * R1;
            r0 += d0 + c;
        }
#pragma unroll
        for (int u = 0; u < kStageUnroll; ++u) {
            const int rr = base + u * NT;
            if (rr < RC) lds[rr] = v[u];
        }
    }
}

// Row-wise staging pays when whole rows fill at least 7/8 of a wave's lanes (21 or
// 29 cells: 63 or 58 lanes; 25 cells would leave 14 idle) and grid indices fit 31 bits.
__device__ inline bool rows_stage_ok(int RL, int64_t G)
{
    return RL <= 64 && (64 / RL) * RL >= 56 && G < 0x7fffffffll;
}

// Row-wise staging of the same region for rows of at most 64 cells along the last
// (contiguous) axis and grids of fewer than 2^31 cells per coil.  Each wave takes
// 64 / RL whole rows per step (lane = row slot * RL + cell), so a lane keeps one
// last-axis cell for the whole loop (its wrapped grid index is computed once) and
// only the leading-axis coordinates of its row advance, with one carry; grid indices
// are 32-bit.  A wave's lanes write consecutive LDS cells.
template <int D, typename Cell>
__device__ inline void stage_region_rows(Cell *lds, const float2 *__restrict__ g0, const float2 *__restrict__ g1,
                                         bool two, const int64_t *nf, const int *org, int R0, int R1, int R2)
{
    constexpr int U = 4; // rows per lane whose loads are in flight together
    const int RL = D == 3 ? R2 : R1;
    const int nrow = D == 3 ? R0 * R1 : R0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rpw = 64 / RL;
    const int k = lane / RL, c = lane - k * RL;
    if (k >= rpw) return;
    const int step = (int)(blockDim.x >> 6) * rpw;
    const int nf0 = (int)nf[0], nf1 = (int)nf[1], nfl = (int)nf[D - 1];
    int ql = org[D - 1] + c;
    if (ql >= nfl) ql -= nfl;
    int rho = wave * rpw + k;
    int r0, r1 = 0, s0 = step, s1 = 0;
    if (D == 3) {
        r0 = rho / R1;
        r1 = rho - r0 * R1;
        s0 = step / R1;
        s1 = step - s0 * R1;
    } else {
        r0 = rho;
    }
    const uint32_t nf2 = D == 3 ? (uint32_t)nf[2] : 1u;
    for (; rho < nrow; rho += U * step) {
        Cell v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (rho + u * step < nrow) {
                int q0 = org[0] + r0;
                if (q0 >= nf0) q0 -= nf0;
                uint32_t off;
                if (D == 3) {
                    int q1 = org[1] + r1;
                    if (q1 >= nf1) q1 -= nf1;
                    off = ((uint32_t)q0 * (uint32_t)nf1 + (uint32_t)q1) * nf2 + (uint32_t)ql;
                } else {
                    off = (uint32_t)q0 * (uint32_t)nf1 + (uint32_t)ql;
                }
                v[u] = load_cell<Cell>(g0, g1, two, off);
            }
            if (D == 3) {
                r1 += s1;
                const int cc = r1 >= R1 ? 1 : 0;
                r1 -= cc * R1;
                r0 += s0 + cc;
            } else {
                r0 += step;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (rho + u * step < nrow) lds[(rho + u * step) * RL + c] = v[u];
    }
}

// acc += w * v on the coils of a staged cell
__device__ inline void fma_cell(float2 &acc, float w, const float2 v)
{
    acc.x += w * v.x;
    acc.y += w * v.y;
}
__device__ inline void fma_cell(float4 &acc, float w, const float4 v)
{
    acc.x += w * v.x;
    acc.y += w * v.y;
    acc.z += w * v.z;
    acc.w += w * v.w;
}

// Lanes of the gather-type kernels when tps lanes share a sample: sample grp of the
// wave, tap share sub; a sample's other lanes are lane + k * stride (k < tps - sub).
// Wide windows (nspread >= 4) space a sample's lanes spw apart, so lanes 0 .. spw-1
// hold consecutive samples and the LDS-bank order of the records (k_bank_order)
// holds for every tps (nspread 5: gather 1.86 -> 1.79 ms); at nspread 3 adjacent
// lanes per sample measured 1% faster.
template <int NS>
__device__ inline void lane_layout(int lane, int tps, int spw, int *grp, int *sub, int *stride)
{
    if (NS >= 4) {
        *sub = lane / spw;
        *grp = lane - *sub * spw;
        *stride = spw;
    } else {
        *grp = lane / tps;
        *sub = lane - *grp * tps;
        *stride = 1;
    }
}

// Tap weights use the hardware exp2 (v_exp_f32) directly.  The exponent is
// coef * u^2 with coef = pi (rat - 1/2) / (rat ns ln 2) and |u| <= ns + 1, so every
// weight is >= 2^-82 for nspread <= 16: far from the denormal range, where the
// hardware exp2 and exp2f agree bit for bit.
template <int D, int NS, bool WRAP>
__device__ __forceinline__ void gather_body(const GatherArgs &a, const int4 item, const int cgi)
{
    constexpr int W = 2 * NS;
    extern __shared__ float4 lds_pair[];
    const int cg0 = cgi * kGatherCoils;
    const bool two = cg0 + 1 < a.nc;

    int org[3] = {0, 0, 0};
    {
        uint32_t r = (uint32_t)item.x; // tile index < 2^31
        for (int ax = D - 1; ax >= 0; --ax) {
            org[ax] = (int)(r % (uint32_t)a.ntiles[ax]) * a.tile[ax];
            r /= (uint32_t)a.ntiles[ax];
        }
    }
    const int R0 = a.region[0], R1 = a.region[1], R2 = (D == 3) ? a.region[2] : 1;
    const int RC = R0 * R1 * R2;

    const float2 *g0 = a.grid + (int64_t)cg0 * a.G;
    if (rows_stage_ok(D == 3 ? R2 : R1, a.G))
        stage_region_rows<D>(lds_pair, g0, g0 + a.G, two, a.nf, org, R0, R1, R2);
    else
        stage_region_flat<D>(lds_pair, g0, g0 + a.G, two, a.nf, org, R1, R2, RC);
    __syncthreads();
    // Threads per sample: a work item's samples are spread over all waves of the
    // workgroup.  The tps lanes of a sample take the leading-axis taps t0 = sub,
    // sub + tps, ... (tps divides W); lane sub 0 then adds the partial sums of lanes
    // sub 1 .. tps-1 in that order, so the result does not depend on timing or on the
    // lane layout (lane_layout).
    const int n = item.z - item.y;
    const int nwaves = kGatherThreads / 64;
    int tps = 1;
#pragma unroll
    for (int d = 2; d <= 8; ++d)
        if (W % d == 0 && n <= nwaves * (64 / d)) tps = d;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int spw = 64 / tps;               // samples per wave
    int grp, sub, stride;
    lane_layout<NS>(lane, tps, spw, &grp, &sub, &stride);
    for (int s0 = 0; s0 < n; s0 += nwaves * spw) {
        const int slot = s0 + wave * spw + grp;
        const bool valid = grp < spw && sub < tps && slot < n;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        int orig = 0;
        if (valid) {
            const int j = item.y + slot;
            const int4 rc = a.rec_cell[j];
            const float4 rf = a.rec_frac[j];
            orig = rc.w;
            int l0 = rc.x - org[0];
            if (l0 < 0) l0 += (int)a.nf[0];
            int l1 = rc.y - org[1];
            if (l1 < 0) l1 += (int)a.nf[1];
            int l2 = 0;
            if (D == 3) {
                l2 = rc.z - org[2];
                if (l2 < 0) l2 += (int)a.nf[2];
            }
            float w1[W], w2[D == 3 ? W : 1];
#pragma unroll
            for (int t = 0; t < W; ++t) {
                const float u1 = rf.y + (float)(NS - t);
                w1[t] = __builtin_amdgcn_exp2f(-a.coef[1] * u1 * u1);
                if (D == 3) {
                    const float u2 = rf.z + (float)(NS - t);
                    w2[t] = __builtin_amdgcn_exp2f(-a.coef[2] * u2 * u2);
                }
            }
#pragma unroll 1
            for (int t0 = sub; t0 < W; t0 += tps) {
                const float u0 = rf.x + (float)(NS - t0);
                const float w0 = __builtin_amdgcn_exp2f(-a.coef[0] * u0 * u0);
                int r0 = l0 + t0;
                if (WRAP && r0 >= R0) r0 -= (int)a.nf[0]; // only when the region spans the whole axis
                float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int t1 = 0; t1 < W; ++t1) {
                    int r1 = l1 + t1;
                    if (WRAP && r1 >= R1) r1 -= (int)a.nf[1];
                    if (D == 3) {
                        const int rowb = (r0 * R1 + r1) * R2;
                        float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                        for (int t2 = 0; t2 < W; ++t2) {
                            int r2 = l2 + t2;
                            if (WRAP && r2 >= R2) r2 -= (int)a.nf[2];
                            fma_cell(q, w2[t2], lds_pair[rowb + r2]);
                        }
                        fma_cell(p, w1[t1], q);
                    } else {
                        fma_cell(p, w1[t1], lds_pair[r0 * R1 + r1]);
                    }
                }
                fma_cell(acc, w0, p);
            }
        }
        // every lane takes part in the exchange (a sample's lanes are in one wave)
        for (int k = 1; k < tps; ++k) {
            const int src = lane + k * stride;
            const float4 o = make_float4(__shfl(acc.x, src), __shfl(acc.y, src), __shfl(acc.z, src),
                                         __shfl(acc.w, src));
            if (sub == 0) {
                acc.x += o.x;
                acc.y += o.y;
                acc.z += o.z;
                acc.w += o.w;
            }
        }
        if (!valid || sub != 0) continue;
        if (a.scale != 1.0f) {
            acc.x *= a.scale;
            acc.y *= a.scale;
            acc.z *= a.scale;
            acc.w *= a.scale;
        }
        const float2 o0 = make_float2(acc.x, acc.y), o1 = make_float2(acc.z, acc.w);
        if (a.layout == GN_COIL_LAST) {
            float2 *o = a.out + (int64_t)orig * a.nc + cg0;
            o[0] = o0;
            if (two) o[1] = o1;
        } else {
            a.out[(int64_t)cg0 * a.M + orig] = o0;
            if (two) a.out[(int64_t)(cg0 + 1) * a.M + orig] = o1;
        }
    }
}

template <int D, int NS, bool WRAP>
__global__ __launch_bounds__(kGatherThreads) void k_gather(GatherArgs a)
{
    const uint32_t n = gridDim.x * gridDim.y;
    const uint32_t w = xcd_swizzle(blockIdx.x + gridDim.x * blockIdx.y, n);
    // coil groups fastest: a tile's coils run side by side and share its sample records in L2
    gather_body<D, NS, WRAP>(a, a.items[w / gridDim.y], (int)(w % gridDim.y));
}

// Batched launch over many plans: bitems[b] = {instance, work item, coil group, 0},
// taken in the XCD-aware order of the plain launch.
template <int D, int NS, bool WRAP>
__global__ __launch_bounds__(kGatherThreads) void k_gather_batch(const GatherArgs *__restrict__ args,
                                                                 const int4 *__restrict__ bitems)
{
    const int4 bi = bitems[xcd_swizzle(blockIdx.x, gridDim.x)];
    const GatherArgs &a = args[bi.x]; // read in place: uniform scalar loads
    gather_body<D, NS, WRAP>(a, a.items[bi.y], bi.z);
}

// ---------------------------------------------------------------------------
// Trajectory gradient: derivative of the type-2 interpolation with respect to
// the sample coordinates, contracted with per-sample complex weights:
//   out[a][j] = sum_c Re( conj(wts[j,c]) * d/dx_a (A image)[j,c] ),
// with d/dx_a w = w * gscale_a * (t + ns - tap), gscale_a = -h_a df / (2 tau),
// the analytic derivative of the Gaussian exp(-(xi - h g)^2 / (4 tau)).
// A staged cell holds a coil pair, or one coil (see traj_grad_dispatch); the window weights
// times their offsets are formed once per sample, so a cell takes 8 FMAs and one 16-byte LDS
// read per pair, where the products formed per cell took 16 to 24 and two 8-byte reads.  The
// sums run per coil and part and meet the sample's weights last: contracting the coils of a
// cell first takes 6 FMAs (256^3-grid UTE, 4 coils, 1048576 samples, nspread 3: 275 us; this
// way 308, per coil 436) but rounds before the derivative's cancellation, which made the
// error of that gradient 4 to 6 % larger.  Staging and lanes per sample as in the gather.
// Bound by the taps' LDS reads and FMAs.
// ---------------------------------------------------------------------------

// Two workgroups per CU are four waves per SIMD: at most 128 registers where their LDS allows
// two (nspread 4 took 131 without the bound: 96^3 x 4 coils 562 -> 780 us).
constexpr int traj_grad_waves(int D, int NS, bool WRAP, bool PAIR) { return !WRAP && (!PAIR || NS <= 5 || D == 2) ? 4 : 1; }

template <int D, int NS, bool WRAP, bool PAIR>
__global__ __launch_bounds__(kGatherThreads, traj_grad_waves(D, NS, WRAP, PAIR)) void k_traj_grad(GatherArgs a, const float2 *__restrict__ wts,
                                                               float *__restrict__ out, float gs0, float gs1, float gs2)
{
    using Cell = std::conditional_t<PAIR, float4, float2>;
    constexpr int W = 2 * NS, NC = PAIR ? 2 : 1; // coils of a staged cell
    extern __shared__ float4 lds_pair[];
    Cell *cells = reinterpret_cast<Cell *>(lds_pair);
    // neighbouring tiles on one XCD, as in the gather; not for the long items of wide windows,
    // whose crowded tiles would share it (64^3 radial, nspread 6, 2 coils: 300 us, in runs 327)
    constexpr bool kRuns = PAIR || NS <= 5;
    const int4 item = a.items[kRuns ? xcd_swizzle(blockIdx.x, gridDim.x) : blockIdx.x];
    int org[3] = {0, 0, 0};
    {
        uint32_t r = (uint32_t)item.x; // tile index < 2^31
        for (int ax = D - 1; ax >= 0; --ax) {
            org[ax] = (int)(r % (uint32_t)a.ntiles[ax]) * a.tile[ax];
            r /= (uint32_t)a.ntiles[ax];
        }
    }
    const int R0 = a.region[0], R1 = a.region[1], R2 = (D == 3) ? a.region[2] : 1;
    const int RC = R0 * R1 * R2;
    // several lanes per sample, as in the gather: the tps lanes of a group take the
    // leading-axis taps t0 = sub, sub + tps, ... and the group's lane 0 adds the
    // partial gradients of the others in lane order
    const int n = item.z - item.y;
    const int nwaves = kGatherThreads / 64;
    int tps = 1;
#pragma unroll
    for (int d = 2; d <= 8; ++d)
        if (W % d == 0 && n <= nwaves * (64 / d)) tps = d;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int spw = 64 / tps;
    int grp, sub, stride;
    lane_layout<NS>(lane, tps, spw, &grp, &sub, &stride);
    for (int s0 = 0; s0 < n; s0 += nwaves * spw) {
        const int slot = s0 + wave * spw + grp;
        const bool valid = grp < spw && sub < tps && slot < n;
        float g0 = 0.f, g1 = 0.f, g2 = 0.f;
        int4 rc = make_int4(0, 0, 0, 0);
        float4 rf = make_float4(0.f, 0.f, 0.f, 0.f);
        int l0 = 0, l1 = 0, l2 = 0;
        // window weights and the same times their offsets (the derivative up to gs)
        float w1[W], v1[W], w2[D == 3 ? W : 1], v2[D == 3 ? W : 1];
        if (valid) {
            rc = a.rec_cell[item.y + slot];
            rf = a.rec_frac[item.y + slot];
            l0 = rc.x - org[0];
            if (l0 < 0) l0 += (int)a.nf[0];
            l1 = rc.y - org[1];
            if (l1 < 0) l1 += (int)a.nf[1];
            if (D == 3) {
                l2 = rc.z - org[2];
                if (l2 < 0) l2 += (int)a.nf[2];
            }
        }
#pragma unroll
        for (int t = 0; t < W; ++t) {
            const float u1 = rf.y + (float)(NS - t);
            w1[t] = __builtin_amdgcn_exp2f(-a.coef[1] * u1 * u1);
            v1[t] = w1[t] * u1;
            if (D == 3) {
                const float u2 = rf.z + (float)(NS - t);
                w2[t] = __builtin_amdgcn_exp2f(-a.coef[2] * u2 * u2);
                v2[t] = w2[t] * u2;
            }
        }
        for (int64_t c0 = 0; c0 < a.nc; c0 += NC) {
            const bool two = PAIR && c0 + 1 < a.nc;
            const float2 *g = a.grid + c0 * a.G;
            float2 wa = make_float2(0.f, 0.f), wb = wa; // the pair's weights of this sample
            if (valid) {
                wa = a.layout == GN_COIL_LAST ? wts[(int64_t)rc.w * a.nc + c0] : wts[c0 * a.M + rc.w];
                if (two) wb = a.layout == GN_COIL_LAST ? wts[(int64_t)rc.w * a.nc + c0 + 1] : wts[(c0 + 1) * a.M + rc.w];
            }
            if (c0 > 0 || s0 > 0) __syncthreads(); // the previous pair's taps have been read
            if (rows_stage_ok(D == 3 ? R2 : R1, a.G))
                stage_region_rows<D>(cells, g, g + a.G, two, a.nf, org, R0, R1, R2);
            else
                stage_region_flat<D>(cells, g, g + a.G, two, a.nf, org, R1, R2, RC);
            __syncthreads();
            if (!valid) continue;
            // value and derivative sums of every coil and part; the weights come last
            Cell dx{}, dy{}, dz{};
#pragma unroll 1
            for (int t0 = sub; t0 < W; t0 += tps) {
                const float u0 = rf.x + (float)(NS - t0);
                const float w0 = __builtin_amdgcn_exp2f(-a.coef[0] * u0 * u0);
                int r0 = l0 + t0;
                if (WRAP && r0 >= R0) r0 -= (int)a.nf[0];
                Cell p{}, py{}, pz{};
#pragma unroll
                for (int t1 = 0; t1 < W; ++t1) {
                    int r1 = l1 + t1;
                    if (WRAP && r1 >= R1) r1 -= (int)a.nf[1];
                    Cell q{};
                    if constexpr (D == 3) {
                        Cell qz{};
                        const int rowb = (r0 * R1 + r1) * R2;
#pragma unroll
                        for (int t2 = 0; t2 < W; ++t2) {
                            int r2 = l2 + t2;
                            if (WRAP && r2 >= R2) r2 -= (int)a.nf[2];
                            const Cell v = cells[rowb + r2];
                            fma_cell(q, w2[t2], v);
                            fma_cell(qz, v2[t2], v);
                        }
                        fma_cell(pz, w1[t1], qz);
                    } else {
                        q = cells[r0 * R1 + r1];
                    }
                    fma_cell(p, w1[t1], q);
                    fma_cell(py, v1[t1], q);
                }
                fma_cell(dx, w0 * u0, p);
                fma_cell(dy, w0, py);
                if constexpr (D == 3) fma_cell(dz, w0, pz);
            }
            // sum over the cell's coils of Re(conj(weight) sum)
            auto contract = [&](const Cell &v) {
                float r = wa.x * v.x + wa.y * v.y;
                if constexpr (PAIR) r += wb.x * v.z + wb.y * v.w;
                return r;
            };
            g0 += contract(dx);
            g1 += contract(dy);
            if constexpr (D == 3) g2 += contract(dz);
        }
        for (int k = 1; k < tps; ++k) {
            const int src = lane + k * stride;
            const float o0 = __shfl(g0, src), o1 = __shfl(g1, src), o2 = __shfl(g2, src);
            if (sub == 0) {
                g0 += o0;
                g1 += o1;
                g2 += o2;
            }
        }
        if (valid && sub == 0) {
            out[rc.w] = g0 * gs0;
            out[a.M + rc.w] = g1 * gs1;
            if (D == 3) out[2 * a.M + rc.w] = g2 * gs2;
        }
    }
}

// ---------------------------------------------------------------------------
// Fused pre-pass (deapodize + zero-pad + coil transpose) and post-pass
// (crop + deapodize + scale + coil transpose).  Frequency k = n - m//2 sits at
// grid index k mod nf (fft/nufft_func.py:761-764, 728-729).
// ---------------------------------------------------------------------------



template <int D>
__device__ __forceinline__ void pad_body(const PrepostArgs &a, const float2 *__restrict__ img, float2 *__restrict__ grid)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t gidx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; gidx < a.G; gidx += stride) {
        int64_t i2 = 0, i1, i0;
        if (D == 3) {
            i2 = gidx % a.nf[2];
            int64_t r = gidx / a.nf[2];
            i1 = r % a.nf[1];
            i0 = r / a.nf[1];
        } else {
            i1 = gidx % a.nf[1];
            i0 = gidx / a.nf[1];
        }
        int64_t n0 = i0 + a.modes[0] / 2;
        if (n0 >= a.nf[0]) n0 -= a.nf[0];
        int64_t n1 = i1 + a.modes[1] / 2;
        if (n1 >= a.nf[1]) n1 -= a.nf[1];
        int64_t n2 = 0;
        bool inside = n0 < a.modes[0] && n1 < a.modes[1];
        if (D == 3) {
            n2 = i2 + a.modes[2] / 2;
            if (n2 >= a.nf[2]) n2 -= a.nf[2];
            inside &= n2 < a.modes[2];
        }
        if (!inside) {
            for (int64_t c = 0; c < a.nc; ++c) grid[c * a.G + gidx] = make_float2(0.f, 0.f);
            continue;
        }
        float d = a.scale * a.deap0[n0] * a.deap1[n1];
        int64_t n = n0 * a.modes[1] + n1;
        if (D == 3) {
            d *= a.deap2[n2];
            n = n * a.modes[2] + n2;
        }
        if (a.sens) { // SENSE: coil c's image is x * S_c
            const float2 x = img[n];
            for (int64_t c = 0; c < a.nc; ++c) {
                const float2 s = (a.layout == GN_COIL_LAST) ? a.sens[n * a.nc + c] : a.sens[c * a.N + n];
                const float2 v = make_float2(x.x * s.x - x.y * s.y, x.x * s.y + x.y * s.x);
                grid[c * a.G + gidx] = make_float2(v.x * d, v.y * d);
            }
            continue;
        }
        for (int64_t c = 0; c < a.nc; ++c) {
            const float2 v = (a.layout == GN_COIL_LAST) ? img[n * a.nc + c] : img[c * a.N + n];
            grid[c * a.G + gidx] = make_float2(v.x * d, v.y * d);
        }
    }
}

template <int D>
__global__ __launch_bounds__(256) void k_pad(PrepostArgs a, const float2 *__restrict__ img, float2 *__restrict__ grid)
{
    pad_body<D>(a, img, grid);
}

// batched: blockIdx.y = instance; args[i].src = image, args[i].dst = grid
template <int D>
__global__ __launch_bounds__(256) void k_pad_batch(const PrepostArgs *__restrict__ args)
{
    const PrepostArgs &a = args[blockIdx.y]; // read in place: uniform scalar loads
    pad_body<D>(a, a.src, a.dst);
}

template <int D>
__device__ __forceinline__ void crop_body(const PrepostArgs &a, const float2 *__restrict__ grid, float2 *__restrict__ img)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; n < a.N; n += stride) {
        int64_t n2 = 0, n1, n0;
        if (D == 3) {
            n2 = n % a.modes[2];
            int64_t r = n / a.modes[2];
            n1 = r % a.modes[1];
            n0 = r / a.modes[1];
        } else {
            n1 = n % a.modes[1];
            n0 = n / a.modes[1];
        }
        int64_t i0 = n0 - a.modes[0] / 2;
        if (i0 < 0) i0 += a.nf[0];
        int64_t i1 = n1 - a.modes[1] / 2;
        if (i1 < 0) i1 += a.nf[1];
        int64_t gi = i0 * a.nf[1] + i1;
        float d = a.scale * a.deap0[n0] * a.deap1[n1];
        if (D == 3) {
            int64_t i2 = n2 - a.modes[2] / 2;
            if (i2 < 0) i2 += a.nf[2];
            gi = gi * a.nf[2] + i2;
            d *= a.deap2[n2];
        }
        if (a.sens) { // SENSE: sum_c conj(S_c) * image_c, coils in order
            float2 acc = make_float2(0.f, 0.f);
            for (int64_t c = 0; c < a.nc; ++c) {
                const float2 v = grid[c * a.G + gi];
                const float2 o = make_float2(v.x * d, v.y * d);
                const float2 s = (a.layout == GN_COIL_LAST) ? a.sens[n * a.nc + c] : a.sens[c * a.N + n];
                acc.x += s.x * o.x + s.y * o.y;
                acc.y += s.x * o.y - s.y * o.x;
            }
            img[n] = acc;
            continue;
        }
        for (int64_t c = 0; c < a.nc; ++c) {
            const float2 v = grid[c * a.G + gi];
            const float2 o = make_float2(v.x * d, v.y * d);
            if (a.layout == GN_COIL_LAST)
                img[n * a.nc + c] = o;
            else
                img[c * a.N + n] = o;
        }
    }
}

template <int D>
__global__ __launch_bounds__(256) void k_crop(PrepostArgs a, const float2 *__restrict__ grid, float2 *__restrict__ img)
{
    crop_body<D>(a, grid, img);
}

// batched: blockIdx.y = instance; args[i].src = grid, args[i].dst = image
template <int D>
__global__ __launch_bounds__(256) void k_crop_batch(const PrepostArgs *__restrict__ args)
{
    const PrepostArgs &a = args[blockIdx.y]; // read in place: uniform scalar loads
    crop_body<D>(a, a.src, a.dst);
}

inline int grid_blocks(int64_t n, int threads, int64_t cap = 1 << 20)
{
    int64_t b = (n + threads - 1) / threads;
    if (b < 1) b = 1;
    return (int)std::min<int64_t>(b, cap);
}

template <typename T>
int dev_alloc(T **p, size_t count, const char *what)
{
    if (*p) {
        (void)hipFree(*p);
        *p = nullptr;
    }
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void **)p, count * sizeof(T));
    if (e != hipSuccess) {
        *p = nullptr;
        return fail(GN_ENOMEM, std::string("hipMalloc failed for ") + what);
    }
    return GN_OK;
}

// Device scratch of set_points: one pool per device, shared by every plan, that only
// grows.  A set_points call holds the pool (its lock) until its last use of the
// scratch has completed on its stream, so plans on other streams and threads never
// see each other's buffers; buffers are requested in the same order on every call,
// and buffer k of a call reuses buffer k of the previous one.
struct ScratchPool {
    std::mutex mu;
    std::vector<void *> ptr;
    std::vector<size_t> cap;
    int *ticket = nullptr; // of the scans, zero between them
    int *ret = nullptr;    // pinned: values the scans return to the host (kRet*)
    int init()
    {
        if (!ticket) {
            int *t = nullptr;
            if (hipMalloc((void **)&t, sizeof(int)) != hipSuccess) return fail(GN_ENOMEM, "hipMalloc failed for the scans");
            const int zero = 0;
            hipError_t e = hipMemcpy(t, &zero, sizeof(int), hipMemcpyHostToDevice);
            if (e != hipSuccess) {
                (void)hipFree(t);
                return hip_fail(e, "scan ticket");
            }
            ticket = t;
        }
        if (!ret && hipHostMalloc((void **)&ret, 16 * sizeof(int)) != hipSuccess) {
            ret = nullptr;
            return fail(GN_ENOMEM, "hipHostMalloc failed for the scan results");
        }
        return GN_OK;
    }
};
enum { kSpreadValu = 0, kSpreadMfma = 1, kSpreadTile = 2, kSpreadSub = 3 }; // SpreadShape::kind
enum { kRetPairs = 0, kRetErr = 2, kRetSpread = 4, kRetGather = 8 };

ScratchPool &scratch_pool()
{
    static std::mutex mu;
    static std::map<int, ScratchPool *> pools;
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> g(mu);
    ScratchPool *&p = pools[dev];
    if (!p) p = new ScratchPool(); // lives until the process ends
    return *p;
}

struct Scratch {
    ScratchPool &pool;
    std::unique_lock<std::mutex> lock;
    hipStream_t stream;
    size_t next = 0;
    explicit Scratch(hipStream_t st) : pool(scratch_pool()), lock(pool.mu), stream(st) {}
    // also on early returns: nothing queued may still use the pool once it is released
    ~Scratch() { (void)hipStreamSynchronize(stream); }
    template <typename T>
    int alloc(T **p, size_t count, const char *what)
    {
        const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
        const size_t k = next++;
        if (k >= pool.ptr.size()) {
            pool.ptr.push_back(nullptr);
            pool.cap.push_back(0);
        }
        if (pool.cap[k] < bytes) {
            if (pool.ptr[k]) (void)hipFree(pool.ptr[k]); // waits for the device
            pool.ptr[k] = nullptr;
            pool.cap[k] = 0;
            const size_t want = bytes + bytes / 4;      // headroom for slightly larger calls
            if (hipMalloc(&pool.ptr[k], want) != hipSuccess) {
                pool.ptr[k] = nullptr;
                *p = nullptr;
                return fail(GN_ENOMEM, std::string("hipMalloc failed for ") + what);
            }
            pool.cap[k] = want;
        }
        *p = (T *)pool.ptr[k];
        return GN_OK;
    }
};

// A buffer owned by the plan that only grows (count elements of T, at least one).
template <typename T>
int grow_alloc(T **p, int64_t *cap, size_t count, const char *what)
{
    count = std::max<size_t>(count, 1);
    if (*p && (size_t)*cap >= count) return GN_OK;
    int rc = dev_alloc(p, count, what);
    *cap = rc ? 0 : (int64_t)count;
    return rc;
}

// Exclusive scan of n ints (see k_scan); bsum: n / kScanTile + 2 ints.
hipError_t device_scan(int *data, int64_t n, int *bsum, Scratch &sc)
{
    const int64_t nb = std::max<int64_t>(1, (n + kScanTile - 1) / kScanTile);
    hipLaunchKernelGGL(k_scan, dim3((unsigned)nb), dim3(kScanThreads), 0, sc.stream, data, n, bsum, sc.pool.ticket);
    return hipGetLastError();
}

// Stable counting sort of n items by keys[i*stride] in [0,K): writes the sorted values
// (vals, or the item indices where it is null); *skeys: the sorted keys (scratch).  Asynchronous on st; the temporary buffers
// belong to sc, which the caller keeps alive until the stream has consumed them.
int stable_sort_by_key(int64_t n, const int *keys, int stride, const int *vals, int64_t K, int *sorted,
                       const int **skeys, hipStream_t st, Scratch &sc)
{
    int rc;
    int kbits = 1;
    while (kbits < 31 && ((int64_t)1 << kbits) < K) ++kbits;
    const int npass = (kbits + kRadixBits - 1) / kRadixBits, pbits = (kbits + npass - 1) / npass;
    // chunks: about 4096 waves over the GPU, 256..4096 items each (below 256 the count
    // array outgrows the items: 98304 spiral samples 176 us with 64, 150 with 128, 145 with
    // 256; 2048 or 8192 waves 3-8 % more time on 1 M samples)
    int64_t wave_len = (n + 4095) / 4096;
    wave_len = std::min<int64_t>(4096, std::max<int64_t>(256, ((wave_len + 63) / 64) * 64));
    const int64_t chunk_len = kRadixWaves * wave_len;
    const int64_t C = std::max<int64_t>(1, (n + chunk_len - 1) / chunk_len);
    const int64_t nKC = ((int64_t)1 << pbits) * C;
    int *cnt = nullptr, *bsum = nullptr, *k0 = nullptr, *v0 = nullptr, *k1 = nullptr, *v1 = nullptr;
    if ((rc = sc.alloc(&cnt, (size_t)nKC, "sort counts")) ||
        (rc = sc.alloc(&bsum, (size_t)(nKC / kScanTile) + 2, "sort scan")) ||
        (rc = sc.alloc(&k0, (size_t)n, "sort keys")) || (rc = sc.alloc(&k1, (size_t)n, "sort keys")) ||
        (rc = sc.alloc(&v0, (size_t)n, "sort values")))
        return rc;
    v1 = sorted;
    const int *kin = keys;
    const int *vin = vals;
    int kstride = stride;
    // ping-pong so that the last pass writes its values into `sorted`
    int *kout[2] = {k0, k1};
    int *vout[2] = {v0, v1};
    int shift = 0;
    hipError_t e = hipSuccess;
    for (int ps = 0; ps < npass && e == hipSuccess; ++ps) {
        const int bits = std::min(pbits, kbits - shift);
        const int bins = 1 << bits;
        const int o = (npass - 1 - ps) % 2 == 0 ? 1 : 0; // the last pass writes slot 1 (sorted)
        const size_t lds = (size_t)bins * sizeof(int);
        hipLaunchKernelGGL(k_radix_count, dim3((unsigned)C), dim3(64 * kRadixWaves), lds, st, n, kin, kstride, shift, bins,
                           chunk_len, (int)C, cnt);
        e = hipGetLastError();
        if (e == hipSuccess) e = device_scan(cnt, (int64_t)bins * C, bsum, sc);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_radix_scatter, dim3((unsigned)C), dim3(64 * kRadixWaves), kRadixWaves * lds, st, n, kin, kstride, vin,
                               shift, bits, chunk_len, (int)C, cnt, bsum, kout[o], vout[o]);
            e = hipGetLastError();
        }
        kin = kout[o];
        vin = vout[o];
        kstride = 1;
        shift += bits;
    }
    if (e != hipSuccess) return hip_fail(e, "stable sort");
    *skeys = kin;
    return GN_OK;
}

} // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

void default_tiles(int dim, int ns, const int64_t *nf, int *tile, int *gtile)
{
    host::default_tiles(dim, ns, nf, tile, gtile);
}

// Orders the records of one gather work item for conflict-free LDS reads in the
// gather.  Every tap adds the same offset to all lanes' staged-cell addresses, so if
// the lanes of each group of 16 start at cells of distinct residues mod 16 (the
// 16-byte cells map to 16 disjoint groups of four LDS banks), every tap of that group
// is free of bank conflicts.  Samples are placed by (rank within their residue class,
// residue): position = sum_v min(size_v, k) + #{v < r : size_v > k} for rank k and
// residue r.  Ranks are taken in record order with wave ballots, so the permutation is
// deterministic.  Each sample's result does not depend on its lane.
static_assert(kGatherChunk <= kGatherThreads, "one record per thread in the bank ordering");

template <int D>
__global__ __launch_bounds__(kGatherThreads) void k_bank_order(GatherArgs a, int4 *cell, float4 *frac)
{
    constexpr int kWaves = kGatherThreads / 64;
    __shared__ int s_cnt[kWaves][16];
    __shared__ int s_sz[16];
    const int4 item = a.items[blockIdx.x];
    const int n = item.z - item.y;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int org[3] = {0, 0, 0};
    {
        uint32_t r = (uint32_t)item.x; // tile index < 2^31
        for (int ax = D - 1; ax >= 0; --ax) {
            org[ax] = (int)(r % (uint32_t)a.ntiles[ax]) * a.tile[ax];
            r /= (uint32_t)a.ntiles[ax];
        }
    }
    int4 rc = make_int4(0, 0, 0, 0);
    float4 rf = make_float4(0.f, 0.f, 0.f, 0.f);
    int res = 16; // no sample
    if (tid < n) {
        rc = cell[item.y + tid];
        rf = frac[item.y + tid];
        int l0 = rc.x - org[0];
        if (l0 < 0) l0 += (int)a.nf[0];
        int l1 = rc.y - org[1];
        if (l1 < 0) l1 += (int)a.nf[1];
        int addr = l0 * a.region[1] + l1;
        if (D == 3) {
            int l2 = rc.z - org[2];
            if (l2 < 0) l2 += (int)a.nf[2];
            addr = addr * a.region[2] + l2;
        }
        res = addr & 15;
    }
    int rank = 0;
    for (int v = 0; v < 16; ++v) {
        const unsigned long long m = __ballot(res == v);
        if (res == v) rank = __popcll(m & ((1ull << lane) - 1ull));
        if (lane == 0) s_cnt[wave][v] = __popcll(m);
    }
    __syncthreads();
    if (tid < 16) {
        int sum = 0;
        for (int w = 0; w < kWaves; ++w) {
            const int c = s_cnt[w][tid];
            s_cnt[w][tid] = sum;
            sum += c;
        }
        s_sz[tid] = sum;
    }
    __syncthreads();
    if (tid < n) {
        const int k = s_cnt[wave][res] + rank;
        int pos = 0;
        for (int v = 0; v < 16; ++v) {
            const int sz = s_sz[v];
            pos += min(sz, k) + ((v < res && sz > k) ? 1 : 0);
        }
        cell[item.y + pos] = rc; // every record of the item was read before the barriers
        frac[item.y + pos] = rf;
    }
}

#define GN_HIP(call)                                                                                                   \
    do {                                                                                                               \
        hipError_t e_ = (call);                                                                                        \
        if (e_ != hipSuccess) return hip_fail(e_, #call);                                                              \
    } while (0)

// Pairs per spread work item, at most kSpreadChunk.  A launch lasts as long as its longest
// item, eight batches of 64 at kSpreadChunk, so smaller spreads take shorter items; the
// partial tiles cost more than that saves once the items fill the chip many times over.
// Items of 512 / 192 / 128 pairs: 43 k pairs (192^2, 8 coils) 36 / 24 / 22 us, 209 k pairs
// (256^2 spiral, 8 coils) 50 / 36 / 38 us, 1.1 M pairs (64^3, 4 coils) 107 / 83 / 82 us,
// 2.9 M pairs (64^3, 8 coils) 202 / 225 / 268 us.  The pairs count once per coil group, and
// in a batch with those of the other instances: 4 instances of 48^3 x 8 coils, 0.8 M pairs
// each, type 1 451 / 482 us (512 / 192), 2 of 64^3 with 1 M 391 / 409.
// Samples spread evenly have the same pairs in every tile: an item a little shorter than
// that would split all of them, so with enough tiles it is 1.5 times the mean (type 1,
// 48^3, 246 k samples, 293 pairs a tile, 8 coils 159 / 239 us (512 / 192), 32 coils 549 /
// 876; 512^2 x 32, 213 pairs a tile, 724 / 1004).  The one-wave kernel in 2-D has items
// enough from 4096 tiles on (128^2, 1 coil, 426 pairs in each of 512 tiles: 37 / 30 us).
int spread_chunk(const gn_plan_s *p, int64_t pairs)
{
    static_assert(kSpreadChunk >= 192, "shorter items than the longest");
    const SpreadShape sh = spread_shape(make_spread_args(p, nullptr, 0), p->geo.dim);
    const double sets = (double)((p->nc + sh.coils - 1) / sh.coils) * p->launch_share;
    const double work = (double)pairs * sets;
    const int chunk = work >= (7 << 18) ? kSpreadChunk : work >= (1 << 17) ? 192 : 128;
    if ((double)p->geo.K * sets < (sh.kind == kSpreadTile && p->geo.dim == 2 ? 4096 : 512)) return chunk;
    const int64_t even = (3 * pairs / (2 * p->geo.K) + 63) / 64 * 64;
    return (int)std::min<int64_t>(kSpreadChunk, std::max<int64_t>(chunk, even));
}

int bin_and_sort(gn_plan_s *p, int64_t M, const void *x, const void *y, const void *z, int coord_f64, double df,
                 const float *dcf)
{
    Geometry &g = p->geo;
    Records &R = p->rec;
    hipStream_t st = p->stream;
    const int64_t K = g.K, Kg = g.Kg;
    int rc;
    if (M > R.cap) {
        if ((rc = dev_alloc(&R.cell, (size_t)M, "records")) || (rc = dev_alloc(&R.frac, (size_t)M, "records")))
            return rc;
        R.cap = M;
    }
    if ((rc = grow_alloc(&R.bin_start, &R.bin_start_cap, (size_t)Kg + 1, "bin offsets"))) return rc;
    R.npairs = 0;

    Scratch sc(st);
    if ((rc = sc.pool.init())) return rc;
    int *ticket = sc.pool.ticket;
    volatile int *ret = sc.pool.ret;
    int *tile_pairs = nullptr; // K + 1 offsets of each spread tile's pairs (scratch)
    if ((rc = sc.alloc(&tile_pairs, (size_t)K + 1, "pairs"))) return rc;

    if (M > 0) {
        int4 *cell = nullptr;
        float4 *frac = nullptr;
        int *sorted = nullptr;
        const int *skeys = nullptr;
        if ((rc = sc.alloc(&cell, (size_t)M, "sort scratch")) || (rc = sc.alloc(&frac, (size_t)M, "sort scratch")) ||
            (rc = sc.alloc(&sorted, (size_t)M, "sort scratch")))
            return rc;
        PrepArgs pa;
        pa.M = M;
        pa.x[0] = x;
        pa.x[1] = y;
        pa.x[2] = z;
        pa.coord_f64 = coord_f64;
        pa.df = df;
        pa.dim = g.dim;
        for (int a = 0; a < 3; ++a) {
            pa.nf[a] = g.nf[a];
            pa.tile[a] = g.gtile[a];
            pa.ntiles[a] = g.ngtiles[a];
        }
        pa.ns = g.ns;
        pa.cell = cell;
        pa.frac = frac;
        pa.err = p->err_flag;
        pa.seq = p->points_seq = p->points_seq == INT32_MAX ? 1 : p->points_seq + 1;
        hipLaunchKernelGGL(k_prep, dim3(grid_blocks(M, 256, INT32_MAX)), dim3(256), 0, st, pa);
        GN_HIP(hipGetLastError());
        // gather-tile sort (stable) -> records in tile order
        if ((rc = stable_sort_by_key(M, &cell[0].w, 4, nullptr, Kg, sorted, &skeys, st, sc))) return rc;
        hipLaunchKernelGGL(k_make_records, dim3(grid_blocks(M + 1, 256, INT32_MAX)), dim3(256), 0, st, M, sorted, cell,
                           frac, dcf, skeys, Kg, R.bin_start, R.cell, R.frac);
        GN_HIP(hipGetLastError());

        // (spread tile, sample) pairs: keys in record order, sorted by tile, records rebuilt in tile order
        TileGeom tg;
        tg.dim = g.dim;
        for (int a = 0; a < 3; ++a) {
            tg.nf[a] = g.nf[a];
            tg.tile[a] = g.tile[a];
            tg.ntiles[a] = g.ntiles[a];
        }
        tg.W = 2 * g.ns;
        int *pcnt = nullptr, *pbsum = nullptr;
        const int64_t nbp = (M + kScanTile - 1) / kScanTile;
        if ((rc = sc.alloc(&pcnt, (size_t)M, "pair counts")) || (rc = sc.alloc(&pbsum, (size_t)nbp + 1, "pair scan")))
            return rc;
        // one host round trip returns the pair total and the coordinate error flag
        hipLaunchKernelGGL(k_pair_scan, dim3((unsigned)nbp), dim3(kScanThreads), 0, st, M, R.cell, tg, pcnt, pbsum,
                           ticket, sc.pool.ret + kRetPairs, p->err_flag);
        GN_HIP(hipGetLastError());
        GN_HIP(hipStreamSynchronize(st));
        if (ret[kRetErr] == p->points_seq) return fail(GN_EINVAL, "non-finite sample coordinate");
        const int64_t P = host::scan_total(ret[kRetPairs], ret[kRetPairs + 1]);
        if (P > (int64_t)INT32_MAX) return fail(GN_EINVAL, "too many (tile, sample) pairs");
        int *pkey = nullptr, *psamp = nullptr, *psorted = nullptr;
        if ((rc = sc.alloc(&pkey, (size_t)P, "pairs")) || (rc = sc.alloc(&psamp, (size_t)P, "pairs")) ||
            (rc = sc.alloc(&psorted, (size_t)P, "pairs")))
            return rc;
        hipLaunchKernelGGL(k_pair_keys, dim3(grid_blocks(M, 256, INT32_MAX)), dim3(256), 0, st, M, R.cell, tg, pcnt,
                           pbsum, pkey, psamp);
        GN_HIP(hipGetLastError());
        if ((rc = stable_sort_by_key(P, pkey, 1, psamp, K, psorted, &skeys, st, sc))) return rc;
        if (P > R.pairs_cap) {
            if ((rc = dev_alloc(&R.pair_a, (size_t)P, "pairs")) || (rc = dev_alloc(&R.pair_b, (size_t)P, "pairs")))
                return rc;
            R.pairs_cap = P;
        }
        hipLaunchKernelGGL(k_pair_records, dim3(grid_blocks(P + 1, 256, INT32_MAX)), dim3(256), 0, st, P, psorted,
                           skeys, K, tile_pairs, R.cell, R.frac, tg, R.pair_a, R.pair_b);
        GN_HIP(hipGetLastError());
        R.npairs = P;
    } else {
        GN_HIP(hipMemsetAsync(R.bin_start, 0, sizeof(int) * (Kg + 1), st));
        GN_HIP(hipMemsetAsync(tile_pairs, 0, sizeof(int) * (K + 1), st));
    }

    // spread work items, partial slots, reduce items, occupancy masks (the spread leaves
    // tiles without pairs unwritten where the first adjoint FFT pass skips them) and gather
    // work items on the device; their counts come back in one synchronisation
    {
        const int64_t P = R.npairs;
        const int chunk = spread_chunk(p, P);
        const int64_t cap_items = K + P / chunk + 1, cap_red = std::min<int64_t>(K, P / chunk + 1);
        const int64_t ncolt = (int64_t)g.ntiles[1] * g.ntiles[2];
        if ((rc = grow_alloc(&R.spread_items, &R.spread_items_cap, (size_t)cap_items, "work items")) ||
            (rc = grow_alloc(&R.reduce_items, &R.reduce_items_cap, (size_t)cap_red, "work items")) ||
            (rc = grow_alloc(&R.gather_items, &R.gather_items_cap, (size_t)(Kg + M / kGatherChunk + 1), "work items")) ||
            (rc = grow_alloc(&R.occ_mask, &R.occ_mask_cap, (size_t)ncolt, "tile masks")))
            return rc;
        auto items = [&](int64_t n, const int *start, int len, int ret_at, int4 *out, int4 *reduce) -> int {
            const int64_t nb = (n + kItemTile - 1) / kItemTile;
            int4 *off = nullptr, *bs = nullptr;
            int r;
            if ((r = sc.alloc(&off, (size_t)n, "work items")) || (r = sc.alloc(&bs, (size_t)nb + 1, "work items")))
                return r;
            hipLaunchKernelGGL(k_item_scan, dim3((unsigned)nb), dim3(kScanThreads), 0, st, n, start, len, off, (int *)bs,
                               ticket, sc.pool.ret + ret_at);
            GN_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_item_write, dim3(grid_blocks(n, 256, INT32_MAX)), dim3(256), 0, st, n, start, len, off,
                               bs, nb, out, reduce);
            GN_HIP(hipGetLastError());
            return GN_OK;
        };
        if ((rc = items(K, tile_pairs, chunk, kRetSpread, R.spread_items, R.reduce_items)) ||
            (rc = items(Kg, R.bin_start, kGatherChunk, kRetGather, R.gather_items, nullptr)))
            return rc;
        R.mask_k = (g.ntiles[0] + 63) / 64;
        hipLaunchKernelGGL(k_occ_masks, dim3(grid_blocks(ncolt, 4)), dim3(256), 0, st, ncolt, g.ntiles[0],
                           R.mask_k, tile_pairs, R.occ_mask);
        GN_HIP(hipGetLastError());
        GN_HIP(hipStreamSynchronize(st));
    }
    R.n_spread_full = ret[kRetSpread];
    R.n_spread_items = ret[kRetSpread] + ret[kRetSpread + 1];
    R.n_slots = ret[kRetSpread + 2];
    R.n_reduce_items = ret[kRetSpread + 3];
    R.n_gather_items = ret[kRetGather];
    const int slots = R.n_slots;
    if (R.n_gather_items > 0) {
        const GatherArgs ga = make_gather_args(p, nullptr);
        if (g.dim == 3)
            hipLaunchKernelGGL(k_bank_order<3>, dim3((unsigned)R.n_gather_items), dim3(kGatherThreads), 0, st, ga,
                               R.cell, R.frac);
        else
            hipLaunchKernelGGL(k_bank_order<2>, dim3((unsigned)R.n_gather_items), dim3(kGatherThreads), 0, st, ga,
                               R.cell, R.frac);
        GN_HIP(hipGetLastError());
    }
    const int64_t TC = (int64_t)g.tile[0] * g.tile[1] * g.tile[2];
    const int64_t need = (int64_t)slots * p->nc * TC;
    if (need > R.partial_cap) {
        if ((rc = dev_alloc(&R.partial, (size_t)need, "partial tiles"))) return rc;
        R.partial_cap = need;
    }
    return GN_OK;
}

namespace {

// Raise the dynamic-LDS limit only for launches that need more than the default 64 KiB.
template <typename K>
void lds_limit(K kernel, size_t lds)
{
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

#ifndef GN_SPREAD_MFMA
#define GN_SPREAD_MFMA 1
#endif
// The matrix-core spread covers whole 64-cell blocks: tiles must be multiples of the
// block (4 per axis in 3-D, 8 in 2-D) of at most kSpreadWavesMax blocks, so that one
// workgroup holds the whole tile.
bool mfma_tiles_ok(const SpreadArgs &a, int dim)
{
    if (!GN_SPREAD_MFMA) return false;
    const int q = dim == 3 ? 4 : 8;
    int nb = 1;
    for (int ax = 0; ax < dim; ++ax) {
        if (a.blk[ax] != q || a.tile[ax] % q != 0) return false;
        nb *= a.tile[ax] / q;
    }
    // phase 2 maps one table column per thread: 64 * waves >= TT rounded up to a power of 2
    const int ttp = a.TT <= 16 ? 16 : a.TT <= 32 ? 32 : a.TT <= 64 ? 64 : 128;
    const int waves = std::min(nb, kSpreadWavesMax);
    // one workgroup per (tile, coil group): it writes the whole tile from its LDS
    return nb <= kSpreadWavesMax && a.TT <= 128 && 64 * waves >= ttp && spread_mfma_lds_bytes(a, waves) <= 160 * 1024;
}

inline size_t spread_lds_bytes(const SpreadArgs &a, int ncg)
{
    return (size_t)kSpreadBatch * a.TT * 4 + (size_t)kSpreadBatch * ncg * 8 + (size_t)kSpreadBatch * 16 +
           (size_t)kSpreadBatch * 32;
}

// the dispatch-order arithmetic of the spread and gather kernels is 32-bit
inline bool grid_ok(dim3 g) { return (uint64_t)g.x * g.y * g.z < (1ull << 31); }

} // namespace

// Kernel and launch shape of a spread.  Default tiles: k_spread_tile for up to 2 coils in
// 2-D and 4 in 3-D (3 coil-major), k_spread_sub for more in 2-D.  3-D with more, and other
// block-aligned tiles, take k_spread_mfma (128^3, 1,048,576 samples, nspread 3: 4 coils
// 499 -> 459 us with k_spread_tile, but 8 coils 571 -> 763 us: its products fill the
// matrix cores without skipping half tiles).  Any other tile takes k_spread.
SpreadShape spread_shape(const SpreadArgs &a, int dim)
{
    SpreadShape s;
    const bool tile = dim == 3 ? a.tile[0] == 4 && a.tile[1] == 4 && a.tile[2] == 8 : a.tile[0] == 8 && a.tile[1] == 16;
    if (tile && dim == 2 && a.nc > 2 && mfma_tiles_ok(a, dim)) {
        s.kind = kSpreadSub;
        // 16 coils per workgroup (32 took 132 registers: 96 -> 82 us at 32 coils); 8 of coil-major
        // samples, each value of which is a cache line of its own, so that a launch's lines stay
        // cached (type 1, uniform samples, 8 x 8 blocks / 16 coils / 8: 320^2 x 32, 158 k, nspread
        // 5 300 / 367 / 300 us; 192^2 x 31, 76 k radial, nspread 3 138 / 131 / 111)
        s.width = a.nc <= 8 || a.layout != GN_COIL_LAST ? 1 : 2;
        s.waves = kSpreadSubWaves;
        s.coils = 8 * s.width;
        s.lds = spread_sub_lds(s.width);
        return s;
    }
    // coil-major samples of 4 coils: a value is a cache line of its own, waited for by one wave
    // (type 1 of 32^3, 117 k uniform samples, nspread 3: k_spread_mfma 87 us, k_spread_tile 95)
    if (tile && (a.nc < 4 || (a.nc == 4 && a.layout == GN_COIL_LAST)) && mfma_tiles_ok(a, dim)) {
        s.kind = kSpreadTile;
        s.width = a.nc == 1 ? 2 : a.nc == 2 ? 4 : 8;
        s.coils = s.width / 2;
        s.lds = spread_tile_lds(dim, s.width);
        return s;
    }
    s.coils = s.width = spread_coil_group(a.nc);
    const int nb = a.nblk[0] * a.nblk[1] * (dim == 3 ? a.nblk[2] : 1);
    s.waves = std::min(nb, kSpreadWavesMax);
    s.nbg = (nb + s.waves - 1) / s.waves;
    s.kind = mfma_tiles_ok(a, dim) ? kSpreadMfma : kSpreadValu;
    s.lds = s.kind == kSpreadMfma ? spread_mfma_lds_bytes(a, s.waves) : spread_lds_bytes(a, s.width);
    return s;
}

namespace {

// f(first, count) over n work items in parts that one launch takes: fewer than 2^32 threads,
// and with `rest` blocks per item fewer than 2^31 blocks (the dispatch order is 32-bit).
template <typename F>
hipError_t item_parts(int n, int threads, int64_t rest, F f)
{
    const int64_t most = std::min((((int64_t)1 << 32) - 1) / threads, (((int64_t)1 << 31) - 1) / rest);
    if (most < 1) return hipErrorInvalidConfiguration;
    hipError_t e = hipSuccess;
    for (int64_t o = 0; o < n && e == hipSuccess; o += most) e = f(o, (unsigned)std::min(most, n - o));
    return e;
}

template <typename K>
hipError_t spread_go(K kernel, int nitems, int64_t ng, const SpreadShape &sh, const SpreadArgs &a, hipStream_t st)
{
    lds_limit(kernel, sh.lds);
    return item_parts(nitems, 64 * sh.waves, ng * sh.nbg, [&](int64_t o, unsigned n) {
        SpreadArgs part = a;
        part.items += o;
        hipLaunchKernelGGL(kernel, dim3(n, (unsigned)ng, (unsigned)sh.nbg), dim3(64 * sh.waves), sh.lds, st, part);
        return hipGetLastError();
    });
}

template <int D>
hipError_t spread_dispatch(const SpreadArgs &a, int nitems, int nritems, const int4 *ritems, int64_t nc,
                           hipStream_t st)
{
    const SpreadShape sh = spread_shape(a, D);
    const int64_t ng = (nc + sh.coils - 1) / sh.coils;
    hipError_t e = hipSuccess;
    if (nitems > 0) {
        switch (sh.kind * 16 + sh.width) {
        case kSpreadSub * 16 + 1: e = spread_go(k_spread_sub<1>, nitems, ng, sh, a, st); break;
        case kSpreadSub * 16 + 2: e = spread_go(k_spread_sub<2>, nitems, ng, sh, a, st); break;
        case kSpreadTile * 16 + 8: e = spread_go(k_spread_tile<3, 8>, nitems, ng, sh, a, st); break; // 3-D only
        case kSpreadTile * 16 + 4: e = spread_go(k_spread_tile<D, 4>, nitems, ng, sh, a, st); break;
        case kSpreadTile * 16 + 2: e = spread_go(k_spread_tile<D, 2>, nitems, ng, sh, a, st); break;
        case kSpreadMfma * 16 + 8: e = spread_go(k_spread_mfma<D, 8>, nitems, ng, sh, a, st); break;
        case kSpreadMfma * 16 + 4: e = spread_go(k_spread_mfma<D, 4>, nitems, ng, sh, a, st); break;
        case kSpreadMfma * 16 + 2: e = spread_go(k_spread_mfma<D, 2>, nitems, ng, sh, a, st); break;
        case kSpreadMfma * 16 + 1: e = spread_go(k_spread_mfma<D, 1>, nitems, ng, sh, a, st); break;
        case kSpreadValu * 16 + 8: e = spread_go(k_spread<D, 8>, nitems, ng, sh, a, st); break;
        case kSpreadValu * 16 + 4: e = spread_go(k_spread<D, 4>, nitems, ng, sh, a, st); break;
        case kSpreadValu * 16 + 2: e = spread_go(k_spread<D, 2>, nitems, ng, sh, a, st); break;
        case kSpreadValu * 16 + 1: e = spread_go(k_spread<D, 1>, nitems, ng, sh, a, st); break;
        default: return hipErrorInvalidValue;
        }
    }
    if (e == hipSuccess && nritems > 0) {
        // several blocks per tile while the tiles are few (48^3, every tile split, 32 coils, type
        // 1: 1103 us with 16 blocks each, 1055 with 4)
        const int64_t want = std::max<int64_t>(4, std::min<int64_t>(kReduceBlocks, 8192 / nritems));
        const int64_t nb = std::min<int64_t>(want, (a.TC * nc + kReduceThreads - 1) / kReduceThreads);
        hipLaunchKernelGGL(k_spread_reduce<D>, dim3((unsigned)nritems, (unsigned)nb), dim3(kReduceThreads), 0, st, a,
                           ritems);
        e = hipGetLastError();
    }
    return e;
}

template <int D, int NS>
hipError_t gather_dispatch(const GatherArgs &a, int nitems, int64_t nc, hipStream_t st)
{
    const size_t lds = (size_t)a.region[0] * a.region[1] * (D == 3 ? a.region[2] : 1) * kGatherCellBytes;
    bool wrap = false;
    for (int ax = 0; ax < D; ++ax) wrap |= a.region[ax] >= a.nf[ax];
    dim3 grid((unsigned)nitems, (unsigned)((nc + kGatherCoils - 1) / kGatherCoils));
    if (!grid_ok(grid)) return hipErrorInvalidConfiguration;
    if (wrap) {
        lds_limit(k_gather<D, NS, true>, lds);
        hipLaunchKernelGGL((k_gather<D, NS, true>), grid, dim3(kGatherThreads), lds, st, a);
    } else {
        lds_limit(k_gather<D, NS, false>, lds);
        hipLaunchKernelGGL((k_gather<D, NS, false>), grid, dim3(kGatherThreads), lds, st, a);
    }
    return hipGetLastError();
}

#define GN_NS_CASES(D, FN, ...)                                                                                        \
    switch (ns) {                                                                                                      \
    case 2: return FN<D, 2>(__VA_ARGS__);                                                                              \
    case 3: return FN<D, 3>(__VA_ARGS__);                                                                              \
    case 4: return FN<D, 4>(__VA_ARGS__);                                                                              \
    case 5: return FN<D, 5>(__VA_ARGS__);                                                                              \
    case 6: return FN<D, 6>(__VA_ARGS__);                                                                              \
    case 7: return FN<D, 7>(__VA_ARGS__);                                                                              \
    case 8: return FN<D, 8>(__VA_ARGS__);                                                                              \
    default: break;                                                                                                    \
    }

#define GN_NS_CASES_2D_EXTRA(FN, ...)                                                                                  \
    switch (ns) {                                                                                                      \
    case 9: return FN<2, 9>(__VA_ARGS__);                                                                              \
    case 10: return FN<2, 10>(__VA_ARGS__);                                                                            \
    case 11: return FN<2, 11>(__VA_ARGS__);                                                                            \
    case 12: return FN<2, 12>(__VA_ARGS__);                                                                            \
    case 13: return FN<2, 13>(__VA_ARGS__);                                                                            \
    case 14: return FN<2, 14>(__VA_ARGS__);                                                                            \
    case 15: return FN<2, 15>(__VA_ARGS__);                                                                            \
    case 16: return FN<2, 16>(__VA_ARGS__);                                                                            \
    default: break;                                                                                                    \
    }

hipError_t spread_any(int dim, int ns, const SpreadArgs &a, int nitems, int nritems, const int4 *ritems, int64_t nc,
                      hipStream_t st)
{
    (void)ns;
    if (dim == 3) return spread_dispatch<3>(a, nitems, nritems, ritems, nc, st);
    return spread_dispatch<2>(a, nitems, nritems, ritems, nc, st);
}

hipError_t gather_any(int dim, int ns, const GatherArgs &a, int nitems, int64_t nc, hipStream_t st)
{
    if (dim == 3) {
        GN_NS_CASES(3, gather_dispatch, a, nitems, nc, st)
    } else {
        GN_NS_CASES(2, gather_dispatch, a, nitems, nc, st)
        GN_NS_CASES_2D_EXTRA(gather_dispatch, a, nitems, nc, st)
    }
    return hipErrorInvalidValue;
}

PrepostArgs make_prepost_impl(const gn_plan_s *p, float scale)
{
    const Geometry &g = p->geo;
    PrepostArgs a;
    a.dim = g.dim;
    for (int ax = 0; ax < 3; ++ax) {
        a.modes[ax] = g.modes[ax];
        a.nf[ax] = g.nf[ax];
    }
    a.G = g.G;
    a.N = g.N;
    a.nc = p->nc;
    a.layout = p->layout;
    a.scale = scale;
    a.deap0 = p->deap;
    a.deap1 = p->deap + g.modes[0];
    a.deap2 = p->deap + g.modes[0] + g.modes[1];
    a.src = nullptr;
    a.dst = nullptr;
    return a;
}

} // namespace

SpreadArgs make_spread_args(const gn_plan_s *p, const float2 *samples, int use_dcf)
{
    const Geometry &g = p->geo;
    SpreadArgs a;
    for (int ax = 0; ax < 3; ++ax) {
        a.nf[ax] = g.nf[ax];
        a.tile[ax] = g.tile[ax];
        a.ntiles[ax] = g.ntiles[ax];
        a.coef[ax] = g.coef[ax];
    }
    for (int ax = 0; ax < 3; ++ax) {
        a.blk[ax] = ax < g.dim ? (g.dim == 3 ? 4 : 8) : 1;
        a.nblk[ax] = (g.tile[ax] + a.blk[ax] - 1) / a.blk[ax];
    }
    a.G = g.G;
    a.M = p->M;
    a.nc = p->nc;
    a.TC = g.tile[0] * g.tile[1] * g.tile[2];
    a.TT = g.tile[0] + g.tile[1] + (g.dim == 3 ? g.tile[2] : 0);
    a.ns = g.ns;
    a.layout = p->layout;
    a.use_dcf = use_dcf && p->has_dcf;
    a.items = p->rec.spread_items;
    a.reduce_items = p->rec.reduce_items;
    a.pair_a = p->rec.pair_a;
    a.pair_b = p->rec.pair_b;
    a.in = samples;
    a.grid = p->grid;
    a.partial = p->rec.partial;
    return a;
}

int launch_spread(gn_plan_s *p, const float2 *samples, int use_dcf, float2 *grid)
{
    const Geometry &g = p->geo;
    SpreadArgs a = make_spread_args(p, samples, use_dcf);
    int nitems = p->rec.n_spread_items;
    if (grid) {
        a.grid = grid; // every tile written (no pass skips cells of this grid)
    } else if (p->fft_custom && p->fft_engine == GN_FFT_AUTO) {
        // the pruned pass C' reads only occupied tiles: empty ones need no zeros.  With
        // one mask bit per tile every empty tile is skipped, so the empty tiles' items
        // (after the others) are not launched at all.
        a.occ = p->rec.occ_mask;
        a.occ_k = p->rec.mask_k;
        if (p->rec.mask_k == 1) nitems = p->rec.n_spread_full;
    }
    hipError_t e = spread_any(g.dim, g.ns, a, nitems, p->rec.n_reduce_items, p->rec.reduce_items, p->nc, p->stream);
    if (e != hipSuccess) return hip_fail(e, "spread launch");
    return GN_OK;
}

GatherArgs make_gather_args(const gn_plan_s *p, float2 *samples)
{
    const Geometry &g = p->geo;
    GatherArgs a;
    for (int ax = 0; ax < 3; ++ax) {
        a.nf[ax] = g.nf[ax];
        a.tile[ax] = g.gtile[ax];
        a.ntiles[ax] = g.ngtiles[ax];
        a.region[ax] = (int)std::min<int64_t>(g.gtile[ax] + 2 * g.ns - 1, g.nf[ax]);
        a.coef[ax] = g.coef[ax];
    }
    a.G = g.G;
    a.M = p->M;
    a.nc = p->nc;
    a.layout = p->layout;
    a.items = p->rec.gather_items;
    a.rec_cell = p->rec.cell;
    a.rec_frac = p->rec.frac;
    a.grid = p->grid;
    a.out = samples;
    return a;
}

int launch_gather(gn_plan_s *p, float2 *samples, const float2 *grid, float scale)
{
    const Geometry &g = p->geo;
    if (p->M == 0 || p->rec.n_gather_items == 0) return GN_OK;
    GatherArgs a = make_gather_args(p, samples);
    if (grid) a.grid = grid;
    a.scale = scale;
    hipError_t e = gather_any(g.dim, g.ns, a, p->rec.n_gather_items, p->nc, p->stream);
    if (e != hipSuccess) return hip_fail(e, "gather launch");
    return GN_OK;
}

namespace {
template <int D, int NS>
hipError_t traj_grad_dispatch(const GatherArgs &a, int nitems, const float2 *wts, float *out, const float *gs,
                              hipStream_t st)
{
    const size_t rc = (size_t)a.region[0] * a.region[1] * (D == 3 ? a.region[2] : 1);
    bool wrap = false;
    for (int ax = 0; ax < D; ++ax) wrap |= a.region[ax] >= a.nf[ax];
    // Coil pairs (16-byte cells) while two workgroups of them fit a CU, else one coil at a time.
    // 96^3, 600,000 samples, the whole call, us, in brackets with the products formed per cell:
    // nspread 3, 2 coils, pairs 201 (233); pairs / single coils: nspread 5, 4 coils 998 / 906
    // (971), 3 coils 961 / 695 (747), 1 coil 509 / 287 (300); nspread 8, 2 coils 2717 / 2160
    // (2338).  A pair costs a missing second coil in full, which three coils with wide windows
    // in 2-D do not win back (256^2, nspread 14: 160 / 123 (125)).
    const bool pair = a.nc > 1 && rc * sizeof(float4) <= 80 * 1024 && !(a.nc == 3 && NS >= 8);
    const size_t lds = rc * (pair ? sizeof(float4) : sizeof(float2));
    auto go = [&](auto kernel) {
        lds_limit(kernel, lds);
        hipLaunchKernelGGL(kernel, dim3((unsigned)nitems), dim3(kGatherThreads), lds, st, a, wts, out, gs[0], gs[1], gs[2]);
    };
    if (pair)
        wrap ? go(k_traj_grad<D, NS, true, true>) : go(k_traj_grad<D, NS, false, true>);
    else
        wrap ? go(k_traj_grad<D, NS, true, false>) : go(k_traj_grad<D, NS, false, false>);
    return hipGetLastError();
}

hipError_t traj_grad_any(int dim, int ns, const GatherArgs &a, int nitems, const float2 *wts, float *out,
                         const float *gs, hipStream_t st)
{
    if (dim == 3) {
        GN_NS_CASES(3, traj_grad_dispatch, a, nitems, wts, out, gs, st)
    } else {
        GN_NS_CASES(2, traj_grad_dispatch, a, nitems, wts, out, gs, st)
        GN_NS_CASES_2D_EXTRA(traj_grad_dispatch, a, nitems, wts, out, gs, st)
    }
    return hipErrorInvalidValue;
}
} // namespace

int launch_traj_grad(gn_plan_s *p, const float2 *wts, float *out)
{
    const Geometry &g = p->geo;
    if (p->M == 0 || p->rec.n_gather_items == 0) return GN_OK;
    GatherArgs a;
    for (int ax = 0; ax < 3; ++ax) {
        a.nf[ax] = g.nf[ax];
        a.tile[ax] = g.gtile[ax];
        a.ntiles[ax] = g.ngtiles[ax];
        a.region[ax] = (int)std::min<int64_t>(g.gtile[ax] + 2 * g.ns - 1, g.nf[ax]);
        a.coef[ax] = g.coef[ax];
    }
    a.G = g.G;
    a.M = p->M;
    a.nc = p->nc;
    a.layout = p->layout;
    a.items = p->rec.gather_items;
    a.rec_cell = p->rec.cell;
    a.rec_frac = p->rec.frac;
    a.grid = p->grid;
    a.out = nullptr;
    float gs[3] = {0.f, 0.f, 0.f};
    const double pi = 3.141592653589793;
    for (int ax = 0; ax < g.dim; ++ax) gs[ax] = (float)(-(2 * pi / (double)g.nf[ax]) * p->df / (2.0 * p->tau));
    hipError_t e = traj_grad_any(g.dim, g.ns, a, p->rec.n_gather_items, wts, out, gs, p->stream);
    if (e != hipSuccess) return hip_fail(e, "trajectory gradient launch");
    return GN_OK;
}

PrepostArgs make_prepost(const gn_plan_s *p, float scale) { return make_prepost_impl(p, scale); }

int launch_pad(gn_plan_s *p, const float2 *image, float scale, bool sense)
{
    PrepostArgs a = make_prepost(p, scale);
    if (sense) a.sens = p->sens;
    dim3 grid(grid_blocks(p->geo.G, 256, 1 << 16));
    if (p->geo.dim == 3)
        hipLaunchKernelGGL(k_pad<3>, grid, dim3(256), 0, p->stream, a, image, p->grid);
    else
        hipLaunchKernelGGL(k_pad<2>, grid, dim3(256), 0, p->stream, a, image, p->grid);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "pad launch");
    return GN_OK;
}

int launch_crop(gn_plan_s *p, float2 *image, float scale, bool sense)
{
    PrepostArgs a = make_prepost(p, scale);
    if (sense) a.sens = p->sens;
    dim3 grid(grid_blocks(p->geo.N, 256, 1 << 16));
    if (p->geo.dim == 3)
        hipLaunchKernelGGL(k_crop<3>, grid, dim3(256), 0, p->stream, a, p->grid, image);
    else
        hipLaunchKernelGGL(k_crop<2>, grid, dim3(256), 0, p->stream, a, p->grid, image);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "crop launch");
    return GN_OK;
}

// x[n] = sum_c conj(S[n, c]) * img[n, c] (coils in order), for SENSE combines whose
// coils do not fit one row-pass block
__global__ __launch_bounds__(256) void k_sense_combine(int64_t N, int64_t nc, int layout, const float2 *__restrict__ sens,
                                                       const float2 *__restrict__ img, float2 *__restrict__ x)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; n < N; n += stride) {
        float2 acc = make_float2(0.f, 0.f);
        for (int64_t c = 0; c < nc; ++c) {
            const int64_t i = layout == GN_COIL_LAST ? n * nc + c : c * N + n;
            const float2 s = sens[i], o = img[i];
            acc.x += s.x * o.x + s.y * o.y;
            acc.y += s.x * o.y - s.y * o.x;
        }
        x[n] = acc;
    }
}

int launch_sense_combine(gn_plan_s *p, const float2 *coil_images, float2 *image)
{
    hipLaunchKernelGGL(k_sense_combine, dim3(grid_blocks(p->geo.N, 256, 1 << 16)), dim3(256), 0, p->stream, p->geo.N,
                       p->nc, p->layout, p->sens, coil_images, image);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GN_OK : hip_fail(e, "SENSE combine");
}

// ---------------------------------------------------------------------------
// Batched launchers: one launch per stage over the work of many plans.
// ---------------------------------------------------------------------------

namespace {
template <typename K>
hipError_t spread_batch_go(K kernel, const SpreadShape &sh, const SpreadArgs *d_args, const int4 *d_items, int n,
                           hipStream_t st)
{
    lds_limit(kernel, sh.lds);
    return item_parts(n, 64 * sh.waves, sh.nbg, [&](int64_t o, unsigned part) {
        hipLaunchKernelGGL(kernel, dim3(part, (unsigned)sh.nbg), dim3(64 * sh.waves), sh.lds, st, d_args, d_items + o);
        return hipGetLastError();
    });
}

template <int D>
hipError_t spread_batch_dispatch(const SpreadShape &sh, const SpreadArgs *d_args, const int4 *d_items, int n,
                                 hipStream_t st)
{
    switch (sh.kind * 16 + sh.width) {
    case kSpreadSub * 16 + 1: return spread_batch_go(k_spread_sub_batch<1>, sh, d_args, d_items, n, st);
    case kSpreadSub * 16 + 2: return spread_batch_go(k_spread_sub_batch<2>, sh, d_args, d_items, n, st);
    case kSpreadTile * 16 + 8: return spread_batch_go(k_spread_tile_batch<3, 8>, sh, d_args, d_items, n, st); // 3-D only
    case kSpreadTile * 16 + 4: return spread_batch_go(k_spread_tile_batch<D, 4>, sh, d_args, d_items, n, st);
    case kSpreadTile * 16 + 2: return spread_batch_go(k_spread_tile_batch<D, 2>, sh, d_args, d_items, n, st);
    case kSpreadMfma * 16 + 8: return spread_batch_go(k_spread_mfma_batch<D, 8>, sh, d_args, d_items, n, st);
    case kSpreadMfma * 16 + 4: return spread_batch_go(k_spread_mfma_batch<D, 4>, sh, d_args, d_items, n, st);
    case kSpreadMfma * 16 + 2: return spread_batch_go(k_spread_mfma_batch<D, 2>, sh, d_args, d_items, n, st);
    case kSpreadMfma * 16 + 1: return spread_batch_go(k_spread_mfma_batch<D, 1>, sh, d_args, d_items, n, st);
    case kSpreadValu * 16 + 8: return spread_batch_go(k_spread_batch<D, 8>, sh, d_args, d_items, n, st);
    case kSpreadValu * 16 + 4: return spread_batch_go(k_spread_batch<D, 4>, sh, d_args, d_items, n, st);
    case kSpreadValu * 16 + 2: return spread_batch_go(k_spread_batch<D, 2>, sh, d_args, d_items, n, st);
    case kSpreadValu * 16 + 1: return spread_batch_go(k_spread_batch<D, 1>, sh, d_args, d_items, n, st);
    default: return hipErrorInvalidValue;
    }
}

template <int D, int NS>
hipError_t gather_batch_dispatch(bool wrap, const GatherArgs *d_args, const int4 *d_items, int n, size_t lds,
                                 hipStream_t st)
{
    if (wrap) {
        lds_limit(k_gather_batch<D, NS, true>, lds);
        hipLaunchKernelGGL((k_gather_batch<D, NS, true>), dim3((unsigned)n), dim3(kGatherThreads), lds, st, d_args,
                           d_items);
    } else {
        lds_limit(k_gather_batch<D, NS, false>, lds);
        hipLaunchKernelGGL((k_gather_batch<D, NS, false>), dim3((unsigned)n), dim3(kGatherThreads), lds, st, d_args,
                           d_items);
    }
    return hipGetLastError();
}
} // namespace

hipError_t launch_spread_batch(int dim, const SpreadShape &sh, const SpreadArgs *d_args, const int4 *d_items, int n,
                               hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    return dim == 3 ? spread_batch_dispatch<3>(sh, d_args, d_items, n, st)
                    : spread_batch_dispatch<2>(sh, d_args, d_items, n, st);
}

hipError_t launch_spread_reduce_batch(int dim, const SpreadArgs *d_args, const int4 *d_items, int n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (dim == 3)
        hipLaunchKernelGGL(k_spread_reduce_batch<3>, dim3((unsigned)n, 4), dim3(kReduceThreads), 0, st, d_args, d_items);
    else
        hipLaunchKernelGGL(k_spread_reduce_batch<2>, dim3((unsigned)n, 4), dim3(kReduceThreads), 0, st, d_args, d_items);
    return hipGetLastError();
}

hipError_t launch_gather_batch(int dim, int ns, bool wrap, const GatherArgs *d_args, const int4 *d_items, int n,
                               size_t lds, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (dim == 3) {
        GN_NS_CASES(3, gather_batch_dispatch, wrap, d_args, d_items, n, lds, st)
    } else {
        GN_NS_CASES(2, gather_batch_dispatch, wrap, d_args, d_items, n, lds, st)
        GN_NS_CASES_2D_EXTRA(gather_batch_dispatch, wrap, d_args, d_items, n, lds, st)
    }
    return hipErrorInvalidValue;
}

hipError_t launch_pad_batch(int dim, const PrepostArgs *d_args, int ninst, int64_t maxG, hipStream_t st)
{
    if (ninst <= 0) return hipSuccess;
    dim3 grid(grid_blocks(maxG, 256, 1 << 14), (unsigned)ninst);
    if (dim == 3)
        hipLaunchKernelGGL(k_pad_batch<3>, grid, dim3(256), 0, st, d_args);
    else
        hipLaunchKernelGGL(k_pad_batch<2>, grid, dim3(256), 0, st, d_args);
    return hipGetLastError();
}

hipError_t launch_crop_batch(int dim, const PrepostArgs *d_args, int ninst, int64_t maxN, hipStream_t st)
{
    if (ninst <= 0) return hipSuccess;
    dim3 grid(grid_blocks(maxN, 256, 1 << 14), (unsigned)ninst);
    if (dim == 3)
        hipLaunchKernelGGL(k_crop_batch<3>, grid, dim3(256), 0, st, d_args);
    else
        hipLaunchKernelGGL(k_crop_batch<2>, grid, dim3(256), 0, st, d_args);
    return hipGetLastError();
}

} // namespace gn
