// Device primitives of the iterative reconstructions (include/gaussnufft_solver.h):
// FP64 deterministic reductions and the Chambolle TV prox in FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <utility>

#include "gaussnufft_solver.h"
#include "gn_host_plan.h"
#include "gn_internal.h"

namespace gn {
namespace {

constexpr int kRedThreads = 256;
constexpr int kRedBlocks = 1024; // partials of one reduction (fixed upper bound)
constexpr int kRedUnroll = 4;    // elements per thread per grid-stride round

// ---------------------------------------------------------------- element loads
struct C2 {
    double re, im;
};

__device__ inline C2 load(const float *p, int64_t i) { return {(double)p[i], 0.0}; }
__device__ inline C2 load(const float2 *p, int64_t i)
{
    float2 v = p[i];
    return {(double)v.x, (double)v.y};
}
__device__ inline C2 load(const double2 *p, int64_t i)
{
    double2 v = p[i];
    return {v.x, v.y};
}

__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block sum of (a, b) in a fixed order: butterfly within each 64-lane wave, then
// the 4 wave sums in wave order.  Result valid in thread 0.
__device__ inline void block_sum2(double &a, double &b)
{
    __shared__ double sa[kRedThreads / 64], sb[kRedThreads / 64];
    a = wave_sum(a);
    b = wave_sum(b);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sa[w] = a;
        sb[w] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = 0;
        b = 0;
        for (int k = 0; k < kRedThreads / 64; ++k) {
            a += sa[k];
            b += sb[k];
        }
    }
}

// OP 0: sum conj(a) b;  OP 1: sum |a - b|^2 (b may be null)
template <typename T, int OP>
__global__ __launch_bounds__(kRedThreads) void k_reduce_partial(const T *__restrict__ a, const T *__restrict__ b,
                                                                int64_t n, double2 *__restrict__ part)
{
    double sr = 0.0, si = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kRedThreads;
    for (int64_t base = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; base < n; base += stride * kRedUnroll) {
#pragma unroll
        for (int u = 0; u < kRedUnroll; ++u) {
            const int64_t i = base + u * stride;
            if (i < n) {
                C2 x = load(a, i);
                if (OP == 0) {
                    C2 y = load(b, i);
                    sr += x.re * y.re + x.im * y.im;
                    si += x.re * y.im - x.im * y.re;
                } else {
                    if (b) {
                        C2 y = load(b, i);
                        x.re -= y.re;
                        x.im -= y.im;
                    }
                    sr += x.re * x.re + x.im * x.im;
                }
            }
        }
    }
    block_sum2(sr, si);
    if (threadIdx.x == 0) part[blockIdx.x] = make_double2(sr, si);
}

__global__ __launch_bounds__(kRedThreads) void k_reduce_final(const double2 *__restrict__ part, int nb, int nout,
                                                              double *__restrict__ out)
{
    double sr = 0.0, si = 0.0;
    for (int k = threadIdx.x; k < nb; k += kRedThreads) {
        sr += part[k].x;
        si += part[k].y;
    }
    block_sum2(sr, si);
    if (threadIdx.x == 0) {
        out[0] = sr;
        if (nout > 1) out[1] = si;
    }
}

int reduce_blocks(int64_t n)
{
    const int64_t per = (int64_t)kRedThreads * kRedUnroll;
    int64_t nb = (n + per - 1) / per;
    if (nb > kRedBlocks) nb = kRedBlocks;
    return (int)nb;
}

template <int OP>
int reduce(int dtype, int64_t n, const void *a, const void *b, void *work, double *out, void *stream)
{
    if (n < 0 || !out || !work || (n > 0 && !a) || (OP == 0 && n > 0 && !b))
        return fail(GN_EINVAL, "reduction: negative size or null pointer");
    hipStream_t s = (hipStream_t)stream;
    double2 *part = (double2 *)work;
    const int nb = reduce_blocks(n);
    if (nb > 0) {
        switch (dtype) {
        case GN_F32:
            k_reduce_partial<float, OP><<<nb, kRedThreads, 0, s>>>((const float *)a, (const float *)b, n, part);
            break;
        case GN_C64:
            k_reduce_partial<float2, OP><<<nb, kRedThreads, 0, s>>>((const float2 *)a, (const float2 *)b, n, part);
            break;
        case GN_C128:
            k_reduce_partial<double2, OP>
                <<<nb, kRedThreads, 0, s>>>((const double2 *)a, (const double2 *)b, n, part);
            break;
        default:
            return fail(GN_EINVAL, "reduction: unknown dtype " + std::to_string(dtype));
        }
    } else if (dtype != GN_F32 && dtype != GN_C64 && dtype != GN_C128) {
        return fail(GN_EINVAL, "reduction: unknown dtype " + std::to_string(dtype));
    }
    k_reduce_final<<<1, kRedThreads, 0, s>>>(part, nb, OP == 0 ? 2 : 1, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "reduction launch");
    return GN_OK;
}

// ---------------------------------------------------------------- TV prox (FP64)
//
// Arrays are C-ordered (s0, s1[, s2], nt): NDIM image axes, then nt trailing
// elements.  grad(x)_a = x[.. i_a+1 ..] - x[.. i_a ..], zero on the last slice of axis a.
// Div(p) = sum_a adjD_a(p_a) with adjD(p)[i] = p[i-1]-p[i] (1 <= i <= s-2),
// adjD(p)[0] = -p[0], adjD(p)[s-1] = p[s-2]: the exact adjoint of grad.

struct TVGeom {
    int s[3];      // image axes (s[2] = 1 for NDIM 2)
    int nt;        // trailing elements per pixel
    int stride[3]; // element strides of the image axes
    int n;         // total elements
};

__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

template <typename T> __device__ inline double2 ld2(const T *p, int i);
template <> __device__ inline double2 ld2<float2>(const float2 *p, int i)
{
    float2 v = p[i];
    return make_double2(v.x, v.y);
}
template <> __device__ inline double2 ld2<double2>(const double2 *p, int i) { return p[i]; }
__device__ inline void st2(float2 *p, int i, double2 v) { p[i] = make_float2((float)v.x, (float)v.y); }
__device__ inline void st2(double2 *p, int i, double2 v) { p[i] = v; }

// principal complex square root (the C99 csqrt branch: Re >= 0, Im takes the sign of b)
__device__ inline double2 csqrt_d(double2 z)
{
    const double a = z.x, b = z.y;
    if (a == 0.0 && b == 0.0) return make_double2(0.0, b);
    const double t = sqrt((fabs(a) + hypot(a, b)) * 0.5);
    if (a >= 0.0) return make_double2(t, b / (2.0 * t));
    return make_double2(fabs(b) / (2.0 * t), copysign(t, b));
}

__device__ inline double2 cdiv_d(double2 a, double2 d)
{
    // Smith's algorithm
    if (fabs(d.x) >= fabs(d.y)) {
        const double r = d.y / d.x, den = d.x + d.y * r;
        return make_double2((a.x + a.y * r) / den, (a.y - a.x * r) / den);
    }
    const double r = d.x / d.y, den = d.x * r + d.y;
    return make_double2((a.x * r + a.y) / den, (a.y * r - a.x) / den);
}

// v / max(amp(v), 1)
template <int NDIM, int AMP> __device__ inline void tv_project(double2 *v)
{
    if (AMP == GN_TV_AMP_SQUARE) {
        // s = sum_a v_a^2 with complex squares; d = sqrt(s); numpy maximum(d, 1) keeps d
        // when d >= 1 in lexicographic (real, imag) order or when d is NaN
        double2 s = make_double2(0.0, 0.0);
#pragma unroll
        for (int a = 0; a < NDIM; ++a)
            s = cadd(s, make_double2(v[a].x * v[a].x - v[a].y * v[a].y, v[a].x * v[a].y + v[a].y * v[a].x));
        // Re d >= 1 is Re s + |s| >= 2: cells clearly below it (a margin of some rounding
        // errors) are done, the others form d and take the rule above on it
        const double a = s.x, b = s.y;
        if (a < 1.0 && b * b < (4.0 - 1e-14) * (1.0 - a)) return;
        const double n = a * a + b * b;
        double2 d;
        if (n < 1e300) {
            // |d|^2 = |s| = m, so v / d = v conj(d) / m: two square roots and two quotients,
            // where csqrt_d and cdiv_d take a scaled hypot and 2 NDIM + 2 quotients
            const double m = sqrt(n), t = sqrt((fabs(a) + m) * 0.5), o = b / (2.0 * t);
            d = a >= 0.0 ? make_double2(t, o) : make_double2(fabs(o), copysign(t, b));
            if (d.x > 1.0 || (d.x == 1.0 && d.y >= 0.0)) {
                const double q = 1.0 / m;
#pragma unroll
                for (int k = 0; k < NDIM; ++k)
                    v[k] = make_double2((v[k].x * d.x + v[k].y * d.y) * q, (v[k].y * d.x - v[k].x * d.y) * q);
            }
            return;
        }
        // beyond the range of a^2 + b^2, infinities, NaN
        d = csqrt_d(s);
        const bool keep = d.x > 1.0 || (d.x == 1.0 && d.y >= 0.0) || isnan(d.x) || isnan(d.y);
        if (keep) {
#pragma unroll
            for (int k = 0; k < NDIM; ++k) v[k] = cdiv_d(v[k], d);
        }
    } else {
        double m = 0.0;
#pragma unroll
        for (int a = 0; a < NDIM; ++a) m += v[a].x * v[a].x + v[a].y * v[a].y;
        m = sqrt(m);
        if (m > 1.0) {
#pragma unroll
            for (int a = 0; a < NDIM; ++a) v[a] = make_double2(v[a].x / m, v[a].y / m);
        }
    }
}

// A Chambolle step as two kernels, one thread per cell: D = Div(G) - y / lambda, then G.
template <int NDIM> __device__ inline void tv_coords(const TVGeom &g, int idx, int *c)
{
    int r = idx / g.nt;
    if (NDIM == 3) {
        c[2] = r % g.s[2];
        r /= g.s[2];
    }
    c[1] = r % g.s[1];
    c[0] = r / g.s[1];
}

// adjD_a(p) at idx, position i of s on the axis
__device__ inline double2 adj_at(const double2 *__restrict__ p, int i, int s, int stride, int idx)
{
    if (i == 0) return make_double2(-p[idx].x, -p[idx].y);
    if (i == s - 1) return p[idx - stride];
    return csub(p[idx - stride], p[idx]);
}

// D = Div(G) - y/lambda (FINAL: f = y - lambda*Div(G)).  first: G is zero.
template <typename T, int NDIM, bool FINAL>
__global__ __launch_bounds__(256) void k_tv_div(TVGeom g, const double2 *__restrict__ G, const T *__restrict__ y,
                                                double lambda, int first, double2 *__restrict__ D, T *__restrict__ f)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= g.n) return;
    int c[3];
    tv_coords<NDIM>(g, idx, c);
    const double2 yv = ld2<T>(y, idx);
    double2 dv = make_double2(0.0, 0.0);
    if (!first) {
#pragma unroll
        for (int a = 0; a < NDIM; ++a) dv = cadd(dv, adj_at(G + (int64_t)a * g.n, c[a], g.s[a], g.stride[a], idx));
    }
    if (FINAL)
        st2(f, idx, make_double2(yv.x - lambda * dv.x, yv.y - lambda * dv.y));
    else
        D[idx] = make_double2(dv.x - yv.x / lambda, dv.y - yv.y / lambda);
}

// G = G - step*grad(D); G = G / max(amp(G), 1).  first: G is zero on entry.
template <int NDIM, int AMP>
__global__ __launch_bounds__(256) void k_tv_step(TVGeom g, double2 *__restrict__ G, const double2 *__restrict__ D,
                                                 double step, int first)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= g.n) return;
    int c[3];
    tv_coords<NDIM>(g, idx, c);
    const double2 d0 = D[idx];
    double2 v[NDIM];
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        const double2 dd = (c[a] < g.s[a] - 1) ? csub(D[idx + g.stride[a]], d0) : make_double2(0.0, 0.0);
        const double2 old = first ? make_double2(0.0, 0.0) : G[(int64_t)a * g.n + idx];
        v[a] = make_double2(old.x - step * dd.x, old.y - step * dd.y);
    }
    tv_project<NDIM, AMP>(v);
#pragma unroll
    for (int a = 0; a < NDIM; ++a) G[(int64_t)a * g.n + idx] = v[a];
}

// Several Chambolle steps per launch.  A step is D = Div(G) - y / lambda, then
// G = G - step grad(D), G = G / max(amp(G), 1); D at a cell needs G there and one cell
// before it on each axis, the new G needs D there and one cell after it.  A block loads
// a region of one cell per thread (32 x 32, or 10 x 10 x 10) with G, D in LDS, runs `iters`
// steps on it, the valid part shrinking by one cell on every side per step, and writes
// the tile that is left; the last launch also writes f = y - lambda Div(G), which takes
// one more cell on the low sides.  Every cell's arithmetic is that of one step per
// launch, so the result does not depend on the split.
// In 2-D the steps of small images are bound by launches and by the latency of the FP64
// chain (square roots and quotients), so up to 7 steps (tiles of 18 x 18) run per launch:
// 256^2, 40 steps: 76 us, against 276 us as two kernels per step (512^2: 208 / 477 us).  In 3-D the field is
// 48 bytes per cell and a halo of more than one cell costs more than it saves: one step
// per launch, D never stored (96^3: 1.06 ms for 40 steps, two kernels 1.49 ms).
// See tv_regions for the shapes that take two kernels per step.
constexpr int kTVThreads = 1024;
constexpr int kTVSteps2 = 7, kTVSteps3 = 1;

template <int NDIM> struct TVRegion;
template <> struct TVRegion<2> {
    static constexpr int r0 = 32, r1 = 32, r2 = 1, st0 = 32, st1 = 1, st2 = 0; // cells and LDS strides
};
template <> struct TVRegion<3> {
    static constexpr int r0 = 10, r1 = 10, r2 = 10, st0 = 100, st1 = 10, st2 = 1; // 1000 threads
};

struct TVLaunch {
    int iters, first, last; // steps; G is zero on entry; write f
    int lo;                 // halo cells before the tile
    int t[3], nt[3];        // tile cells and tiles per axis
};

template <typename T, int NDIM, int AMP>
__global__ __launch_bounds__(kTVThreads) void k_tv_steps(TVGeom g, TVLaunch L, const T *__restrict__ y, double lambda,
                                                         double step, const double2 *__restrict__ gin,
                                                         double2 *__restrict__ gout, T *__restrict__ f)
{
    using R = TVRegion<NDIM>;
    __shared__ double2 sG[NDIM][kTVThreads], sD[kTVThreads];
    const int tid = threadIdx.x;
    const int r[3] = {R::r0, R::r1, R::r2}, st[3] = {R::st0, R::st1, R::st2};
    const int l[3] = {tid / R::st0, (tid / R::st1) % R::r1, tid % R::r2};
    int c[3];
    // Blocks go to the 8 XCDs in turn: each takes a run of neighbouring tiles, whose halos
    // then come from its L2.  Trailing elements fastest: the blocks of one tile share its
    // cache lines.
    const int per = gridDim.x / 8, nx = per * 8;
    int b = (int)blockIdx.x < nx ? (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int t = b % g.nt;
    b /= g.nt;
    bool in = l[0] < R::r0, tile = true;
    int idx = t;
#pragma unroll
    for (int a = NDIM - 1; a >= 0; --a) {
        c[a] = (b % L.nt[a]) * L.t[a] - L.lo + l[a];
        b /= L.nt[a];
        in = in && c[a] >= 0 && c[a] < g.s[a];
        tile = tile && l[a] >= L.lo && l[a] < L.lo + L.t[a];
        idx += c[a] * g.stride[a];
    }
    double2 v[NDIM], yv = make_double2(0.0, 0.0);
#pragma unroll
    for (int a = 0; a < NDIM; ++a) v[a] = make_double2(0.0, 0.0);
    if (in) {
        yv = ld2<T>(y, idx);
        if (!L.first) {
#pragma unroll
            for (int a = 0; a < NDIM; ++a) v[a] = gin[(int64_t)a * g.n + idx];
        }
    }
    const double2 yl = make_double2(yv.x / lambda, yv.y / lambda);
#pragma unroll
    for (int a = 0; a < NDIM; ++a) sG[a][tid] = v[a];
    auto div = [&]() {
        double2 dv = make_double2(0.0, 0.0);
#pragma unroll
        for (int a = 0; a < NDIM; ++a) {
            const double2 p = l[a] > 0 ? sG[a][tid - st[a]] : make_double2(0.0, 0.0);
            dv = cadd(dv, c[a] == 0 ? make_double2(-v[a].x, -v[a].y) : c[a] == g.s[a] - 1 ? p : csub(p, v[a]));
        }
        return dv;
    };
    for (int it = 0; it < L.iters; ++it) {
        __syncthreads();
        const double2 dv = div();
        const double2 d0 = make_double2(dv.x - yl.x, dv.y - yl.y);
        sD[tid] = d0;
        __syncthreads();
        if (in) {
#pragma unroll
            for (int a = 0; a < NDIM; ++a) {
                const bool next = c[a] < g.s[a] - 1 && l[a] < r[a] - 1;
                const double2 dd = next ? csub(sD[tid + st[a]], d0) : make_double2(0.0, 0.0);
                v[a] = make_double2(v[a].x - step * dd.x, v[a].y - step * dd.y);
            }
            tv_project<NDIM, AMP>(v);
#pragma unroll
            for (int a = 0; a < NDIM; ++a) sG[a][tid] = v[a];
        }
    }
    if (!L.last) {
        if (in && tile) {
#pragma unroll
            for (int a = 0; a < NDIM; ++a) gout[(int64_t)a * g.n + idx] = v[a];
        }
        return;
    }
    __syncthreads();
    const double2 dv = div();
    if (in && tile) st2(f, idx, make_double2(yv.x - lambda * dv.x, yv.y - lambda * dv.y));
}

// Steps and tiles of launch k of n.
template <int NDIM> TVLaunch tv_launch(const TVGeom &g, int niter, int k, int n, int64_t *blocks)
{
    using R = TVRegion<NDIM>;
    const int r[3] = {R::r0, R::r1, R::r2};
    TVLaunch L;
    L.iters = (int)((int64_t)niter * (k + 1) / n - (int64_t)niter * k / n);
    L.first = k == 0;
    L.last = k == n - 1;
    L.lo = L.iters + L.last;
    *blocks = g.nt;
    for (int a = 0; a < 3; ++a) {
        L.t[a] = a < NDIM ? r[a] - L.iters - L.lo : 1;
        L.nt[a] = a < NDIM ? (g.s[a] + L.t[a] - 1) / L.t[a] : 1;
        *blocks *= L.nt[a];
    }
    return L;
}

template <int NDIM> int tv_launches(int niter)
{
    const int most = NDIM == 2 ? kTVSteps2 : kTVSteps3;
    return std::max(1, (int)(((int64_t)niter + most - 1) / most)); // the steps are shared out evenly
}

// Whether the steps run on LDS regions.  A region costs its block the same however few of
// its cells the array fills (thin axes, small images with many trailing elements), and a
// trailing dimension makes its accesses uncoalesced; two kernels per step cost launches and
// passes over the field.
// 2-D: up to 1024 blocks, or 200 cells per block and step (430 for a single step).
// Microseconds, two kernels / regions (cells): 3 x 3 x 1000, 40 steps 265 / 130; 16384 x 2
// 255 / 250; 8 x 8 x 4096 (64) 343 / 481; 65536 x 2 (36) 288 / 760; 24 x 24 x 4096 (144) x 1.32;
// 14 x 14 x 4096 (196) x 0.67; 40 x 40 x 4096 (213) x 0.94, a single step (400) x 1.13; 64 x 64
// x 256, a single step (455) x 0.86.
// 3-D, one step per launch: one trailing element and 435 cells or more, else the smaller
// estimate, microseconds from 898 measured calls: a launch of regions 5 or 0.009 per block
// (6.5 or 0.02 with a trailing dimension), one of the other kernels 3 or 9e-6 per element.
// 256 x 256 x 2, 40 steps (127 cells) 382 / 569; 256 x 256 x 8, 3 steps (329) 54 / 66; 100^3
// (449) 1600 / 1221; 61 x 29 x 24, 2 steps 20 / 13; 64^3 x 8 (501) 2956 / 3506.
// Regions keep the dual field twice, 16 ndim bytes per element against 16 for D: above
// kTVTwiceMax elements (24 GiB of fields once, in 3-D) the memory is left to the caller.
// They also need every launch's blocks to fit one launch (2^22 of 1024 threads); the two
// kernels' 256-thread blocks fit for every array that is taken.
constexpr int64_t kTVTwiceMax = (int64_t)1 << 29;

template <int NDIM> bool tv_regions(const TVGeom &g, int niter)
{
    if (g.n > kTVTwiceMax) return false;
    const int n = tv_launches<NDIM>(niter);
    int64_t block_steps = 0;
    double regions = 0.0;
    for (int k = 0; k < n; ++k) {
        int64_t blocks = 0;
        const TVLaunch L = tv_launch<NDIM>(g, niter, k, n, &blocks);
        if (!host::launch_fits(blocks, kTVThreads)) return false;
        block_steps += blocks * L.iters;
        regions += g.nt == 1 ? std::max(5.0, 0.009 * (double)blocks) : std::max(6.5, 0.02 * (double)blocks);
    }
    if (niter == 0) return true;
    const auto filled = [&](int64_t cells) { return (int64_t)g.n * niter >= cells * block_steps; };
    if (NDIM == 2) return block_steps <= (int64_t)1024 * niter || filled(niter == 1 ? 430 : 200);
    return (g.nt == 1 && filled(435)) || regions <= (2.0 * niter + 1.0) * std::max(3.0, 9e-6 * (double)g.n);
}

template <typename T, int NDIM, int AMP>
int tv_prox(TVGeom g, const T *y, double lambda, double step, int niter, double2 *work, T *f, hipStream_t s)
{
    if (tv_regions<NDIM>(g, niter)) {
        const int n = tv_launches<NDIM>(niter);
        double2 *cur = work, *next = work + (int64_t)NDIM * g.n;
        for (int k = 0; k < n; ++k) {
            int64_t blocks = 0;
            const TVLaunch L = tv_launch<NDIM>(g, niter, k, n, &blocks);
            k_tv_steps<T, NDIM, AMP><<<(unsigned)blocks, kTVThreads, 0, s>>>(g, L, y, lambda, step, cur, next, f);
            std::swap(cur, next);
        }
    } else {
        double2 *G = work, *D = work + (int64_t)NDIM * g.n;
        const unsigned nb = (unsigned)(((int64_t)g.n + 255) / 256);
        for (int it = 0; it < niter; ++it) {
            k_tv_div<T, NDIM, false><<<nb, 256, 0, s>>>(g, G, y, lambda, it == 0, D, f);
            k_tv_step<NDIM, AMP><<<nb, 256, 0, s>>>(g, G, D, step, it == 0);
        }
        k_tv_div<T, NDIM, true><<<nb, 256, 0, s>>>(g, G, y, lambda, niter == 0, D, f);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? GN_OK : hip_fail(e, "TV prox launch");
}

template <typename T>
int tv_prox_any(int ndim, int amp, TVGeom g, const T *y, double lambda, double step, int niter, double2 *work, T *f,
                hipStream_t s)
{
    if (amp == GN_TV_AMP_SQUARE)
        return ndim == 2 ? tv_prox<T, 2, GN_TV_AMP_SQUARE>(g, y, lambda, step, niter, work, f, s)
                         : tv_prox<T, 3, GN_TV_AMP_SQUARE>(g, y, lambda, step, niter, work, f, s);
    return ndim == 2 ? tv_prox<T, 2, GN_TV_AMP_MODULUS>(g, y, lambda, step, niter, work, f, s)
                     : tv_prox<T, 3, GN_TV_AMP_MODULUS>(g, y, lambda, step, niter, work, f, s);
}

// ---------------------------------------------------------------------------
// One IST or FISTA update.  Bound by the launch: 256^2 elements are 3 MB of traffic.  As
// separate elementwise passes with temporaries the same update took 11 launches, about 45 us of a
// 270 us iteration (256^2, 32 coils); as one kernel the iteration takes 37 us less.
// Products with real factors, and the signs of sums, keep the terms of a complex product with
// imaginary part 0, so that infinities and NaN end up where complex arithmetic puts them.
// The quotient is a product with the reciprocal, as in a complex division, so that every
// rounding is the separate passes': with a / d 20 iterations of 12 inputs ended 1.4 % further
// from their 64-bit values.  (In FP64, rounded once per output, they end 60 % further: a
// phantom's regions of one value meet the roundings alike, and these offset the operator's.)
// ---------------------------------------------------------------------------
__device__ inline float2 scale_c(float2 v, float s)
{
    return make_float2(v.x * s - v.y * 0.f, v.x * 0.f + v.y * s);
}

__device__ inline float2 add_c(float2 a, float2 b, float sign)
{
    const float2 t = scale_c(b, sign);
    return make_float2(a.x + t.x, a.y + t.y);
}

__global__ void k_soft_step(int64_t n, const float2 *__restrict__ g, const float2 *__restrict__ b,
                            float2 *__restrict__ acc, float step, float th, float2 *__restrict__ x,
                            const float2 *__restrict__ x_pre, float beta, float2 *__restrict__ y)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float2 r = g[i], a = acc[i], xp = make_float2(0.f, 0.f);
    if (b) r = add_c(r, b[i], -1.f);
    if (y) xp = x_pre[i];
    a = add_c(a, scale_c(r, step), -1.f);
    acc[i] = a;
    const float m = hypotf(a.x, a.y), d = m + 1e-6f, c = m - th;
    const float q = 1.f / d;
    const float2 u = scale_c(make_float2((a.x + a.y * 0.f) * q, (a.y - a.x * 0.f) * q), c < 0.f ? 0.f : c);
    x[i] = u;
    if (y) y[i] = add_c(u, scale_c(add_c(u, xp, -1.f), beta), 1.f);
}

} // namespace
} // namespace gn

using namespace gn;

extern "C" {

int64_t gn_reduce_work_bytes(void) { return (int64_t)kRedBlocks * (int64_t)sizeof(double2); }

int gn_dot_f64(int dtype, int64_t n, const void *a, const void *b, void *work, double *out, void *stream)
{
    return reduce<0>(dtype, n, a, b, work, out, stream);
}

int gn_sqdist_f64(int dtype, int64_t n, const void *a, const void *b, void *work, double *out, void *stream)
{
    return reduce<1>(dtype, n, a, b, work, out, stream);
}

int64_t gn_tv_work_bytes(int ndim, const int64_t *shape, int64_t nt)
{
    if ((ndim != 2 && ndim != 3) || !shape || nt < 0) return 0;
    int64_t n = nt;
    for (int a = 0; a < ndim; ++a) {
        if (shape[a] < 0) return 0;
        n *= shape[a];
    }
    // the dual field before and after a launch of regions, or the field and D (see tv_regions)
    return (n > kTVTwiceMax ? ndim + 1 : 2 * ndim) * n * (int64_t)sizeof(double2);
}

int gn_tv_prox(int dtype, int ndim, const int64_t *shape, int64_t nt, const void *y, double lambda, double step,
               int niter, int amp_rule, void *work, void *f, void *stream)
{
    if ((ndim != 2 && ndim != 3) || !shape) return fail(GN_EINVAL, "TV prox: ndim must be 2 or 3");
    int64_t n = nt;
    for (int a = 0; a < ndim; ++a) {
        if (shape[a] < 2)
            return fail(GN_EINVAL, "TV prox: every image axis needs at least 2 samples (axis " + std::to_string(a) +
                                       " has " + std::to_string(shape[a]) + ")");
        n *= shape[a];
    }
    if (nt < 1) return fail(GN_EINVAL, "TV prox: nt must be >= 1");
    if (n >= (int64_t)1 << 31) return fail(GN_EINVAL, "TV prox: array too large (>= 2^31 elements)");
    if (!y || !f || !work) return fail(GN_EINVAL, "TV prox: null pointer");
    if (y == f) return fail(GN_EINVAL, "TV prox: y and f must not alias");
    if (!(lambda > 0.0) || !std::isfinite(lambda)) return fail(GN_EINVAL, "TV prox: lambda must be positive");
    if (niter < 0) return fail(GN_EINVAL, "TV prox: niter < 0");
    if (amp_rule != GN_TV_AMP_SQUARE && amp_rule != GN_TV_AMP_MODULUS)
        return fail(GN_EINVAL, "TV prox: unknown amplitude rule");
    TVGeom g;
    g.s[0] = (int)shape[0];
    g.s[1] = (int)shape[1];
    g.s[2] = ndim == 3 ? (int)shape[2] : 1;
    g.nt = (int)nt;
    g.stride[2] = (int)nt;
    g.stride[1] = ndim == 3 ? g.s[2] * (int)nt : (int)nt;
    g.stride[0] = g.s[1] * g.stride[1];
    g.n = (int)n;
    hipStream_t s = (hipStream_t)stream;
    double2 *w = (double2 *)work;
    if (dtype == GN_C64)
        return tv_prox_any<float2>(ndim, amp_rule, g, (const float2 *)y, lambda, step, niter, w, (float2 *)f, s);
    if (dtype == GN_C128)
        return tv_prox_any<double2>(ndim, amp_rule, g, (const double2 *)y, lambda, step, niter, w, (double2 *)f, s);
    return fail(GN_EINVAL, "TV prox: dtype must be GN_C64 or GN_C128");
}

int gn_soft_step(int64_t n, const void *g, const void *b, void *acc, double step, double th, void *x,
                 const void *x_pre, double beta, void *y, void *stream)
{
    constexpr int kThreads = 256;
    if (n < 0) return fail(GN_EINVAL, "soft step: element count out of range");
    if (n == 0) return GN_OK;
    if (!g || !acc || !x || (y && !x_pre)) return fail(GN_EINVAL, "soft step: null pointer");
    if (x == acc || x == g || x == b || x == x_pre || x == y || (y && (y == acc || y == g || y == b || y == x_pre)) ||
        acc == g || acc == b || acc == x_pre)
        return fail(GN_EINVAL, "soft step: outputs must not alias");
    constexpr int64_t kPart = (int64_t)1 << 31; // elements of one launch, which has fewer than 2^32 threads
    static_assert(host::launch_fits(kPart / kThreads, kThreads), "one launch");
    for (int64_t o = 0; o < n; o += kPart) {
        const int64_t m = std::min(kPart, n - o);
        k_soft_step<<<(unsigned)((m + kThreads - 1) / kThreads), kThreads, 0, (hipStream_t)stream>>>(
            m, (const float2 *)g + o, b ? (const float2 *)b + o : nullptr, (float2 *)acc + o, (float)step, (float)th,
            (float2 *)x + o, y ? (const float2 *)x_pre + o : nullptr, (float)beta, y ? (float2 *)y + o : nullptr);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? GN_OK : hip_fail(e, "soft step launch");
}

} // extern "C"
