// Cartesian complex-to-complex FFTs over the leading axes of a C-order array whose
// trailing dimensions are a batch (coils), interleaved element by element -- the
// layout of the reference's cuFFT wrappers -- with the centring shifts and the
// k-space mask of the masked Cartesian operators fused.
//
// Lengths the in-LDS transform covers take one kernel pass per axis (k_fft_axis): the
// shifts are index offsets of its loads and stores, the mask and the scale multiply the
// last pass's stores, and the passes run from the input into the output and then in
// place, with no workspace.  Other lengths, and an output that partly overlaps the
// input, use rocFFT between a pass before and a pass after it.
//
//   forward: out = [ifftshift] ( FFT( [fftshift] in ) ) * mask       (unnormalized)
//   inverse: out = [ifftshift] ( IFFT( [fftshift] in ) ) / prod(shape)
//
// rocFFT plans are cached per (rank, shape, batch, direction) for the process; the
// shifted copy lives in a grow-only workspace per device.
#include <hip/hip_runtime.h>
#include <rocfft/rocfft.h>

#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "gn_fft_device.h"
#include "gn_internal.h"

namespace gn {
namespace {

struct CPlan {
    rocfft_plan plan = nullptr;
    rocfft_execution_info info = nullptr;
    void *work = nullptr;
};

std::mutex g_cfft_mu;
std::map<std::tuple<int, int, int64_t, int64_t, int64_t, int64_t, int, int>, CPlan> g_cfft_plans;
std::map<int, std::pair<void *, size_t>> g_cfft_ws;

struct ShiftArgs {
    int rank;
    int64_t n[3];      // transformed lengths (leading axes)
    int64_t batch;     // interleaved batch elements
    int64_t total;     // prod(n) * batch
    int pre;           // roll the input by n/2 (fftshift) while copying
    int post;          // take the output from position (k + n/2) mod n (ifftshift)
    float scale;
    const float *mask; // null, prod(n) (broadcast over the batch) or prod(n) * batch entries
    int64_t mask_batch;
};

// dst[e] = src[roll(e)] (* mask[e] * scale): e = (index of the leading axes) * batch + b.
// pre: fftshift (source index m - n/2); post: ifftshift (source index k + n/2).
__global__ __launch_bounds__(256) void k_shift_copy(ShiftArgs a, const float2 *__restrict__ src,
                                                    float2 *__restrict__ dst, int post)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < a.total; e += stride) {
        const int64_t b = e % a.batch;
        int64_t r = e / a.batch;
        int64_t srcpos = 0, mul = 1;
        int64_t pos = r;
        for (int ax = a.rank - 1; ax >= 0; --ax) {
            const int64_t n = a.n[ax];
            const int64_t i = r % n;
            r /= n;
            int64_t s = i;
            if (post ? a.post : a.pre) {
                s = post ? i + n / 2 : i - n / 2;
                if (s >= n) s -= n;
                if (s < 0) s += n;
            }
            srcpos += s * mul;
            mul *= n;
        }
        float2 v = src[srcpos * a.batch + b];
        if (post) {
            float f = a.scale;
            if (a.mask) f *= a.mask_batch > 1 ? a.mask[pos * a.batch + b] : a.mask[pos];
            v = make_float2(v.x * f, v.y * f);
        }
        dst[e] = v;
    }
}

// ---------------------------------------------------------------------------
// One axis of the transform.  The array is (slabs, L, ncols) with ncols contiguous
// (the trailing axes and the batch); a block takes S slabs x C columns (C = ncols when
// S > 1, so that its elements are one contiguous run) as S * C lines in LDS.  Input row
// n enters at FFT position n + in_off, output row n is FFT index n + out_off (mod L).
// Bound by memory: each pass reads and writes the array once.  512-thread blocks of 16
// lines (128-byte row segments), fewer lines while the launch has fewer than two blocks
// per CU.  Measured at 256 x 256 x 32 (16.8 MB), masked forward then inverse through the
// operator: 47 us, against 147 us for shift pass, rocFFT, shift pass and a wait per call.
// Short lines come by the hundred, 2048 elements a block: 16 lines of 2 or 3 points are a
// block of 256 bytes (2-D 1024 x 2 of 8192: 1381 us, with 1024 lines 172, rocFFT 717).
// ---------------------------------------------------------------------------
constexpr int kAxisThreads = 512;
constexpr int kAxisLines = 16;
constexpr int kAxisElems = 2048;              // elements of a block of short lines, at least
constexpr int kAxisUnroll = 4;                // global loads in flight per thread
constexpr int64_t kAxisBlocks = 512;          // two blocks per CU
constexpr size_t kAxisLdsMax = 64 * 1024;

struct AxisArgs {
    const float2 *src;
    float2 *dst;       // src, or an array that does not overlap it
    int L;
    int C, S;
    int64_t ncols, nslabs;
    int64_t ncb;       // column blocks
    int in_off, out_off;
    int vec;           // 1: two columns per lane (16-byte accesses)
    float sign, scale;
    const float *mask; // last pass only, or null
    int64_t mask_div;  // elements per mask entry: 1 or the batch
    Stages st;
    const float2 *tw;
    const int *pinv;
};

template <bool GEN>
__global__ __launch_bounds__(kAxisThreads, GEN ? 6 : 1) void k_fft_axis(AxisArgs a)
{
    extern __shared__ float2 lds_axis[];
    const int lines = a.C * a.S, estride = lines + 1;
    float2 *tw = lds_axis, *buf = tw + a.L;
    float2 *alt = buf + a.L * estride;
    int *spinv = (int *)(GEN && a.st.dbl ? alt + a.L * estride : alt);
    const int64_t sb = blockIdx.x / a.ncb, slab0 = sb * a.S, col0 = (blockIdx.x - sb * a.ncb) * a.C;
    const int ns = (int)min((int64_t)a.S, a.nslabs - slab0), nc = (int)min((int64_t)a.C, a.ncols - col0);
    const int64_t base = slab0 * a.L * a.ncols + col0;
    const int ws = a.vec, cw = nc >> ws; // vec: nc is even
    const int total = ns * a.L * cw;
    const float rcw = 1.0f / (float)cw, rL = 1.0f / (float)a.L;
    // element e of the block: lane columns j, j + ws; row n; slab s (line s * C + j)
    auto place = [&](int e, int &line, int &n) -> int64_t {
        const int r = fdiv(e, cw, rcw), j = (e - r * cw) << ws;
        const int s = fdiv(r, a.L, rL);
        n = r - s * a.L;
        line = s * a.C + j;
        return base + (int64_t)r * a.ncols + j; // (s * L + n) * ncols + j
    };
    load_tables(tw, spinv, a.tw, a.pinv, a.L, a.sign);
    __syncthreads();
    for (int e0 = threadIdx.x; e0 < total; e0 += kAxisUnroll * kAxisThreads) {
        float4 v[kAxisUnroll];
        int at[kAxisUnroll];
#pragma unroll
        for (int u = 0; u < kAxisUnroll; ++u) {
            const int e = e0 + u * kAxisThreads;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (e < total) {
                int line, n;
                const float2 *p = a.src + place(e, line, n);
                if (ws) {
                    v[u] = *reinterpret_cast<const float4 *>(p);
                } else {
                    const float2 t = *p;
                    v[u].x = t.x;
                    v[u].y = t.y;
                }
                int q = n + a.in_off;
                if (q >= a.L) q -= a.L;
                at[u] = spinv[q] * estride + line;
            }
        }
#pragma unroll
        for (int u = 0; u < kAxisUnroll; ++u)
            if (e0 + u * kAxisThreads < total) {
                buf[at[u]] = make_float2(v[u].x, v[u].y);
                if (ws) buf[at[u] + 1] = make_float2(v[u].z, v[u].w);
            }
    }
    __syncthreads();
    const float2 *res = (lines & 1) == 0 ? fft_lines<2, GEN>(buf, alt, lines, 1, estride, a.L, a.st, tw, a.sign)
                                         : fft_lines<1, GEN>(buf, alt, lines, 1, estride, a.L, a.st, tw, a.sign);
    for (int e = threadIdx.x; e < total; e += kAxisThreads) {
        int line, n;
        const int64_t g = place(e, line, n);
        int q = n + a.out_off;
        if (q >= a.L) q -= a.L;
        const float2 lo = res[q * estride + line];
        float f0 = a.scale, f1 = a.scale;
        if (a.mask) {
            // mask_div is 1 or the batch, which divides ncols
            f0 *= a.mask_div == 1 ? a.mask[g] : a.mask[g / a.mask_div];
            if (ws) f1 *= a.mask_div == 1 ? a.mask[g + 1] : a.mask[(g + 1) / a.mask_div];
        }
        if (ws) {
            const float2 hi = res[q * estride + line + 1];
            *reinterpret_cast<float4 *>(a.dst + g) = make_float4(lo.x * f0, lo.y * f0, hi.x * f1, hi.y * f1);
        } else {
            a.dst[g] = make_float2(lo.x * f0, lo.y * f0);
        }
    }
}

// Tables per (device, length), kept until the process ends: lengths are at most 2048,
// 12 bytes per point.  Under g_cfft_mu.
std::map<std::pair<int, int>, FFTAxis> g_axis_tables;

int axis_table(int dev, int L, FFTAxis **ax)
{
    auto it = g_axis_tables.find({dev, L});
    if (it == g_axis_tables.end()) {
        FFTAxis t;
        const int rc = fft_axis_init(&t, L);
        if (rc) {
            fft_axis_free(&t);
            return rc;
        }
        it = g_axis_tables.emplace(std::make_pair(dev, L), t).first;
    }
    *ax = &it->second;
    return GN_OK;
}

// Lines (columns x slabs) a block of the axis pass may hold: 16, more of short ones so that
// the block has kAxisElems elements, fewer while they exceed kAxisLdsMax.
int axis_lines(int L)
{
    int lines = kAxisLines;
    while (2 * lines * L <= kAxisElems) lines *= 2;
    while (lines > 1 && col_lds(L, lines, host::fft_direct_sums(L)) > kAxisLdsMax) lines /= 2;
    return lines;
}

// The axis passes apply: every length is 1 or covered (and not faster with rocFFT), the
// output is the input or does not overlap it, and the blocks of every axis fit one launch
// (2^23 blocks of about 2048 elements; larger arrays are left to rocFFT, whose shift passes
// loop).
bool axis_passes_ok(int rank, const int64_t *n, int64_t total, const void *in, const void *out)
{
    bool any = false;
    int64_t slabs = 1;
    for (int a = 0; a < rank; ++a) {
        if (n[a] == 1) continue;
        const int64_t ncols = total / (slabs * n[a]);
        if (n[a] > 2048 || (ncols > 1 && !host::axis_strided_ok((int)n[a])) || !fft_length_supported(n[a])) return false;
        const auto sp = host::axis_split(slabs, ncols, axis_lines((int)n[a]), kAxisBlocks);
        if (!host::launch_fits(sp.blocks, kAxisThreads)) return false;
        any = true;
        slabs *= n[a];
    }
    const uintptr_t i = (uintptr_t)in, o = (uintptr_t)out, bytes = (uintptr_t)total * sizeof(float2);
    const bool overlap = i != o && i < o + bytes && o < i + bytes;
    return any && !overlap;
}

// Everything that can fail is done for every axis before the first launch: a pass
// overwrites the output, which may be the input.
int axis_passes(const ShiftArgs &sh, bool fwd, const float2 *in, float2 *out, hipStream_t st)
{
    int dev = 0;
    (void)hipGetDevice(&dev);
    AxisArgs pass[3];
    unsigned blocks[3];
    int np = 0;
    int64_t slabs = 1;
    for (int ax = 0; ax < sh.rank; ++ax) {
        const int64_t n = sh.n[ax];
        if (n == 1) continue;
        FFTAxis *t = nullptr;
        const int rc = axis_table(dev, (int)n, &t);
        if (rc) return rc;
        AxisArgs &a = pass[np];
        a.src = np ? out : in;
        a.dst = out;
        a.L = (int)n;
        a.nslabs = slabs;
        a.ncols = sh.total / (slabs * n);
        a.st = make_stages(*t);
        const auto sp = host::axis_split(slabs, a.ncols, axis_lines(a.L), kAxisBlocks);
        a.C = sp.C;
        a.S = sp.S;
        a.ncb = sp.ncb;
        blocks[np] = (unsigned)sp.blocks;
        a.vec = a.ncols % 2 == 0 && a.C % 2 == 0 && (((uintptr_t)a.src | (uintptr_t)a.dst) & 15) == 0 ? 1 : 0;
        // fftshift: input row n sits at position n + L/2; ifftshift: output row n is index n + L/2
        a.in_off = sh.pre ? a.L / 2 : 0;
        a.out_off = sh.post ? a.L / 2 : 0;
        a.sign = fwd ? -1.0f : 1.0f;
        a.scale = 1.0f;
        a.mask = nullptr;
        a.mask_div = sh.mask_batch > 1 ? 1 : sh.batch;
        a.tw = t->tw;
        a.pinv = t->pinv;
        const size_t lds = col_lds(a.L, a.C * a.S, a.st.dbl);
        if (lds > kAxisLdsMax) { // long lines with a second buffer
            const hipError_t e = hipFuncSetAttribute(a.st.gen ? (const void *)k_fft_axis<true> : (const void *)k_fft_axis<false>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return hip_fail(e, "FFT axis pass");
        }
        slabs *= n;
        ++np;
    }
    pass[np - 1].scale = sh.scale;
    pass[np - 1].mask = sh.mask;
    for (int k = 0; k < np; ++k) {
        const AxisArgs &a = pass[k];
        hipLaunchKernelGGL(a.st.gen ? k_fft_axis<true> : k_fft_axis<false>, dim3(blocks[k]), dim3(kAxisThreads),
                           col_lds(a.L, a.C * a.S, a.st.dbl), st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, "FFT axis pass");
    }
    return GN_OK;
}

int cfft_plan(int rank, const int64_t *n, int64_t batch, bool forward, CPlan **out)
{
    static std::once_flag once;
    std::call_once(once, []() { rocfft_setup(); });
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto key = std::make_tuple(dev, rank, n[0], rank > 1 ? n[1] : 1, rank > 2 ? n[2] : 1, batch, forward ? 1 : 0, 0);
    auto it = g_cfft_plans.find(key);
    if (it != g_cfft_plans.end()) {
        *out = &it->second;
        return GN_OK;
    }
    size_t lengths[3], strides[3];
    for (int a = 0; a < rank; ++a) lengths[a] = (size_t)n[rank - 1 - a]; // fastest first
    strides[0] = (size_t)batch;
    for (int a = 1; a < rank; ++a) strides[a] = strides[a - 1] * lengths[a - 1];
    rocfft_plan_description desc = nullptr;
    rocfft_status s = rocfft_plan_description_create(&desc);
    if (s != rocfft_status_success) return fail(GN_EROCFFT, "rocFFT description");
    s = rocfft_plan_description_set_data_layout(desc, rocfft_array_type_complex_interleaved,
                                                rocfft_array_type_complex_interleaved, nullptr, nullptr, rank, strides,
                                                1, rank, strides, 1);
    CPlan cp;
    if (s == rocfft_status_success)
        s = rocfft_plan_create(&cp.plan, rocfft_placement_inplace,
                               forward ? rocfft_transform_type_complex_forward : rocfft_transform_type_complex_inverse,
                               rocfft_precision_single, rank, lengths, (size_t)batch, desc);
    rocfft_plan_description_destroy(desc);
    if (s != rocfft_status_success) return fail(GN_EROCFFT, "rocFFT plan create (Cartesian FFT)");
    size_t wsz = 0;
    rocfft_plan_get_work_buffer_size(cp.plan, &wsz);
    if ((s = rocfft_execution_info_create(&cp.info)) != rocfft_status_success)
        return fail(GN_EROCFFT, "rocFFT execution info");
    if (wsz) {
        if (hipMalloc(&cp.work, wsz) != hipSuccess) return fail(GN_ENOMEM, "hipMalloc failed for the rocFFT work buffer");
        if (rocfft_execution_info_set_work_buffer(cp.info, cp.work, wsz) != rocfft_status_success)
            return fail(GN_EROCFFT, "rocFFT work buffer");
    }
    auto ins = g_cfft_plans.emplace(key, cp);
    *out = &ins.first->second;
    return GN_OK;
}

} // namespace
} // namespace gn

using namespace gn;

extern "C" {

int gn_fft_c2c(int rank, const int64_t *shape, int64_t batch, int direction, int flags, const float *mask,
               int64_t mask_batch, const void *in, void *out, void *stream)
{
    set_error("");
    if (rank < 1 || rank > 3 || !shape || batch < 1 || !in || !out)
        return fail(GN_EINVAL, "gn_fft_c2c: bad arguments");
    if (direction != GN_FFT_FORWARD && direction != GN_FFT_INVERSE) return fail(GN_EINVAL, "gn_fft_c2c: direction");
    if (mask && mask_batch != 1 && mask_batch != batch) return fail(GN_EINVAL, "gn_fft_c2c: mask batch");
    ShiftArgs a;
    a.rank = rank;
    a.total = batch;
    for (int ax = 0; ax < 3; ++ax) a.n[ax] = ax < rank ? shape[ax] : 1;
    for (int ax = 0; ax < rank; ++ax) {
        if (shape[ax] < 1) return fail(GN_EINVAL, "gn_fft_c2c: non-positive length");
        a.total *= shape[ax];
    }
    a.batch = batch;
    a.pre = (flags & GN_FFT_SHIFT_IN) ? 1 : 0;
    a.post = (flags & GN_FFT_SHIFT_OUT) ? 1 : 0;
    const bool fwd = direction == GN_FFT_FORWARD;
    a.scale = fwd ? 1.0f : (float)(1.0 / (double)(a.total / batch));
    a.mask = mask;
    a.mask_batch = mask_batch;
    hipStream_t st = (hipStream_t)stream;
    std::lock_guard<std::mutex> g(g_cfft_mu);
    if (axis_passes_ok(rank, a.n, a.total, in, out)) {
        const int r = axis_passes(a, fwd, (const float2 *)in, (float2 *)out, st);
        if (r || (flags & GN_FFT_ASYNC)) return r;
        hipError_t e = hipStreamSynchronize(st);
        return e == hipSuccess ? GN_OK : hip_fail(e, "FFT synchronize");
    }
    CPlan *cp = nullptr;
    int rc = cfft_plan(rank, a.n, batch, fwd, &cp);
    if (rc) return rc;
    if (rocfft_execution_info_set_stream(cp->info, st) != rocfft_status_success)
        return fail(GN_EROCFFT, "rocFFT set stream");
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto &ws = g_cfft_ws[dev];
    const size_t bytes = (size_t)a.total * sizeof(float2);
    if (ws.second < bytes) {
        if (ws.first) {
            (void)hipStreamSynchronize(st);
            (void)hipFree(ws.first);
        }
        ws.first = nullptr;
        ws.second = 0;
        if (hipMalloc(&ws.first, bytes) != hipSuccess) return fail(GN_ENOMEM, "hipMalloc failed for the FFT workspace");
        ws.second = bytes;
    }
    float2 *w = (float2 *)ws.first;
    const int nb = (int)std::min<int64_t>((a.total + 255) / 256, 1 << 16);
    // input (shifted) into the workspace, transform in place, output (shifted, masked, scaled)
    hipLaunchKernelGGL(k_shift_copy, dim3(nb), dim3(256), 0, st, a, (const float2 *)in, w, 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "FFT pre-pass");
    void *buf[1] = {w};
    if (rocfft_execute(cp->plan, buf, nullptr, cp->info) != rocfft_status_success)
        return fail(GN_EROCFFT, "rocFFT execute (Cartesian FFT)");
    hipLaunchKernelGGL(k_shift_copy, dim3(nb), dim3(256), 0, st, a, (const float2 *)w, (float2 *)out, 1);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "FFT post-pass");
    // the workspace is shared by every call on this device: calls must not overlap
    e = hipStreamSynchronize(st);
    return e == hipSuccess ? GN_OK : hip_fail(e, "FFT synchronize");
}

} // extern "C"
