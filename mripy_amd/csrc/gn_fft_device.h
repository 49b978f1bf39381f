// In-LDS mixed-radix FFT of many lines, shared by the pruned NUFFT passes (gn_fft.hip)
// and the Cartesian FFTs (gn_cfft.hip): butterflies, stage loop, table staging, and
// the streaming 16-byte accesses.
#pragma once

#include <hip/hip_runtime.h>

#include "gn_host_plan.h"
#include "gn_internal.h"

namespace gn {
namespace {

// Streaming 16-byte accesses: every grid element a pass reads or writes is touched
// once per pass and the next pass runs over the whole grid, so the column passes load
// and store, and pass A' loads its grid lines and stores its image pairs, with the
// nontemporal hint (measured at 128^3 x 8 coils: fwd+adj 2.54 -> 2.39 ms).  Pass A's
// 8-byte grid stores, the spread's tile stores and the gather's sample stores were
// slower with it.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load_stream(const float2 *p)
{
    const f32x4_t t = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t *>(p));
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ void store_stream(float2 *p, float4 v)
{
    const f32x4_t t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x4_t *>(p));
}

__device__ inline float2 cmul(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ inline float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// multiply by (sign * i)
__device__ inline float2 mul_si(float2 a, float s) { return make_float2(-s * a.y, s * a.x); }

// Radix-R DFT of v[0..R) in registers (e^{sign 2 pi i / R} roots): v[k] becomes
// output k.
template <int R>
__device__ __forceinline__ void dft_small(float2 *v, float sign)
{
    if (R == 2) {
        const float2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if (R == 4) {
        const float2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const float2 s13 = cadd(v[1], v[3]), d13 = mul_si(csub(v[1], v[3]), sign);
        v[0] = cadd(s02, s13);
        v[1] = cadd(d02, d13);
        v[2] = csub(s02, s13);
        v[3] = csub(d02, d13);
    } else if (R == 3) {
        const float c1 = -0.5f, s1 = 0.86602540378443864676f * sign;
        const float2 a = cadd(v[1], v[2]), b = csub(v[1], v[2]);
        const float2 m = make_float2(v[0].x + c1 * a.x, v[0].y + c1 * a.y);
        const float2 r = make_float2(-s1 * b.y, s1 * b.x);
        v[0] = cadd(v[0], a);
        v[1] = cadd(m, r);
        v[2] = csub(m, r);
    } else if (R == 8) {
        // X[m] = E[m] + w^m O[m], X[m + 4] = E[m] - w^m O[m]: E, O the 4-point DFTs of
        // the even and odd inputs, w = e^{sign 2 pi i / 8}
        const float2 s04 = cadd(v[0], v[4]), d04 = csub(v[0], v[4]);
        const float2 s26 = cadd(v[2], v[6]), d26 = mul_si(csub(v[2], v[6]), sign);
        const float2 e0 = cadd(s04, s26), e1 = cadd(d04, d26), e2 = csub(s04, s26), e3 = csub(d04, d26);
        const float2 s15 = cadd(v[1], v[5]), d15 = csub(v[1], v[5]);
        const float2 s37 = cadd(v[3], v[7]), d37 = mul_si(csub(v[3], v[7]), sign);
        const float2 o0 = cadd(s15, s37), o1 = cadd(d15, d37), o2 = csub(s15, s37), o3 = csub(d15, d37);
        const float r2 = 0.70710678118654752440f;
        // w^1 = (1 + sign i) / sqrt 2, w^2 = sign i, w^3 = (-1 + sign i) / sqrt 2
        const float2 t1 = make_float2(r2 * (o1.x - sign * o1.y), r2 * (o1.y + sign * o1.x));
        const float2 t2 = mul_si(o2, sign);
        const float2 t3 = make_float2(r2 * (-o3.x - sign * o3.y), r2 * (-o3.y + sign * o3.x));
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, t1);
        v[5] = csub(e1, t1);
        v[2] = cadd(e2, t2);
        v[6] = csub(e2, t2);
        v[3] = cadd(e3, t3);
        v[7] = csub(e3, t3);
    } else if (R == 5) {
        const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
        const float s1 = 0.95105651629515357212f * sign, s2 = 0.58778525229247312917f * sign;
        const float2 a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]);
        const float2 a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
        const float2 m1 = make_float2(v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y);
        const float2 m2 = make_float2(v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y);
        // r1 = i (s1 b1 + s2 b2), r2 = i (s2 b1 - s1 b2)
        const float2 r1 = make_float2(-(s1 * b1.y + s2 * b2.y), s1 * b1.x + s2 * b2.x);
        const float2 r2 = make_float2(-(s2 * b1.y - s1 * b2.y), s2 * b1.x - s1 * b2.x);
        v[0] = cadd(v[0], cadd(a1, a2));
        v[1] = cadd(m1, r1);
        v[4] = csub(m1, r1);
        v[2] = cadd(m2, r2);
        v[3] = csub(m2, r2);
    }
}

// cos / sin of 2 pi k / R for the prime register butterflies, correctly rounded.
template <int R>
struct PrimeRoots;
template <>
struct PrimeRoots<7> {
    static constexpr float c[4] = {1.0f, 0.62348980185873359f, -0.22252093395631434f, -0.90096886790241903f};
    static constexpr float s[4] = {0.0f, 0.7818314824680298f, 0.97492791218182362f, 0.43388373911755823f};
};
template <>
struct PrimeRoots<11> {
    static constexpr float c[6] = {1.0f, 0.84125353283118121f, 0.41541501300188644f, -0.142314838273285f, -0.65486073394528499f, -0.95949297361449737f};
    static constexpr float s[6] = {0.0f, 0.54064081745559756f, 0.90963199535451833f, 0.9898214418809328f, 0.75574957435425827f, 0.28173255684142967f};
};
template <>
struct PrimeRoots<13> {
    static constexpr float c[7] = {1.0f, 0.88545602565320991f, 0.56806474673115592f, 0.12053668025532301f, -0.35460488704253545f, -0.74851074817110119f, -0.97094181742605201f};
    static constexpr float s[7] = {0.0f, 0.46472317204376851f, 0.82298386589365635f, 0.99270887409805397f, 0.93501624268541483f, 0.66312265824079519f, 0.23931566428755768f};
};

// Radix-R butterfly for an odd prime R on LDS elements base + k * qstride (arguments as
// butterfly below).  The inputs j and R - j enter as their sum and difference, so each
// output pair (k, R - k) takes (R - 1) / 2 real products of each; an output pair is
// stored as soon as it is formed and the twiddles of a second line are read again, which
// keeps the kernels near 64 registers.
template <int R, bool TW, int NL>
__device__ __forceinline__ void butterfly_prime(float2 *buf, int base, int qstride, int lstep, const float2 *tw,
                                                int twstep, int t, float sign)
{
    constexpr int H = (R - 1) / 2;
#pragma unroll 1
    for (int l = 0; l < NL; ++l) {
        float2 *x = buf + base + l * lstep;
        const float2 x0 = x[0];
        float2 s[H + 1], d[H + 1], sum = x0;
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            float2 u = x[j * qstride], v = x[(R - j) * qstride];
            if (TW) {
                u = cmul(u, tw[t * j * twstep]);
                v = cmul(v, tw[t * (R - j) * twstep]);
            }
            s[j] = cadd(u, v);
            d[j] = csub(u, v);
            sum = cadd(sum, s[j]);
        }
        x[0] = sum;
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            float2 a = x0, b = make_float2(0.f, 0.f);
#pragma unroll
            for (int j = 1; j <= H; ++j) {
                const int m = (j * k) % R;
                const float c = PrimeRoots<R>::c[m > H ? R - m : m];
                const float q = m > H ? -PrimeRoots<R>::s[R - m] : PrimeRoots<R>::s[m];
                a.x += s[j].x * c;
                a.y += s[j].y * c;
                b.x += d[j].x * q;
                b.y += d[j].y * q;
            }
            const float2 r = make_float2(-sign * b.y, sign * b.x);
            x[k * qstride] = cadd(a, r);
            x[(R - k) * qstride] = csub(a, r);
        }
    }
}

// One radix-r butterfly on LDS elements at base + k*qstride (k < r) of a line, after
// twiddling element k by w_g^{t k}: tw[(t k L / g)] (the table in LDS already holds
// the twiddles of this transform's sign).  TW = false for the first stage (g = r, all
// twiddles 1).  Otherwise every element is multiplied, t = 0 included (tw[0] = 1 and
// x * 1 - y * 0 = x exactly), so the lanes of a wave take no per-element branches.
// NL = 2: the same butterfly on two lines (elements base + k*qstride and lstep after
// them), which share the index arithmetic and the twiddle reads.
template <int R, bool TW, int NL>
__device__ __forceinline__ void butterfly(float2 *buf, int base, int qstride, int lstep, const float2 *tw, int twstep,
                                          int t, float sign)
{
    float2 w[R];
    if (TW) {
#pragma unroll
        for (int k = 1; k < R; ++k) w[k] = tw[t * k * twstep];
    }
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        float2 v[R];
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = buf[base + k * qstride + l * lstep];
        if (TW) {
#pragma unroll
            for (int k = 1; k < R; ++k) v[k] = cmul(v[k], w[k]);
        }
        dft_small<R>(v, sign);
#pragma unroll
        for (int k = 0; k < R; ++k) buf[base + k * qstride + l * lstep] = v[k];
    }
}

// floor(n / d) for 0 <= n < 2^22, 1 <= d <= 2^12, with r = 1/d: the float estimate
// is within one of the quotient, and one correction step each way makes it exact.
__device__ inline int fdiv(int n, int d, float r)
{
    int q = (int)((float)n * r);
    q -= (q * d > n) ? 1 : 0;
    q += ((q + 1) * d <= n) ? 1 : 0;
    return q;
}

// A stage of odd prime radix r > kFFTRadixMax by direct sums on the matrix cores, from buf
// into alt.  First every input pair (m, r - m) of a butterfly is twiddled and replaced by
// its sum s_m and difference d_m in place; then
//     X_k, X_{r-k} = x0 + sum_m c_mk s_m  +-  i sum_m s_mk d_m,   k = 0 .. h = (r - 1) / 2,
// c and s the real and imaginary parts of w_r^{mk} from the twiddle table: two real
// products (outputs k) x (pairs m) x (columns: re and im of every butterfly of every line).
// A wave takes 16 outputs and CT groups of 16 columns, with one v_mfma_f32_16x16x4_f32
// per product, column group and 4 pairs; one table read (both parts) feeds 2 CT products.
// Lane layout as in the matrix-core spread: A[i][k] and B[k][j] in lanes i + 16 k and
// j + 16 k, D[4 g + v][j] in register v of lane j + 16 g.  The sums are folded every
// kPrimeFold steps (16 pairs), which keeps the rounding error of 125 terms at that of a
// Bluestein transform.  Bound by the matrix cores ((r - 1)^2 / 2 FP32 products per complex
// point); as plain FMAs it was bound by LDS reads and index arithmetic: 226^3 x 4, pad +
// FFT of a type 2: 0.86 ms, with the matrix cores 0.69 ms (pad pass + rocFFT: 1.97 ms).
typedef float prime_f32x4 __attribute__((ext_vector_type(4)));
constexpr int kPrimeFold = 4;
template <int CT>
__device__ __forceinline__ void prime_products(const float2 *buf, float2 *alt, int nlines, int lstride, int estride,
                                               int r, int q, int wstep, int nb, const float2 *tw)
{
    const int h = (r - 1) / 2, nu = nb * nlines; // columns / 2
    const int nkt = (h + 16) / 16, nct = (2 * nu + 16 * CT - 1) / (16 * CT);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    const float *in = (const float *)buf;
    float *out = (float *)alt;
    const int ms = 2 * q * estride; // floats between a butterfly's elements
    for (int unit = wave; unit < nkt * nct; unit += (int)(blockDim.x >> 6)) {
        const int ct = unit / nkt, kt = unit - ct * nkt;
        int at[CT];
        bool ok[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int col = (ct * CT + c) * 16 + j;
            ok[c] = col < 2 * nu;
            const int u = min(col >> 1, nu - 1);
            const int bidx = u / nlines, line = u - bidx * nlines;
            const int blk = bidx / q, t = bidx - blk * q;
            at[c] = 2 * (line * lstride + (blk * r * q + t) * estride) + (col & 1);
        }
        // table index of (output kt * 16 + j, pair m): m k mod r, stepped by 4 pairs
        // (outputs past h, up to 16 nkt - 1 < r, are computed and not stored)
        const int k = kt * 16 + j;
        const int step = (4 * k) % r;
        int w = ((1 + g) * k) % r;
        prime_f32x4 sc[CT], ss[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) sc[c] = ss[c] = prime_f32x4{0.f, 0.f, 0.f, 0.f};
        for (int m0 = 1; m0 <= h; m0 += 4 * kPrimeFold) {
            prime_f32x4 pc[CT], ps[CT];
#pragma unroll
            for (int c = 0; c < CT; ++c) pc[c] = ps[c] = prime_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int f = 0; f < kPrimeFold; ++f) {
                const int m = min(m0 + 4 * f + g, r - 1); // pairs past h get zero factors
                const bool on = m <= h;
                const float2 v = tw[w * wstep];
                const float cv = on ? v.x : 0.f, sv = on ? v.y : 0.f;
                w += step;
                if (w >= r) w -= r;
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const float s = in[at[c] + m * ms], d = in[at[c] + (r - m) * ms];
                    pc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(cv, s, pc[c], 0, 0, 0);
                    ps[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv, d, ps[c], 0, 0, 0);
                }
            }
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                sc[c] += pc[c];
                ss[c] += ps[c];
            }
        }
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const float x0 = in[at[c]];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // the other part of the same column pair (quad_perm [1, 0, 3, 2])
                const float o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(ss[c][v]), 0xb1, 0xf, 0xf, false));
                const float i = (j & 1) ? o : -o, x = x0 + sc[c][v];
                const int ko = kt * 16 + 4 * g + v;
                if (ok[c] && ko <= h) {
                    out[at[c] + ko * ms] = x + i;
                    if (ko) out[at[c] + (r - ko) * ms] = x - i;
                }
            }
        }
    }
}

__device__ __forceinline__ void prime_stage(float2 *buf, float2 *alt, int nlines, int lstride, int estride, int r, int q,
                                            int twstep, int nb, const float2 *tw)
{
    const int h = (r - 1) / 2;
    const float rnl = __builtin_amdgcn_rcpf((float)nlines), rh = __builtin_amdgcn_rcpf((float)h);
    for (int w = threadIdx.x; w < h * nb * nlines; w += blockDim.x) {
        const int i = fdiv(w, nlines, rnl), j = w - i * nlines;
        const int bidx = fdiv(i, h, rh), m = i - bidx * h + 1;
        const int blk = bidx / q, t = bidx - blk * q;
        const int base = j * lstride + (blk * r * q + t) * estride;
        float2 *pa = buf + base + m * q * estride, *pb = buf + base + (r - m) * q * estride;
        float2 a = *pa, b = *pb;
        if (t) {
            a = cmul(a, tw[t * m * twstep]);
            b = cmul(b, tw[t * (r - m) * twstep]);
        }
        *pa = cadd(a, b);
        *pb = csub(a, b);
    }
    __syncthreads();
    // two column groups per wave while that leaves a unit for every wave
    if (((h + 16) / 16) * ((nb * nlines + 15) / 16) >= (int)(blockDim.x >> 6))
        prime_products<2>(buf, alt, nlines, lstride, estride, r, q, q * twstep, nb, tw);
    else
        prime_products<1>(buf, alt, nlines, lstride, estride, r, q, q * twstep, nb, tw);
    __syncthreads();
}

// In-place FFT of `nlines` lines of length L held in LDS: element i of line j at
// buf[j * lstride + i * estride].  All threads of the block take part.  NL = 2 (nlines
// even): a thread takes the same butterfly on lines j and j + nlines / 2, so that the
// lanes of a wave still read consecutive lines in each of the two reads.  GEN: also the
// prime radices 7, 11, 13, and larger ones through alt, a second buffer of the same
// layout (st.dbl); returns the buffer that holds the result.  Without GEN that is buf,
// and the kernels keep the registers of the common lengths.
template <int NL, bool GEN>
__device__ __forceinline__ float2 *fft_lines(float2 *buf, float2 *alt, int nlines, int lstride, int estride, int L,
                                             const Stages &st, const float2 *tw, float sign)
{
    const int nw = nlines / NL; // line groups
    // fdiv corrects its quotient estimate, so approximate reciprocals suffice
    const float rl = __builtin_amdgcn_rcpf((float)nw);
    // power-of-two line counts and butterfly groups index with shifts
    const int lgl = (nw & (nw - 1)) == 0 ? __builtin_ctz(nw) : -1;
    for (int s = 0; s < st.n; ++s) {
        const int r = st.radix[s];
        const int q = st.q[s];         // butterfly span before this stage
        if (GEN && r > host::kFFTRadixMax) {
            prime_stage(buf, alt, nlines, lstride, estride, r, q, st.tws[s], st.nb[s], tw);
            float2 *o = buf;
            buf = alt;
            alt = o;
            continue;
        }
        const int g = r * q;
        const int twstep = st.tws[s];  // L / g
        const int nbl = st.nb[s] * nw; // butterflies of all line groups
        const float rq = __builtin_amdgcn_rcpf((float)q);
        const int lgq = (q & (q - 1)) == 0 ? __builtin_ctz(q) : -1;
        for (int w = threadIdx.x; w < nbl; w += blockDim.x) {
            // line groups fastest: neighbouring threads work on neighbouring lines
            const int bidx = lgl >= 0 ? (w >> lgl) : fdiv(w, nw, rl);
            const int j = w - bidx * nw;
            const int blk = lgq >= 0 ? (bidx >> lgq) : fdiv(bidx, q, rq);
            const int t = bidx - blk * q;
            const int base = j * lstride + (blk * g + t) * estride;
            if (s == 0) {
                switch (r) {
                case 2: butterfly<2, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 3: butterfly<3, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 4: butterfly<4, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 8: butterfly<8, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                default:
                    if constexpr (GEN) {
                        if (r == 7) {
                            butterfly_prime<7, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                        if (r == 11) {
                            butterfly_prime<11, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                        if (r == 13) {
                            butterfly_prime<13, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                    }
                    butterfly<5, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                    break;
                }
            } else {
                switch (r) {
                case 2: butterfly<2, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 3: butterfly<3, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 4: butterfly<4, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 8: butterfly<8, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                default:
                    if constexpr (GEN) {
                        if (r == 7) {
                            butterfly_prime<7, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                        if (r == 11) {
                            butterfly_prime<11, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                        if (r == 13) {
                            butterfly_prime<13, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                            break;
                        }
                    }
                    butterfly<5, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign);
                    break;
                }
            }
        }
        __syncthreads();
    }
    return buf;
}

// Stage the twiddles of a transform of this sign (the table holds e^{-2 pi i k/L}; sign
// -1 keeps it, +1 conjugates it) and the digit-reversal map of a length-n transform in
// LDS.  Both loads of an entry are issued before either is used.
__device__ inline void load_tables(float2 *tw_dst, int *pinv_dst, const float2 *tw, const int *pinv, int n, float sign)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float2 w = tw[i];
        const int q = pinv[i];
        tw_dst[i] = make_float2(w.x, -sign * w.y);
        pinv_dst[i] = q;
    }
}

} // namespace
} // namespace gn
