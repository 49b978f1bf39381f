// In-LDS mixed-radix FFT of many lines, shared by the pruned NUFFT passes (gn_fft.hip)
// and the Cartesian FFTs (gn_cfft.hip): butterflies, stage loop, table staging, and
// the streaming 16-byte accesses.
#pragma once

#include <hip/hip_runtime.h>

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

// In-place FFT of `nlines` lines of length L held in LDS: element i of line j at
// buf[j * lstride + i * estride].  All threads of the block take part.  NL = 2 (nlines
// even): a thread takes the same butterfly on lines j and j + nlines / 2, so that the
// lanes of a wave still read consecutive lines in each of the two reads.
template <int NL>
__device__ __forceinline__ void fft_lines(float2 *buf, int nlines, int lstride, int estride, int L, const Stages &st,
                                          const float2 *tw, float sign)
{
    const int nw = nlines / NL; // line groups
    // fdiv corrects its quotient estimate, so approximate reciprocals suffice
    const float rl = __builtin_amdgcn_rcpf((float)nw);
    // power-of-two line counts and butterfly groups index with shifts
    const int lgl = (nw & (nw - 1)) == 0 ? __builtin_ctz(nw) : -1;
    for (int s = 0; s < st.n; ++s) {
        const int r = st.radix[s];
        const int q = st.q[s];         // butterfly span before this stage
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
                default: butterfly<5, false, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                }
            } else {
                switch (r) {
                case 2: butterfly<2, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 3: butterfly<3, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 4: butterfly<4, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                case 8: butterfly<8, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                default: butterfly<5, true, NL>(buf, base, q * estride, nw * lstride, tw, twstep, t, sign); break;
                }
            }
        }
        __syncthreads();
    }
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
