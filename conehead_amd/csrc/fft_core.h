// fft_core.h -- butterflies of the FFT passes, and the beams, block orders,
// line pairs and support flags of a launch, shared by the general passes
// (spectral.hip) and the two-stage passes (fft_pair.h).
#pragma once

#include "ch_internal.h"

namespace ch {

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b)
{
    return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b)
{
    return make_float2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ float2 cscale(float2 a, float s)
{
    return make_float2(a.x * s, a.y * s);
}
// -i * a for the forward transform, +i * a for the inverse
template <bool INV>
__device__ __forceinline__ float2 rot(float2 a)
{
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <bool INV>
__device__ __forceinline__ void dft2(float2& a, float2& b)
{
    const float2 t = a;
    a = cadd(t, b);
    b = csub(t, b);
}

template <bool INV>
__device__ __forceinline__ void dft4(float2& a, float2& b, float2& c,
                                     float2& d)
{
    const float2 t0 = cadd(a, c), t1 = csub(a, c);
    const float2 t2 = cadd(b, d), t3 = rot<INV>(csub(b, d));
    a = cadd(t0, t2);
    c = csub(t0, t2);
    b = cadd(t1, t3);
    d = csub(t1, t3);
}

// dft4 of (a, b, 0, 0), c and d not read: a + c and b + d are a and b, so
// every nonzero output has the bits dft4 gives it (only the sign of an
// exact zero may differ).
template <bool INV>
__device__ __forceinline__ void dft4h(float2& a, float2& b, float2& c,
                                      float2& d)
{
    const float2 t3 = rot<INV>(b);
    c = csub(a, b);
    d = csub(a, t3);
    const float2 a0 = a;
    a = cadd(a0, b);
    b = cadd(a0, t3);
}

// dft<INV, H>: the DFT of v in place.  H: the upper half v[R/2 ..] of an
// even-length v is zero and not read (the first layer of each
// decomposition drops its zero terms, as in dft4h).
template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[2])
{
    if (H)
        v[1] = v[0];
    else
        dft2<INV>(v[0], v[1]);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[4])
{
    if (H)
        dft4h<INV>(v[0], v[1], v[2], v[3]);
    else
        dft4<INV>(v[0], v[1], v[2], v[3]);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[8])
{
    // even and odd halves, then X[k] = E[k] + w^k O[k], X[k+4] = E - w^k O
    float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    if (H) {
        dft4h<INV>(e0, e1, e2, e3);
        dft4h<INV>(o0, o1, o2, o3);
    } else {
        dft4<INV>(e0, e1, e2, e3);
        dft4<INV>(o0, o1, o2, o3);
    }
    const float h = 0.70710678118654752f;
    // w^1 = (h, -h) forward, (h, h) inverse; w^3 = (-h, -h) / (-h, h)
    const float2 w1o = INV ? make_float2(h * (o1.x - o1.y), h * (o1.x + o1.y))
                           : make_float2(h * (o1.x + o1.y), h * (o1.y - o1.x));
    const float2 w2o = rot<INV>(o2);
    const float2 w3o = INV
                           ? make_float2(-h * (o3.x + o3.y), h * (o3.x - o3.y))
                           : make_float2(h * (o3.y - o3.x), -h * (o3.x + o3.y));
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, w1o);
    v[5] = csub(e1, w1o);
    v[2] = cadd(e2, w2o);
    v[6] = csub(e2, w2o);
    v[3] = cadd(e3, w3o);
    v[7] = csub(e3, w3o);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[3])
{
    static_assert(!H, "odd length");
    const float s3 = 0.86602540378443865f;  // sin(pi / 3)
    const float2 t1 = cadd(v[1], v[2]);
    const float2 t2 = csub(v[0], cscale(t1, 0.5f));
    const float2 t3 = rot<INV>(cscale(csub(v[1], v[2]), s3));
    v[0] = cadd(v[0], t1);
    v[1] = cadd(t2, t3);
    v[2] = csub(t2, t3);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[5])
{
    static_assert(!H, "odd length");
    const float c1 = 0.30901699437494742f;   // cos(2 pi / 5)
    const float c2 = -0.80901699437494742f;  // cos(4 pi / 5)
    const float s1 = 0.95105651629515357f;   // sin(2 pi / 5)
    const float s2 = 0.58778525229247313f;   // sin(4 pi / 5)
    const float2 a = v[0];
    const float2 sbe = cadd(v[1], v[4]), dbe = csub(v[1], v[4]);
    const float2 scd = cadd(v[2], v[3]), dcd = csub(v[2], v[3]);
    const float2 a1 = cadd(a, cadd(cscale(sbe, c1), cscale(scd, c2)));
    const float2 a2 = cadd(a, cadd(cscale(sbe, c2), cscale(scd, c1)));
    const float2 b1 = rot<INV>(cadd(cscale(dbe, s1), cscale(dcd, s2)));
    const float2 b2 = rot<INV>(csub(cscale(dbe, s2), cscale(dcd, s1)));
    v[0] = cadd(a, cadd(sbe, scd));
    v[1] = cadd(a1, b1);
    v[4] = csub(a1, b1);
    v[2] = cadd(a2, b2);
    v[3] = csub(a2, b2);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[16])
{
    // 4 x 4: DFT4 over n1 of x[4 n1 + n2], twiddle W16^(n2 k1), DFT4 over
    // n2, output k1 + 4 k2
    const float c8 = 0.92387953251128674f, s8 = 0.38268343236508977f;
    const float h = 0.70710678118654752f;
    const float sg = INV ? 1.0f : -1.0f;
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        if (H)
            dft4h<INV>(v[n2], v[4 + n2], v[8 + n2], v[12 + n2]);
        else
            dft4<INV>(v[n2], v[4 + n2], v[8 + n2], v[12 + n2]);
    }
    // after this v[n2 + 4 k1] holds y[n2][k1]; W16^m = (cos, sg sin)
    const float2 w1 = make_float2(c8, sg * s8), w2 = make_float2(h, sg * h),
                 w3 = make_float2(s8, sg * c8), w6 = make_float2(-h, sg * h),
                 w9 = make_float2(-c8, -sg * s8);
    v[1 + 4] = cmul(v[1 + 4], w1);
    v[1 + 8] = cmul(v[1 + 8], w2);
    v[1 + 12] = cmul(v[1 + 12], w3);
    v[2 + 4] = cmul(v[2 + 4], w2);
    v[2 + 8] = rot<INV>(v[2 + 8]);
    v[2 + 12] = cmul(v[2 + 12], w6);
    v[3 + 4] = cmul(v[3 + 4], w3);
    v[3 + 8] = cmul(v[3 + 8], w6);
    v[3 + 12] = cmul(v[3 + 12], w9);
    float2 o[16];
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        float2 a = v[4 * k1], b = v[4 * k1 + 1], c = v[4 * k1 + 2],
               d = v[4 * k1 + 3];
        dft4<INV>(a, b, c, d);
        o[k1] = a;
        o[k1 + 4] = b;
        o[k1 + 8] = c;
        o[k1 + 12] = d;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
        v[i] = o[i];
}

// 9 = 3 x 3: DFT3 over n1 of x[3 n1 + n2], twiddle W9^(n2 k1), DFT3 over
// n2, output k1 + 3 k2.
template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[9])
{
    static_assert(!H, "odd length");
    // W9^m = (cos, -sin) forward, (cos, sin) inverse, at m = n2 k1
    constexpr float c[5] = {
        1.0f, 0.76604444311897801f, 0.17364817766693041f,
        -0.49999999999999978f, -0.93969262078590832f};
    constexpr float s[5] = {
        0.0f, 0.64278760968653925f, 0.98480775301220802f,
        0.86602540378443871f, 0.34202014332566888f};
    float2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
        float2 u[3];
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1)
            u[n1] = v[3 * n1 + n2];
        dft<INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            const int m = n2 * k1;
            t[k1][n2] = m == 0 ? u[k1]
                               : cmul(u[k1], make_float2(c[m], INV ? s[m]
                                                                   : -s[m]));
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        dft<INV>(t[k1]);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2)
            v[k1 + 3 * k2] = t[k1][k2];
    }
}

// N = A B with A and B coprime: the index maps n = B a + A b and k = (k mod A,
// k mod B) turn the DFT into A- and B-point ones without twiddles.  Zero
// inputs given as constants fold away (the two-stage passes are compiled
// without signed zeros).
template <int A, int B, bool INV>
__device__ __forceinline__ void dft_coprime(float2 (&v)[A * B])
{
    constexpr int N = A * B;
    float2 t[A][B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        float2 u[A];
#pragma unroll
        for (int a = 0; a < A; ++a)
            u[a] = v[(B * a + A * b) % N];
        dft<INV>(u);
#pragma unroll
        for (int k = 0; k < A; ++k)
            t[k][b] = u[k];
    }
#pragma unroll
    for (int k = 0; k < A; ++k)
        dft<INV>(t[k]);
#pragma unroll
    for (int k = 0; k < N; ++k)
        v[k] = t[k % A][k % B];
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[10])
{
    dft_coprime<2, 5, INV>(v);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[12])
{
    dft_coprime<4, 3, INV>(v);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[15])
{
    dft_coprime<3, 5, INV>(v);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[18])
{
    dft_coprime<2, 9, INV>(v);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[20])
{
    dft_coprime<4, 5, INV>(v);
}

template <bool INV, bool H = false>
__device__ __forceinline__ void dft(float2 (&v)[24])
{
    dft_coprime<8, 3, INV>(v);
}

// The beams of one launch: TERMA and dose grids from device tables (a
// batch) or one pointer each (a single beam); work grid b at a_beam * b.
// Workgroups take blockIdx.x = group * n_beams + beam, so consecutive
// workgroups are the same columns of different beams (K^ chunks are read
// once per launch from HBM and then from L2).
struct BeamIO {
    const float* t;
    float* d;
    const float* const* t_tab;
    float* const* d_tab;
    const int32_t* acc_tab;
    int32_t accumulate;
    int32_t n_beams;
    int64_t a_beam;
};

__device__ __forceinline__ int beam_of_block(const BeamIO& io)
{
    return (int)(blockIdx.x % (unsigned)io.n_beams);
}
__device__ __forceinline__ int group_of_block(const BeamIO& io)
{
    return (int)(blockIdx.x / (unsigned)io.n_beams);
}

// Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has
// its own L2.  The y passes take their work in XCD-major order instead:
// XCD k runs a contiguous range of logical blocks, so the two halves of a
// 128-byte line (neighbouring 8-column groups) meet in one L2.  The work
// per block is uniform, so the ranges stay balanced.
constexpr unsigned kXcds = 8;
struct BlockXY {
    unsigned x, y;
};
__device__ __forceinline__ BlockXY xcd_major_block(bool on)
{
    const unsigned nx = gridDim.x, total = gridDim.x * gridDim.y;
    unsigned l = blockIdx.x + nx * blockIdx.y;
    if (on && total % kXcds == 0)
        l = (l % kXcds) * (total / kXcds) + l / kXcds;
    BlockXY b;
    b.x = l % nx;
    b.y = l / nx;
    return b;
}

// Line pair w of a z-pass workgroup: lines (x, y) and (x, y + 1) of the
// grid, y even; valid = false past the last pair.
struct LinePair {
    int64_t x;
    int32_t y;
    bool valid;
};
__device__ __forceinline__ LinePair line_pair(int64_t p, int32_t X,
                                              int32_t Y)
{
    const int Yp = (Y + 1) / 2;
    LinePair lp;
    lp.valid = p < (int64_t)X * Yp;
    lp.x = lp.valid ? p / Yp : 0;
    lp.y = lp.valid ? 2 * (int)(p - lp.x * Yp) : 0;
    return lp;
}

// Zero support of a beam's work grid, so the forward passes skip what is
// zero: z_fwd records per line pair whether it holds a nonzero value (and
// writes the pair's spectra only then); the forward y pass reads those
// flags, skips a slab whose pairs are all zero (recording it in the slab
// flags) and reads only the nonzero rows of the others; the convolution
// pass reads only the rows x of nonzero slabs.  The flags are int32 at
// `off` (complex points after the beam's work grid): X * yp pair flags
// (pair p = x * yp + y / 2), then X slab flags at xyp = X * yp.  off < 0:
// no flags (every row is read).
struct Support {
    int64_t off;
    int32_t yp, xyp;
};
constexpr int kMaxFlagRows = 512;   // pairs per slab and slabs (X) with flags

__host__ __device__ __forceinline__ Support no_support()
{
    Support sp;
    sp.off = -1;
    sp.yp = sp.xyp = 0;
    return sp;
}

}  // namespace ch
