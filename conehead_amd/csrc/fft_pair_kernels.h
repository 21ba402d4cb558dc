// fft_pair_kernels.h -- kernels and launches of the two-stage FFT passes
// (fft_pair.h), instantiated per frame length by fft_pair_*.hip.  Compiled
// without signed zeros, so the padded inputs' zero terms fold away.
#pragma once

#include "fft_pair.h"

namespace ch {
namespace {

template <int R1, int R2>
struct Pair {
    static_assert(R1 % 2 == 0, "half stages");
    static constexpr int F = R1 * R2;
    static constexpr int T = R1 > R2 ? R1 : R2;   // threads per line
    static constexpr int K = F / 2 + 1;           // half spectrum
    // twiddles kept in LDS; W^(m + F / 2) = -W^m gives the rest.  At 400
    // points the whole table would leave room for two workgroups of 16
    // lines per CU instead of three (LDS is granted in 1280-byte pieces).
    static constexpr int tw_len = F == 400 ? 224 : F;
    // z passes: pitch of a line's slots, (major, minor) at major * pitch +
    // minor with an odd pitch, so neighbouring threads hit different banks
    // whether they step the minor or the major index
    static constexpr int P2 = R2 | 1;             // forward: (r, j), j < R2
    static constexpr int P1 = R1 | 1;             // inverse: (r, j), j < R1
    static constexpr int fwd_line = R1 * P2 > F + 1 ? R1 * P2 : F + 1;
    static constexpr int inv_line = R2 * P1;
};

__device__ __forceinline__ void load_table(float2* s_tw, const float2* g,
                                           int F)
{
    for (int i = threadIdx.x; i < F; i += blockDim.x)
        s_tw[i] = g[i];
}

__device__ __forceinline__ const float2* at(const float2* base, uint32_t off)
{
    return (const float2*)((const char*)base + off);
}
__device__ __forceinline__ float2* at(float2* base, uint32_t off)
{
    return (float2*)((char*)base + off);
}

// v[r] *= W_F^(r j), conjugated for the inverse; j < F / R.
template <int R, bool INV, class P>
__device__ __forceinline__ void twiddle(float2 (&v)[R],
                                        const float2* __restrict__ tw, int j)
{
#pragma unroll
    for (int r = 1; r < R; ++r) {
        float2 t;
        if (r * (P::F / R - 1) < P::tw_len) {
            t = tw[r * j];
        } else {
            const bool far = r * j >= P::tw_len;
            t = tw[far ? r * j - P::F / 2 : r * j];
            t.x = far ? -t.x : t.x;
            t.y = far ? -t.y : t.y;
        }
        if (INV)
            t.y = -t.y;
        v[r] = cmul(v[r], t);
    }
}

// ------------------------------------------------------------ columns ----
// Slot (j, r) of column w: element ((j * R1 + (r ^ (j & 1))) * 16 + w.  The
// swap of neighbours on odd j puts the groups of 16 columns that neighbouring
// threads touch in different halves of the banks (R1 is even); it costs no
// instruction per access, since r even and r odd take one base each.
template <int R1>
struct Slots {
    float2* even;
    float2* odd;
    // thread j: its own slots (j, r), r < R1
    __device__ __forceinline__ Slots(float2* s, int j, int w)
    {
        const int p = j & 1;
        even = s + (j * R1 + p) * kPairLines + w;
        odd = s + (j * R1 - p) * kPairLines + w;
    }
    __device__ __forceinline__ float2& operator[](int r) const
    {
        return (r & 1 ? odd : even)[r * kPairLines];
    }
};
template <int R1>
struct SlotsAcross {
    float2* even;
    float2* odd;
    // thread j < R1: slots (r, j), r < R2
    __device__ __forceinline__ SlotsAcross(float2* s, int j, int w)
    {
        even = s + j * kPairLines + w;
        odd = s + (j ^ 1) * kPairLines + w;
    }
    __device__ __forceinline__ float2& operator[](int r) const
    {
        return (r & 1 ? odd : even)[r * R1 * kPairLines];
    }
};

struct ColThread {
    int w, j;
    bool ok;
};
__device__ __forceinline__ ColThread col_thread(int lw, int n_left)
{
    ColThread t;
    t.w = threadIdx.x & ((1 << lw) - 1);
    t.j = threadIdx.x >> lw;
    t.ok = t.w < n_left;
    return t;
}

constexpr int kMaxFlags = 512;

// The forward y transforms of slab blockIdx.y: rows n < n_in in, all F rows
// out.  With flags, a slab of zero pairs is skipped (its flag recorded) and
// zero rows are not read.
template <int R1, int R2>
__global__ __launch_bounds__((Pair<R1, R2>::T * kPairLines)) void pair_y_fwd(
    BeamIO io, float2* __restrict__ A, uint32_t row_stride,
    int64_t outer_stride, int32_t n_cols, int32_t n_in,
    const float2* __restrict__ g_tw, int32_t lw, Support sp)
{
    using P = Pair<R1, R2>;
    __shared__ float2 s_tw[P::tw_len];
    __shared__ float2 s_a[P::F * kPairLines];
    __shared__ uint8_t s_rows[kMaxFlags];
    const int beam = beam_of_block(io);
    const int k0 = group_of_block(io) << lw;
    float2* grid = A + beam * io.a_beam;
    const bool flagged = sp.off >= 0;
    if (flagged) {
        int32_t* flags = (int32_t*)(grid + sp.off);
        int any = 0;
        for (int i = threadIdx.x; i < sp.yp; i += blockDim.x) {
            const int32_t f = flags[(int64_t)blockIdx.y * sp.yp + i];
            s_rows[i] = (uint8_t)f;
            any |= f;
        }
        any = __syncthreads_or(any);
        if (threadIdx.x == 0)
            flags[sp.xyp + blockIdx.y] = any ? 1 : 0;
        if (!any)
            return;
    }
    load_table(s_tw, g_tw, P::tw_len);
    const ColThread t = col_thread(lw, n_cols - k0);
    float2* base = grid + blockIdx.y * outer_stride + k0;
    const uint32_t rs = row_stride * (uint32_t)sizeof(float2);
    const uint32_t off0 = t.j * rs + t.w * (uint32_t)sizeof(float2);
    if (t.j < R2) {
        float2 v[R1];
        bool nz[R1 / 2];
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r) {
            const int n = t.j + r * R2;
            nz[r] = t.ok && n < n_in && (!flagged || s_rows[n >> 1] != 0);
        }
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            v[r] = make_float2(0.0f, 0.0f);
            if (r < R1 / 2 && nz[r < R1 / 2 ? r : 0])
                v[r] = *at(base, off0 + r * R2 * rs);
        }
        dft<false>(v);
        const Slots<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R1; ++r)
            slot[r] = v[r];
    }
    __syncthreads();
    if (t.j < R1) {
        float2 v[R2];
        const SlotsAcross<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R2; ++r)
            v[r] = slot[r];
        twiddle<R2, false, P>(v, s_tw, t.j);
        dft<false>(v);
        if (t.ok) {
#pragma unroll
            for (int r = 0; r < R2; ++r)
                *at(base, off0 + r * R1 * rs) = v[r];
        }
    }
}

// The inverse y transforms of slab blockIdx.y: all F rows in, rows n <
// n_out <= F / 2 out.
template <int R1, int R2>
__global__ __launch_bounds__((Pair<R1, R2>::T * kPairLines)) void pair_y_inv(
    BeamIO io, float2* __restrict__ A, uint32_t row_stride,
    int64_t outer_stride, int32_t n_cols, int32_t n_out,
    const float2* __restrict__ g_tw, int32_t lw)
{
    using P = Pair<R1, R2>;
    __shared__ float2 s_tw[P::tw_len];
    __shared__ float2 s_a[P::F * kPairLines];
    const int beam = beam_of_block(io);
    const int k0 = group_of_block(io) << lw;
    load_table(s_tw, g_tw, P::tw_len);
    const ColThread t = col_thread(lw, n_cols - k0);
    float2* base = A + beam * io.a_beam + blockIdx.y * outer_stride + k0;
    const uint32_t rs = row_stride * (uint32_t)sizeof(float2);
    const uint32_t off0 = t.j * rs + t.w * (uint32_t)sizeof(float2);
    if (t.j < R1) {
        float2 v[R2];
#pragma unroll
        for (int r = 0; r < R2; ++r) {
            v[r] = make_float2(0.0f, 0.0f);
            if (t.ok)
                v[r] = *at(base, off0 + r * R1 * rs);
        }
        dft<true>(v);
        const SlotsAcross<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R2; ++r)
            slot[r] = v[r];
    }
    __syncthreads();
    if (t.j < R2) {
        float2 v[R1];
        const Slots<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R1; ++r)
            v[r] = slot[r];
        twiddle<R1, true, P>(v, s_tw, t.j);
        dft<true>(v);
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r)
            if (t.ok && t.j + r * R2 < n_out)
                *at(base, off0 + r * R2 * rs) = v[r];
    }
}

// x transforms of row blockIdx.y of the frame, times K^, inverse x
// transforms; rows x < n_in in and out.  With flags, zero slabs are not
// read.
template <int R1, int R2>
__global__ __launch_bounds__((Pair<R1, R2>::T * kPairLines)) void pair_conv(
    BeamIO io, float2* __restrict__ A, uint32_t row_stride,
    int64_t outer_stride, int32_t n_cols, int32_t n_in,
    const float2* __restrict__ g_tw, const float2* __restrict__ khat,
    uint32_t k_row_stride, int64_t k_outer_stride, int32_t lw, Support sp)
{
    using P = Pair<R1, R2>;
    __shared__ float2 s_tw[P::tw_len];
    __shared__ float2 s_a[P::F * kPairLines];
    const int beam = beam_of_block(io);
    const int k0 = group_of_block(io) << lw;
    float2* grid = A + beam * io.a_beam;
    const int32_t* flags =
        sp.off >= 0 ? (const int32_t*)(grid + sp.off) + sp.xyp : nullptr;
    load_table(s_tw, g_tw, P::tw_len);
    const ColThread t = col_thread(lw, n_cols - k0);
    float2* base = grid + blockIdx.y * outer_stride + k0;
    const float2* kb = khat + blockIdx.y * k_outer_stride + k0;
    const uint32_t rs = row_stride * (uint32_t)sizeof(float2);
    const uint32_t krs = k_row_stride * (uint32_t)sizeof(float2);
    const uint32_t off0 = t.j * rs + t.w * (uint32_t)sizeof(float2);
    if (t.j < R2) {
        float2 v[R1];
        bool nz[R1 / 2];
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r) {
            const int n = t.j + r * R2;
            nz[r] = t.ok && n < n_in;
            if (flags && nz[r])
                nz[r] = flags[n] != 0;
        }
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            v[r] = make_float2(0.0f, 0.0f);
            if (r < R1 / 2 && nz[r < R1 / 2 ? r : 0])
                v[r] = *at(base, off0 + r * R2 * rs);
        }
        dft<false>(v);
        const Slots<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R1; ++r)
            slot[r] = v[r];
    }
    // K^ while the other wavefronts finish
    float2 kv[R2];
    if (t.j < R1) {
        const uint32_t koff = t.j * krs + t.w * (uint32_t)sizeof(float2);
#pragma unroll
        for (int r = 0; r < R2; ++r) {
            kv[r] = make_float2(0.0f, 0.0f);
            if (t.ok)
                kv[r] = *at(kb, koff + r * R1 * krs);
        }
    }
    __syncthreads();
    if (t.j < R1) {
        float2 v[R2];
        const SlotsAcross<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R2; ++r)
            v[r] = slot[r];
        twiddle<R2, false, P>(v, s_tw, t.j);
        dft<false>(v);
#pragma unroll
        for (int r = 0; r < R2; ++r)
            v[r] = cmul(v[r], kv[r]);
        dft<true>(v);
        // back to the slots this thread alone has read
#pragma unroll
        for (int r = 0; r < R2; ++r)
            slot[r] = v[r];
    }
    __syncthreads();
    if (t.j < R2) {
        float2 v[R1];
        const Slots<R1> slot(s_a, t.j, t.w);
#pragma unroll
        for (int r = 0; r < R1; ++r)
            v[r] = slot[r];
        twiddle<R1, true, P>(v, s_tw, t.j);
        dft<true>(v);
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r)
            if (t.ok && t.j + r * R2 < n_in)
                *at(base, off0 + r * R2 * rs) = v[r];
    }
}

// ------------------------------------------------------------ z lines ----

// Two real z lines of T as one complex line (z_fwd_kernel's pairing,
// spectra and flags).  Line pair w = tid / T of the workgroup.
template <int R1, int R2>
__global__ __launch_bounds__((Pair<R1, R2>::T * kPairLines)) void pair_z_fwd(
    BeamIO io, float2* __restrict__ A, int32_t X, int32_t Y, int32_t Z,
    int32_t a_rows, int32_t kp, const float2* __restrict__ g_tw, int32_t W,
    Support sp)
{
    using P = Pair<R1, R2>;
    __shared__ float2 s_tw[P::tw_len];
    __shared__ float2 s_a[P::fwd_line * kPairLines];
    __shared__ int32_t s_vote[kPairLines];
    if (threadIdx.x < kPairLines)
        s_vote[threadIdx.x] = 0;
    load_table(s_tw, g_tw, P::tw_len);
    __syncthreads();
    const int beam = beam_of_block(io);
    const float* __restrict__ T = io.t_tab ? io.t_tab[beam] : io.t;
    A += beam * io.a_beam;
    const int w = threadIdx.x / P::T, j = threadIdx.x - w * P::T;
    const int64_t pair = (int64_t)group_of_block(io) * W + w;
    const LinePair lp = line_pair(pair, X, Y);
    const bool two = lp.y + 1 < Y;
    const float* row = T + (lp.x * Y + lp.y) * (int64_t)Z;
    float2* out = A + (lp.x * a_rows + lp.y) * (int64_t)kp;
    int32_t* flags = sp.off >= 0 ? (int32_t*)(A + sp.off) : nullptr;
    float2* line = s_a + w * P::fwd_line;
    if (j < R2) {
        float2 v[R1];
        bool nz = false;
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            v[r] = make_float2(0.0f, 0.0f);
            const int n = j + r * R2;
            if (r < R1 / 2 && lp.valid && n < Z) {
                v[r].x = row[n];
                if (two)
                    v[r].y = row[Z + n];
                nz = nz || v[r].x != 0.0f || v[r].y != 0.0f;
            }
        }
        if (nz)
            s_vote[w] = 1;
        dft<false>(v);
#pragma unroll
        for (int r = 0; r < R1; ++r)
            line[r * P::P2 + j] = v[r];
    }
    __syncthreads();
    const bool keep = !flags || s_vote[w] != 0;
    if (flags) {
        if (lp.valid && j == 0)
            flags[pair] = keep ? 1 : 0;
        int any = 0;
        for (int q = 0; q < kPairLines; ++q)
            any |= s_vote[q];
        if (!any)
            return;  // workgroup-uniform
    }
    float2 v[R2];
    if (j < R1) {
#pragma unroll
        for (int r = 0; r < R2; ++r)
            v[r] = line[j * P::P2 + r];
        twiddle<R2, false, P>(v, s_tw, j);
        dft<false>(v);
    }
    __syncthreads();
    if (j < R1) {
#pragma unroll
        for (int r = 0; r < R2; ++r)
            line[j + r * R1] = v[r];
    }
    __syncthreads();
    if (!lp.valid || !keep)
        return;
#pragma unroll
    for (int i = 0; i < (P::K + P::T - 1) / P::T; ++i) {
        const int k = j + i * P::T;
        if (k >= P::K)
            break;
        const float2 c = line[k];
        const float2 cm = line[k == 0 ? 0 : P::F - k];
        out[k] = make_float2(0.5f * (c.x + cm.x), 0.5f * (c.y - cm.y));
        if (two)
            out[kp + k] =
                make_float2(0.5f * (c.y + cm.y), -0.5f * (c.x - cm.x));
    }
}

// Two half spectra as one complex line and back (z_inv_kernel's extension).
template <int R1, int R2>
__global__ __launch_bounds__((Pair<R1, R2>::T * kPairLines)) void pair_z_inv(
    BeamIO io, const float2* __restrict__ A, int32_t X, int32_t Y, int32_t Z,
    int32_t a_rows, int32_t kp, const float2* __restrict__ g_tw, int32_t W)
{
    using P = Pair<R1, R2>;
    __shared__ float2 s_tw[P::tw_len];
    __shared__ float2 s_a[P::inv_line * kPairLines];
    load_table(s_tw, g_tw, P::tw_len);
    const int beam = beam_of_block(io);
    float* __restrict__ D = io.d_tab ? io.d_tab[beam] : io.d;
    const int accumulate = io.acc_tab ? io.acc_tab[beam] : io.accumulate;
    A += beam * io.a_beam;
    const int w = threadIdx.x / P::T, j = threadIdx.x - w * P::T;
    const LinePair lp =
        line_pair((int64_t)group_of_block(io) * W + w, X, Y);
    const bool two = lp.y + 1 < Y;
    const float2* row = A + (lp.x * a_rows + lp.y) * (int64_t)kp;
    float* out = D + (lp.x * Y + lp.y) * (int64_t)Z;
    float2* line = s_a + w * P::inv_line;
    constexpr int half = P::F / 2;
    if (j < R1) {
        float2 v[R2];
#pragma unroll
        for (int r = 0; r < R2; ++r) {
            const int k = j + r * R1;
            const int kk = k <= half ? k : P::F - k;
            float2 a = make_float2(0.0f, 0.0f), b = a;
            if (lp.valid) {
                a = row[kk];
                if (two)
                    b = row[kp + kk];
            }
            if (k > half) {
                a.y = -a.y;
                b.y = -b.y;
            }
            if (k == 0 || k == half) {
                a.y = 0.0f;
                b.y = 0.0f;
            }
            v[r] = make_float2(a.x - b.y, a.y + b.x);
        }
        dft<true>(v);
#pragma unroll
        for (int r = 0; r < R2; ++r)
            line[r * P::P1 + j] = v[r];
    }
    __syncthreads();
    if (j >= R2 || !lp.valid)
        return;
    float2 v[R1];
#pragma unroll
    for (int r = 0; r < R1; ++r)
        v[r] = line[j * P::P1 + r];
    twiddle<R1, true, P>(v, s_tw, j);
    dft<true>(v);
#pragma unroll
    for (int r = 0; r < R1 / 2; ++r) {
        const int n = j + r * R2;
        if (n >= Z)
            continue;
        if (accumulate) {
            out[n] += v[r].x;
            if (two)
                out[Z + n] += v[r].y;
        } else {
            out[n] = v[r].x;
            if (two)
                out[Z + n] = v[r].y;
        }
    }
}

// ------------------------------------------------------------ launches ----

inline int log2_lines(int W)
{
    return W == 16 ? 4 : (W == 8 ? 3 : (W == 4 ? 2 : 1));
}
inline unsigned z_groups(const BeamIO& io, int X, int Y, int W)
{
    return (unsigned)(((int64_t)X * ((Y + 1) / 2) + W - 1) / W * io.n_beams);
}
inline dim3 col_grid(const BeamIO& io, int n_cols, int n_outer, int W)
{
    return dim3((unsigned)((int64_t)((n_cols + W - 1) / W) * io.n_beams),
                (unsigned)n_outer);
}

template <int R1, int R2>
struct PairLaunch {
    using P = Pair<R1, R2>;
    static ch_status z_fwd(const BeamIO& io, float2* A, int X, int Y, int Z,
                           int a_rows, int kp, const float2* tw,
                           hipStream_t s, int W, const Support& sp)
    {
        hipLaunchKernelGGL((pair_z_fwd<R1, R2>), dim3(z_groups(io, X, Y, W)),
                           dim3(P::T * W), 0, s, io, A, X, Y, Z, a_rows, kp,
                           tw, W, sp);
        CH_HIP(hipGetLastError());
        return CH_OK;
    }
    static ch_status z_inv(const BeamIO& io, const float2* A, int X, int Y,
                           int Z, int a_rows, int kp, const float2* tw,
                           hipStream_t s, int W)
    {
        hipLaunchKernelGGL((pair_z_inv<R1, R2>), dim3(z_groups(io, X, Y, W)),
                           dim3(P::T * W), 0, s, io, A, X, Y, Z, a_rows, kp,
                           tw, W);
        CH_HIP(hipGetLastError());
        return CH_OK;
    }
    static ch_status y_fwd(const BeamIO& io, float2* A, uint32_t row_stride,
                           int64_t outer_stride, int n_outer, int n_cols,
                           int n_in, const float2* tw, hipStream_t s, int W,
                           const Support& sp)
    {
        hipLaunchKernelGGL((pair_y_fwd<R1, R2>),
                           col_grid(io, n_cols, n_outer, W), dim3(P::T * W),
                           0, s, io, A, row_stride, outer_stride, n_cols,
                           n_in, tw, log2_lines(W), sp);
        CH_HIP(hipGetLastError());
        return CH_OK;
    }
    static ch_status y_inv(const BeamIO& io, float2* A, uint32_t row_stride,
                           int64_t outer_stride, int n_outer, int n_cols,
                           int n_out, const float2* tw, hipStream_t s, int W)
    {
        hipLaunchKernelGGL((pair_y_inv<R1, R2>),
                           col_grid(io, n_cols, n_outer, W), dim3(P::T * W),
                           0, s, io, A, row_stride, outer_stride, n_cols,
                           n_out, tw, log2_lines(W));
        CH_HIP(hipGetLastError());
        return CH_OK;
    }
    static ch_status conv(const BeamIO& io, float2* A, uint32_t row_stride,
                          int64_t outer_stride, int n_outer, int n_cols,
                          int n_in, const float2* tw, const float2* khat,
                          uint32_t k_row_stride, int64_t k_outer_stride,
                          hipStream_t s, int W, LaunchTimer* timer,
                          const Support& sp)
    {
        const dim3 grid = col_grid(io, n_cols, n_outer, W);
        const int32_t lw = log2_lines(W);
        if (timer)
            timer->launch(pair_conv<R1, R2>, grid, dim3(P::T * W), 0, io, A,
                          row_stride, outer_stride, (int32_t)n_cols,
                          (int32_t)n_in, tw, khat, k_row_stride,
                          k_outer_stride, lw, sp);
        else
            hipLaunchKernelGGL((pair_conv<R1, R2>), grid, dim3(P::T * W), 0,
                               s, io, A, row_stride, outer_stride, n_cols,
                               n_in, tw, khat, k_row_stride, k_outer_stride,
                               lw, sp);
        CH_HIP(hipGetLastError());
        return CH_OK;
    }
};

}  // namespace

#define CH_PAIR(F, R1, R2)                                                  \
    static_assert(R1 * R2 == F, "frame length");                            \
    PairFns pair_fns_##F()                                                  \
    {                                                                       \
        using L = PairLaunch<R1, R2>;                                       \
        return PairFns{L::z_fwd, L::z_inv, L::y_fwd, L::y_inv, L::conv};    \
    }

}  // namespace ch
