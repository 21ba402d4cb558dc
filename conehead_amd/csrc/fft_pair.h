// fft_pair.h -- the five FFT passes for frames of two radices, F = R1 R2.
//
// The even 5-smooth frames from 72 to 400 points (but 250) split into two
// radices of at most 24, so a transform is two register stages with one
// exchange through LDS between them, where the general passes (spectral.hip)
// need three to five stages for lengths like 360 or 400.  Both radices and the
// length are template constants: indices fold into addresses, and the first
// stage drops the zero half of its input and the last one the cropped half
// of its output (R1 is even, and an even frame is at least twice the grid).
//
// Stage 1 (forward): thread j < R2 transforms rows j + r R2, r < R1 (rows
// from F / 2 up are padding), giving slots (j, r).  Stage 2: thread j < R1
// takes slots (r, j), r < R2, times W_F^(r j), and its outputs are rows
// j + r R1.  The inverse runs the stages the other way round: thread j < R1
// transforms rows j + r R1 over r < R2, then thread j < R2 takes slots
// (r, j), r < R1, times conj W_F^(r j), giving rows j + r R2, those below
// F / 2 kept.  In the convolution pass the product with K^ and the
// inverse's first stage stay in the registers of forward stage 2, whose
// results go back to the slots that thread read, so the pass needs two
// exchanges and one LDS buffer.
//
// Up to kPairLines lines per workgroup, max(R1, R2) threads per line.  The
// column passes keep a column per thread group of neighbouring threads
// (kPairLines columns are a 128-byte line), the z passes give neighbouring
// threads neighbouring points of one line, since their lines are contiguous.
//
// Measured per beam against the general passes (z forward, y forward,
// convolution, y inverse, z inverse; us by kernel trace on MI355X):
//                    general                      two stages
//   40^3             5.4  5.6   6.7  4.8  6.6     4.1  4.2   5.0  3.6  4.0
//   128^3            10.8 10.5  29.9 13.8 14.0    8.0  8.1  26.2 11.0  9.4
//   173 x 97 x 141   16.5 19.8  77.8 25.6 24.8    11.4 13.5 45.7 13.4 13.2
//   200 x 200 x 160  27.8 52.4 205.6 52.6 43.8    23.4 35.9 120.7 34.0 22.6
// The convolution pass moves 412 MB at 200 x 200 x 160, 82 us at the 5.0 TB/s
// a copy reaches; 135 MB, 27 us, at 128^3: bound by HBM there, elsewhere by
// the loads in flight (two to four workgroups per CU, by LDS and registers:
// larger radix first, since K^ is held beside the second).
// 16 lines per workgroup measured best in every pass of every size (8: up to
// 18 % slower in the convolution pass), so it is the default.
#pragma once

#include "fft_core.h"

namespace ch {

constexpr int kPairLines = 16;

// The launches of one frame length; W lines per workgroup (2, 4, 8 or 16).
// The column passes take the row and outer strides of the work grid in
// complex points, as col_kernel does.
struct PairFns {
    ch_status (*z_fwd)(const BeamIO& io, float2* A, int X, int Y, int Z,
                       int a_rows, int kp, const float2* tw, hipStream_t s,
                       int W, const Support& sp);
    ch_status (*z_inv)(const BeamIO& io, const float2* A, int X, int Y,
                       int Z, int a_rows, int kp, const float2* tw,
                       hipStream_t s, int W);
    ch_status (*y_fwd)(const BeamIO& io, float2* A, uint32_t row_stride,
                       int64_t outer_stride, int n_outer, int n_cols,
                       int n_in, const float2* tw, hipStream_t s, int W,
                       const Support& sp);
    ch_status (*y_inv)(const BeamIO& io, float2* A, uint32_t row_stride,
                       int64_t outer_stride, int n_outer, int n_cols,
                       int n_out, const float2* tw, hipStream_t s, int W);
    ch_status (*conv)(const BeamIO& io, float2* A, uint32_t row_stride,
                      int64_t outer_stride, int n_outer, int n_cols, int n_in,
                      const float2* tw, const float2* khat,
                      uint32_t k_row_stride, int64_t k_outer_stride,
                      hipStream_t s, int W, LaunchTimer* timer,
                      const Support& sp);
};

// The launches of frame length F; false when it has no pair of radices.
bool fft_pair(int F, PairFns* out);

// The frame lengths (batch.PAIR_FRAMES has them too), X(F) for each; their
// radices and launches are defined by translation unit (fft_pair_*.hip).
#define CH_PAIR_FRAMES(X)                                                   \
    X(72) X(80) X(90) X(96) X(100) X(108) X(120) X(128) X(144) X(150)       \
    X(160) X(162) X(180) X(192) X(200) X(216) X(240) X(256) X(270) X(288)   \
    X(300) X(320) X(324) X(360) X(384) X(400)
#define CH_PAIR_DECLARE(F) PairFns pair_fns_##F();
CH_PAIR_FRAMES(CH_PAIR_DECLARE)
#undef CH_PAIR_DECLARE

}  // namespace ch
