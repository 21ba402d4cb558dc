// aperture.h -- beam aperture transmission at a raster cell (row i, col j)
// of the 4000 x 4000, 0.1 mm grid of conehead/block.py, evaluated from a
// compact description.  The raster builder (raster.hip) and the TERMA hit
// test (terma.hip) call the same functions, so the analytic lookups and the
// materialised raster agree bit for bit.
#pragma once

#include "ch_internal.h"

namespace ch {

// Leaf transmission table of conehead/block.py:155-164: 1 - area, area =
// ones with edge rows 0.2/0.5/0.75 (the rows counted from the far edge are
// assigned last and win) and the last 15 columns scaled by
// numpy.linspace(1, 0, 15).  area's edge factor in row rr of a leaf of w
// rows:
inline float leaf_edge(int rr, int w)
{
    if (rr == w - 1) return 0.20f;
    if (rr == w - 2) return 0.50f;
    if (rr == w - 3) return 0.75f;
    if (rr == 0) return 0.20f;
    if (rr == 1) return 0.50f;
    if (rr == 2) return 0.75f;
    return 1.0f;
}
// and the edge factor e in the q-th of the last 15 columns (arange * step +
// start, last point exact; compiled without contraction).
constexpr int kTaper = 15;
__device__ __forceinline__ float leaf_taper(float e, int q)
{
    const double step = (0.0 - 1.0) / 14;
    const double lin = q == 14 ? 0.0 : (double)q * step + 1.0;
    return (float)((double)e * lin);
}

// Leaf-table layout (int32): [0] n_pairs, [1] W (bank width), [2] roff
// (raster row of bank row 0), [3] jx0, [4] jx1 (column jaws, tenths of mm),
// [5] jy0, [6] jy1 (bank-row jaws), [7] start of the row table, then
// bound[n_pairs + 1], ends of bank A [n_pairs], ends of bank B [n_pairs],
// and at [7] (16-byte aligned) the row table: per raster row 4 int32
// {column of bank A's tip, column of bank B's tip, bits of A's edge factor,
// bits of B's}, so a cell's value needs its row's entry (one 16-byte load)
// and two compares.  A closed row (outside the bank or the Y jaws) is under
// bank A with factor 1 everywhere, an open one (no leaf) under neither.
// Behind the row table, per row the last row of its run: rows of the same
// leaf pair (high 16 bits) and rows with the same entry (low 16 bits).
constexpr int kMlcHeader = 8;
constexpr int kMlcRows = 4000;
constexpr int kMlcFar = 1 << 20;   // a column past every raster column

__host__ __device__ __forceinline__ int mlc_row_table_start(int n_pairs)
{
    return (kMlcHeader + 3 * n_pairs + 1 + 3) & ~3;
}

__device__ __forceinline__ int4 mlc_row(const int32_t* __restrict__ t,
                                        int row)
{
    return reinterpret_cast<const int4*>(t + t[7])[row];
}

// Leaf bank and jaws of conehead/block.py:130-196 (bank centred on raster
// row 2000; rows outside the bank are blocked) at column col of a row with
// entry e: bank B (:189-190) is assigned after bank A (:187-188), the
// jaws (:193-196) last.
__device__ __forceinline__ float mlc_cell(const int32_t* __restrict__ t,
                                          const int4& e, int col)
{
    const bool in_b = col >= e.y && col < 3999;
    const bool in_a = col < e.x;
    float f = in_b ? __int_as_float(e.w) : (in_a ? __int_as_float(e.z) : 0.0f);
    // columns from the tip into the leaf
    const int q = in_b ? col - e.y : e.x - 1 - col;
    if ((in_a || in_b) && q < kTaper)
        f = leaf_taper(f, kTaper - 1 - q);
    const bool jaw = col < 2000 + t[3] || col >= 2000 + t[4];
    return jaw ? 0.0f : 1.0f - f;
}

__device__ __forceinline__ float mlc_value(const int32_t* __restrict__ t,
                                           int row, int col)
{
    return mlc_cell(t, mlc_row(t, row), col);
}

// Transmission of every cell of the block [i0, i1] x [j0, j1] (raster
// rows and columns, inside the raster, j1 <= 3998) when it is one
// constant, else -1.  Row runs whose columns all lie between the tips are
// open, and rows wholly under one leaf clear of its taper have 1 minus its
// edge factor (0 in its interior); a block that straddles a tip, a taper
// or a jaw, or whose runs differ, is not constant.
__device__ __forceinline__ float mlc_block_value(const int32_t* __restrict__ t,
                                                 int i0, int i1, int j0,
                                                 int j1)
{
    const int jx0 = 2000 + t[3], jx1 = 2000 + t[4];
    if (j1 < jx0 || j0 >= jx1)
        return 0.0f;  // behind a jaw
    if (j0 < jx0 || j1 >= jx1)
        return -1.0f;
    const int32_t* runs = t + t[7] + 4 * kMlcRows;
    float v = -1.0f;
    for (int r = i0; r <= i1;) {
        const int4 e = mlc_row(t, r);
        const int end = runs[r];
        const bool open = j0 >= e.x && j1 < e.y;
        float f = 0.0f;
        if (!open) {
            if (j0 >= e.y + kTaper)
                f = __int_as_float(e.w);
            else if (j1 < e.x - kTaper && j1 < e.y)
                f = __int_as_float(e.z);
            else
                return -1.0f;
        }
        const float here = 1.0f - f;
        if (r != i0 && here != v)
            return -1.0f;
        v = here;
        r = 1 + (open ? end >> 16 : end & 0xffff);
    }
    return v;
}

__device__ __forceinline__ float rects_block_value(const int32_t* __restrict__ t,
                                                   int n, int i0, int i1,
                                                   int j0, int j1)
{
    bool any = false;
    for (int k = 0; k < n; ++k) {
        const int a = t[4 * k], b = t[4 * k + 1], c = t[4 * k + 2],
                  d = t[4 * k + 3];
        if (i0 >= a && i1 < b && j0 >= c && j1 < d)
            return 1.0f;  // inside one rectangle
        if (i1 >= a && i0 < b && j1 >= c && j0 < d)
            any = true;   // touches this rectangle
    }
    return any ? -1.0f : 0.0f;
}

// Union of half-open rectangles [r0, r1) x [c0, c1) of ones
// (Block.set_square, conehead/block.py:73-77), layout n x 4.
__device__ __forceinline__ float rects_value(const int32_t* __restrict__ t,
                                             int n, int row, int col)
{
    for (int k = 0; k < n; ++k)
        if (row >= t[4 * k] && row < t[4 * k + 1] && col >= t[4 * k + 2] &&
            col < t[4 * k + 3])
            return 1.0f;
    return 0.0f;
}

}  // namespace ch
