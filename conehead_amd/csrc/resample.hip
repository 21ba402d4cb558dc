// resample.hip -- linear resampling of phantom densities onto a dose grid.
//
// The reference builds scipy's RegularGridInterpolator (method 'linear',
// bounds_error False, fill_value 0) on the phantom axes
// linspace(o_a, o_a + n_a s_a, n_a) (conehead/conehead.py:525-533) and
// evaluates it at the dose grid's axes built the same way, laid out by
// np.meshgrid with indexing 'xy' (:562-567), so output[i][j][k] is the
// value at (x_j, y_i, z_k).  The arithmetic follows numpy and scipy in FP64 without contraction: linspace nodes are
// k * step + start with the last node equal to stop, the cell of a
// coordinate is searchsorted(nodes, x) - 1 clamped to [0, n - 2], points
// outside [node_0, node_{n-1}] give 0, and the eight corner weights are
// products of (1 - t) and t accumulated corner by corner in
// itertools.product order.
#include <algorithm>

#include "ch_internal.h"

#include <cmath>
#include <cstring>

namespace ch {

struct Axis {
    double start, stop, step;   // step = (stop - start) / (n - 1)
    int n;
};

// numpy.linspace(start, stop, n)[k]
__device__ __forceinline__ double node(const Axis& a, int k)
{
    if (a.n == 1)
        return a.start;
    if (k == a.n - 1)
        return a.stop;
    return (double)k * a.step + a.start;
}

// Cell index (-1 when x is outside the axis) and fraction of x.
__device__ __forceinline__ void locate(const Axis& a, double x, int& i,
                                       double& t)
{
    const double first = node(a, 0), last = node(a, a.n - 1);
    i = -1;
    t = 0.0;
    if (!(x >= first && x <= last))
        return;
    if (a.n == 1) {
        i = 0;
        return;
    }
    // searchsorted(side='left'): first k with node(k) >= x
    int lo = 0, hi = a.n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (node(a, mid) < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    i = lo - 1;
    i = i < 0 ? 0 : (i > a.n - 2 ? a.n - 2 : i);
    const double g0 = node(a, i), g1 = node(a, i + 1);
    t = (x - g0) / (g1 - g0);
}

// A voxel's three searches and divisions cost far more than its eight loads,
// so they are shared: a wavefront's lanes lie along z, `width` of them on a
// row, and take kRows rows one after the other.  A lane finds its own z once;
// lane r finds x and y of the wavefront's r-th row, and the others fetch them
// from it.  The width is 64, or down to 4 for dose grids of few slices, where
// the lanes of a wavefront lie on up to 16 rows at a time.
// 512 x 512 x 120 onto 160 x 160 x 128: 82 -> 19 us.
template <int kRows>
__global__ __launch_bounds__(256) void resample_kernel(
    const float* __restrict__ src, int sx, int sy, int sz, Axis ax, Axis ay,
    Axis az, float* __restrict__ dst, int dx, int dy, int dz, Axis bx,
    Axis by, Axis bz, int swap, int width, int z_groups)
{
    const int lane = threadIdx.x & 63;
    const int64_t rows = (int64_t)dx * dy;
    const int per = kRows * (64 / width);         // rows of a wavefront, <= 64
    const int zg = (int)(blockIdx.x % (unsigned)z_groups);
    const int64_t first = ((int64_t)(blockIdx.x / (unsigned)z_groups) * 4 +
                           (threadIdx.x >> 6)) * per;
    if (first >= rows)
        return;
    const int64_t mine = min(first + (lane & (per - 1)), rows - 1);
    const int a = (int)(mine / dy), b = (int)(mine % dy);
    int ix, iy, i2;
    double tx, ty, t2;
    locate(ax, swap ? node(bx, b) : node(bx, a), ix, tx);
    locate(ay, swap ? node(by, a) : node(by, b), iy, ty);
    const int c = zg * width + (lane & (width - 1));
    locate(az, node(bz, min(c, dz - 1)), i2, t2);
    const int sub = lane / width;
    const int o2 = sz == 1 ? 0 : 1, o1 = sy == 1 ? 0 : sz;
    const int64_t o0 = sx == 1 ? 0 : (int64_t)sy * sz;
    const double u2 = 1.0 - t2;
#pragma unroll (kRows > 1 ? 2 : 1)
    for (int k = 0; k < kRows; ++k) {
        const int r = k * (64 / width) + sub;
        const int i0 = __shfl(ix, r), i1 = __shfl(iy, r);
        const double t0 = __shfl(tx, r), t1 = __shfl(ty, r);
        if (first + r >= rows || c >= dz)
            continue;
        float out = 0.0f;
        if ((i0 | i1 | i2) >= 0) {
            const float* p = src + ((int64_t)i0 * sy + i1) * sz + i2;
            const float f[8] = {p[0],       p[o2],      p[o1],
                                p[o1 + o2], p[o0],      p[o0 + o2],
                                p[o0 + o1], p[o0 + o1 + o2]};
            const double u0 = 1.0 - t0, u1 = 1.0 - t1;
            const double w[4] = {u0 * u1, u0 * t1, t0 * u1, t0 * t1};
            double v = 0.0;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v = v + (double)f[e] * (w[e >> 1] * (e & 1 ? t2 : u2));
            out = (float)v;
        }
        dst[(first + r) * dz + c] = out;
    }
}

// CT numbers to densities: a piecewise-linear calibration curve evaluated
// as numpy.interp does (clamped to the end values outside the curve, the
// node's own density at a node, slope * (x - x_j) + y_j between nodes, FP64
// without contraction), then a per-label override for the voxels of a
// label map (structures forced to a density).  Both tables travel in the
// kernel arguments.
struct CtTable {
    double hu[CH_CT_MAX_POINTS];
    double rho[CH_CT_MAX_POINTS];
    double slope[CH_CT_MAX_POINTS];
    float at[CH_CT_MAX_POINTS];  // the least float >= hu
    float override_rho[256];  // NaN: keep the curve's density
    int n;
};

// Entry m of the tables in LDS serves the numbers with m nodes at or below
// them: m = 0 and m = n are the clamps.  Comparing in FP32 with the least
// float at or above a node decides as the FP64 comparison does.
struct CtLds {
    double hu[CH_CT_MAX_POINTS + 1];
    double slope[CH_CT_MAX_POINTS + 1];
    double rho[CH_CT_MAX_POINTS + 1];
    float over[256];
};

// Nodes at or below x (exact for both types of CT numbers).
__device__ __forceinline__ int ct_nodes(const CtTable& c, float x)
{
    int m = 0;
    for (int k = 0; k < c.n; ++k)
        m += x >= c.at[k] ? 1 : 0;
    return m;
}
// The density with m nodes at or below xf, from entry m of the tables.
__device__ __forceinline__ float ct_density(const CtTable& c, float xf, int m,
                                            double h, double slope, double r)
{
    const double x = (double)xf;
    const bool flat = (m == 0 && xf == xf) || m == c.n;
    // a NaN has m = 0 and takes the slope
    return flat || x == h ? (float)r : (float)(slope * (x - h) + r);
}
__device__ __forceinline__ float ct_density(const CtTable& c, const CtLds& t,
                                            float xf)
{
    const int m = ct_nodes(c, xf);
    return ct_density(c, xf, m, t.hu[m], t.slope[m], t.rho[m]);
}

// G groups of four voxels per thread, a workgroup's 256 threads side by side
// in each: 8-byte loads of int16, 16-byte stores.  The curve and the overrides
// are read from LDS; with the nodes searched in FP64 and the entries read from
// the kernel arguments the kernel ran at 1.6 TB/s.  512 x 512 x 120 with
// labels: 137 -> 49 us (4.5 TB/s).  G = 0: a voxel per thread, its entry of
// the tables read from the arguments, for series too small to fill the chip,
// where filling LDS and several voxels in a row are latency (ct_groups).
template <typename T>
struct alignas(sizeof(T)) Ct4 {
    T v[4];
};
struct Label4 {
    uint8_t v[4];
};
struct Rho4 {
    float v[4];
};

template <typename T>
__global__ __launch_bounds__(256) void ct_small_kernel(
    const T* __restrict__ hu, const uint8_t* __restrict__ labels, int64_t n,
    CtTable c, float* __restrict__ rho)
{
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= n)
        return;
    const T x = hu[i];
    const float o = labels ? c.override_rho[labels[i]] : NAN;
    const int m = ct_nodes(c, (float)x), j = m == 0 ? 0 : m - 1;
    const float v = ct_density(c, (float)x, m, c.hu[j], c.slope[j], c.rho[j]);
    rho[i] = o == o ? o : v;
}

template <typename T, int G>
__global__ __launch_bounds__(256) void ct_kernel(
    const T* __restrict__ hu, const uint8_t* __restrict__ labels, int64_t n,
    CtTable c, float* __restrict__ rho)
{
    __shared__ CtLds t;
    for (int m = threadIdx.x; m <= c.n; m += 256) {
        const int j = m == 0 ? 0 : m - 1;
        t.hu[m] = c.hu[j];
        t.slope[m] = c.slope[j];
        t.rho[m] = c.rho[j];
    }
    if (labels)
        t.over[threadIdx.x] = c.override_rho[threadIdx.x];
    __syncthreads();
    const int64_t base = blockIdx.x * (int64_t)(1024 * G);
    if (base + 1024 * G <= n) {
        Ct4<T> x[G];
        Label4 l[G] = {};
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int64_t i = base + 1024 * g + 4 * threadIdx.x;
            x[g] = *(const Ct4<T>*)(hu + i);
            if (labels)
                l[g] = *(const Label4*)(labels + i);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            Rho4 v;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v.v[q] = ct_density(c, t, (float)x[g].v[q]);
                if (labels) {
                    const float o = t.over[l[g].v[q]];
                    v.v[q] = o == o ? o : v.v[q];
                }
            }
            *(Rho4*)(rho + base + 1024 * g + 4 * threadIdx.x) = v;
        }
        return;
    }
    for (int64_t i = base + threadIdx.x; i < n; i += 256) {
        float v = ct_density(c, t, (float)hu[i]);
        if (labels) {
            const float o = t.over[labels[i]];
            v = o == o ? o : v;
        }
        rho[i] = v;
    }
}

// us for G = 0, 1 and 4, int16 with labels (the FP64 search took 2.7 at 2^15
// voxels, 3.0 at 2^18, 7.6 at 1.6 M and 37 at 8 M):
//   2^15   2.4  3.4  7.7     1 M     4.9  4.3  8.2     8 M     29  17  19
//   2^18   2.7  3.6  7.8     1.6 M   6.7  5.6  8.8     31 M   105  49  47
static int ct_groups(int64_t n)
{
    return n <= 1 << 19 ? 0 : n <= 1 << 24 ? 1 : 4;
}
template <typename T>
static void ct_launch(const T* d_ct, const uint8_t* d_labels, int64_t n,
                      const CtTable& c, float* d_rho, hipStream_t s)
{
    const int g = ct_groups(n);
    const int64_t per = g == 0 ? 256 : 1024 * g;
    void (*kernel)(const T*, const uint8_t*, int64_t, CtTable, float*) =
        ct_small_kernel<T>;
    if (g == 1)
        kernel = ct_kernel<T, 1>;
    else if (g == 4)
        kernel = ct_kernel<T, 4>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((n + per - 1) / per)),
                       dim3(256), 0, s, d_ct, d_labels, n, c, d_rho);
}

static Axis axis(double origin, double spacing, int n)
{
    Axis a;
    a.start = origin;
    a.stop = origin + (double)n * spacing;
    a.step = n > 1 ? (a.stop - a.start) / (double)(n - 1) : 0.0;
    a.n = n;
    return a;
}

// Rows a lane takes, by the lanes its z row and the others' fill (lanes): more
// rows share more searches, fewer fill the chip.  us for 8, 4, 2 and 1 rows,
// and for three searches per voxel:
//   50^3 onto itself         160 K lanes   5.7  4.7  4.7  5.2     5.5
//   64^3 onto 32^3            32 K         6.3  5.0  4.3  4.0     4.7
//   512 x 512 x 120 onto 40^3 102 K        6.6  5.4  4.7  5.0     5.2
//   128^3 onto 64^3          262 K         6.8  5.5  5.4  6.6     9.0
//   256 x 256 x 60 onto 128 x 128 x 20
//                            524 K         7.5  6.5  7.4 10.2    10.6
//   80^3 onto itself         819 K         7.2  8.3 10.1 14.4
// Narrow rows (width 4 or 8) take at most two: 512 x 512 x 120 onto one slice
// of 512 x 512 (1 M lanes) 13.8 us with four, 13.2 with two, 18.7 with one
// (15.2 with three searches per voxel; 20 with the width kept at 16).
static int resample_rows(int64_t lanes, int width)
{
    const int kr = lanes < 1 << 16   ? 1
                   : lanes < 1 << 17 ? 2
                   : lanes < 600000  ? 4
                                     : 8;
    return width < 16 ? std::min(kr, 2) : kr;
}

}  // namespace ch

using namespace ch;

extern "C" {

ch_status ch_resample_linear(const float* d_src, const int32_t src_shape[3],
                             const double src_origin[3],
                             const double src_spacing[3], float* d_dst,
                             const int32_t dst_shape[3],
                             const double dst_origin[3],
                             const double dst_spacing[3], int32_t xy_swap,
                             void* stream)
{
    CH_REQUIRE(d_src && d_dst && src_shape && src_origin && src_spacing &&
                   dst_shape && dst_origin && dst_spacing,
               "ch_resample_linear: null pointer");
    for (int k = 0; k < 3; ++k) {
        CH_REQUIRE(src_shape[k] > 0 && dst_shape[k] > 0,
                   "ch_resample_linear: empty grid");
        CH_REQUIRE(src_spacing[k] > 0 && dst_spacing[k] > 0,
                   "ch_resample_linear: spacing must be > 0");
    }
    CH_REQUIRE(!xy_swap || dst_shape[0] == dst_shape[1],
               "ch_resample_linear: the 'xy' layout needs size[0] == size[1] "
               "(got %d x %d)",
               dst_shape[0], dst_shape[1]);
    const int64_t n = (int64_t)dst_shape[0] * dst_shape[1] * dst_shape[2];
    CH_REQUIRE(n < (1LL << 31), "ch_resample_linear: grid too large");
    int width = 4;
    while (width < 64 && width < dst_shape[2])
        width *= 2;
    const int z_groups = (dst_shape[2] + width - 1) / width;
    const int64_t rows = (int64_t)dst_shape[0] * dst_shape[1];
    const int kr = resample_rows(rows * z_groups * width, width);
    const int64_t per_group = 4 * kr * (64 / width);
    const int64_t groups = (rows + per_group - 1) / per_group;
    auto kernel = resample_kernel<1>;
    if (kr == 2)
        kernel = resample_kernel<2>;
    else if (kr == 4)
        kernel = resample_kernel<4>;
    else if (kr == 8)
        kernel = resample_kernel<8>;
    hipLaunchKernelGGL(
        kernel, dim3((unsigned)(groups * z_groups)), dim3(256), 0,
        (hipStream_t)stream, d_src, src_shape[0], src_shape[1], src_shape[2],
        axis(src_origin[0], src_spacing[0], src_shape[0]),
        axis(src_origin[1], src_spacing[1], src_shape[1]),
        axis(src_origin[2], src_spacing[2], src_shape[2]), d_dst,
        dst_shape[0], dst_shape[1], dst_shape[2],
        axis(dst_origin[0], dst_spacing[0], dst_shape[0]),
        axis(dst_origin[1], dst_spacing[1], dst_shape[1]),
        axis(dst_origin[2], dst_spacing[2], dst_shape[2]), xy_swap ? 1 : 0,
        width, z_groups);
    CH_HIP(hipGetLastError());
    return CH_OK;
}

ch_status ch_ct_to_density(const void* d_ct, int32_t ct_type, int64_t n,
                           const double* curve_hu, const double* curve_rho,
                           int32_t n_points, const uint8_t* d_labels,
                           const float* override_rho, float* d_rho,
                           void* stream)
{
    CH_REQUIRE(d_ct && d_rho && curve_hu && curve_rho,
               "ch_ct_to_density: null pointer");
    CH_REQUIRE(ct_type == CH_CT_I16 || ct_type == CH_CT_F32,
               "ch_ct_to_density: unknown CT number type %d", ct_type);
    CH_REQUIRE(n >= 0 && n < (1LL << 40), "ch_ct_to_density: bad count");
    CH_REQUIRE(n_points >= 1 && n_points <= CH_CT_MAX_POINTS,
               "ch_ct_to_density: the curve needs 1 to %d points (got %d)",
               CH_CT_MAX_POINTS, n_points);
    CH_REQUIRE(!d_labels || override_rho,
               "ch_ct_to_density: a label map needs its override table");
    CtTable c;
    memset(&c, 0, sizeof(c));
    c.n = n_points;
    for (int k = 0; k < n_points; ++k) {
        CH_REQUIRE(std::isfinite(curve_hu[k]) && std::isfinite(curve_rho[k]),
                   "ch_ct_to_density: curve point %d is not finite", k);
        CH_REQUIRE(k == 0 || curve_hu[k] > curve_hu[k - 1],
                   "ch_ct_to_density: curve CT numbers must increase "
                   "(point %d)", k);
        c.hu[k] = curve_hu[k];
        c.rho[k] = curve_rho[k];
        c.at[k] = (float)curve_hu[k];
        if ((double)c.at[k] < curve_hu[k])
            c.at[k] = nextafterf(c.at[k], INFINITY);
    }
    for (int k = 0; k + 1 < n_points; ++k)
        c.slope[k] = (c.rho[k + 1] - c.rho[k]) / (c.hu[k + 1] - c.hu[k]);
    for (int k = 0; k < 256; ++k)
        c.override_rho[k] = override_rho ? override_rho[k] : NAN;
    if (n == 0)
        return CH_OK;
    if (ct_type == CH_CT_I16)
        ct_launch((const int16_t*)d_ct, d_labels, n, c, d_rho,
                  (hipStream_t)stream);
    else
        ct_launch((const float*)d_ct, d_labels, n, c, d_rho,
                  (hipStream_t)stream);
    CH_HIP(hipGetLastError());
    return CH_OK;
}

}  // extern "C"
