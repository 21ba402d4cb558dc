// physics.hip -- physics-mode convolution: cones aligned with the beam and
// kernel increments looked up at the radiological distance.
//
// The reference convolves with world-fixed cones and geometric distances
// and lists kernel tilting as a milestone (README.md:22).  Here the caller
// rotates the cone set into the beam frame (the directions handed to
// ch_plan_create), and for a receiving voxel v and cone c with path offsets
// o_m and exit t-values t_m the increments are
//   R_m = sum_{j<=m} rho(v - o_j) (t_j - t_{j-1}),  t_{-1} = 0,
//   k_m = cum[i(R_m)] - cum[i(R_{m-1})],  i(R) = min(|floor(100 R - 5)|, 5995)
// (the index of cuda_dose, conehead/conehead.py:453-463, taken at R instead
// of t), and dose[v] = sum_c sum_m k_m T(v - o_m).  The path lengths
// t_m - t_{m-1} come from the plan (CH_SEM_RADIOLOGICAL).
//
// The gather keeps the direct gather's layout: a wavefront owns a 1 x 4 x 16
// output tile and reads padded copies of the grids.  Every lane walks its
// cone from its own voxel (R needs the whole path), loading densities only
// up to the first tap of the tile's union range and densities and T from
// there on.  A workgroup of 8 wavefronts stages each kernel row in LDS once
// and runs the cones of that row.  R, the index and the increments are FP64;
// the sums are FP32 with compensation.
//
// What bounds it is the latency of the loads and of the path sum they feed,
// with vector issue at half of its rate, so
//   - a workgroup's wavefronts are neighbouring tiles that walk the same cone
//     at about the same time, so one reads what another has read (rad_tiles);
//   - tap addresses are a scalar base per tap plus the lane's own offset, no
//     vector arithmetic and no range check: every tap of a range lies inside
//     the padded grids for every lane (the tile's end points are within the
//     range's box or on the way to it, and the padding covers the tile), and
//     the taps past the range end take its last one with path length 0 and
//     T = 0, which adds nothing;
//   - T follows the densities, so one base serves both loads; one 8-byte
//     load of (density, T) costs more than the two (a wavefront's 4-byte
//     load takes 5 cycles of the vector cache, its 8-byte load 16);
//   - a row starts kRadLead entries into its LDS array, so the truncated
//     100 R is its slot;
//   - a chunk whose T is 0 for the whole wavefront (the corners of an
//     oblique beam's box) needs one lookup instead of eight;
//   - a staged row's loads are all in flight before the first store;
//   - the ends of a path and of a range go in chunks of four taps with wide
//     scalar loads of their table entries (rad_chunk): short ranges, in thin
//     grids, are mostly ends (chunks of eight 2 to 5 % slower);
//   - the path sum stays a product and a sum, whose indices are the FP64
//     oracle's: fused multiply-adds were 2.5 % faster.
// 144 cones, 96^3 voxels with the gantry at 0 and at 20 degrees: 1359 -> 1195
// and 2498 -> 1928 us; 128^3 at 0 3448 -> 3040.
#include <algorithm>
#include <climits>

#include "ch_internal.h"

namespace ch {

typedef __attribute__((address_space(4))) const int32_t c_i32;
typedef __attribute__((address_space(4))) const double c_f64;

struct RadJob {
    const float* grids;    // padded densities and, after them, T
    float* dose;
    const int32_t* box;
    const int32_t* lin;    // per tap: byte offset into the padded densities
    const double* seg;     // per tap: path length inside the voxel
    const int32_t* ftT;    // first-step tables, cone-minor
    const ConeMeta* meta;
    const int32_t* perm;   // cones ordered by kernel row
    const int32_t* row_begin;
    const double* cum;
    double* parts;         // n_parts > 1: the sums of each part of the rows
    int32_t row_len, n_rows, n_parts;
    int32_t X, Y, Z, n_cones, accumulate, nty, ntz;
    int32_t wx, wy, wz;    // a workgroup's tiles: wx wy wz = kRadWaves
};

constexpr int kRadTY = 4, kRadTZ = 16;   // a wavefront's y and z voxels
constexpr int kRadWaves = 8;
constexpr int kRadRow = kMaxIndex + 1;
constexpr int kRadLead = 5;   // unused entries before a row in LDS

// trunc(x) as int32, saturating (v_cvt_i32_f64 clamps to the int32 range
// and reads NaN as 0; a C++ cast of an out-of-range value is undefined).
__device__ __forceinline__ int trunc_sat(double x)
{
    int r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// |floor(x - 5)| clamped to kMaxIndex, x = 100 R as the FP64 product.
__device__ __forceinline__ int rad_index_of(double x)
{
    const double f = floor(x - 5.0);
    if (!(f < 2147483647.0 && f > -2147483648.0))
        return kMaxIndex;
    int i = (int)f;
    i = i < 0 ? -i : i;
    return i > kMaxIndex ? kMaxIndex : i;
}

__device__ __forceinline__ void rad_kahan(float& s, float& c, float x)
{
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// The row's value at |floor(100 R - 5)| (clamped); s_cum: the row after
// kRadLead unused entries.
__device__ __forceinline__ double rad_at(const double* s_cum, double R)
{
    return s_cum[rad_index_of(R * 100.0) + kRadLead];
}

// The lane's element of a grid at a tap: base (uniform) minus the tap's byte
// offset in scalar registers, kept apart from the lane's offset by the empty
// asm, so a load needs no vector address arithmetic.
__device__ __forceinline__ float tap_load(const char* base, int64_t tap,
                                          uint32_t voff)
{
    uint64_t p = (uint64_t)base - (uint64_t)tap;
    asm("" : "+s"(p));
    typedef __attribute__((address_space(1))) const float g_float;
    typedef __attribute__((address_space(1))) const char g_char;
    asm("" : "+v"(voff));
    return *(g_float*)((g_char*)p + voff);
}

// N taps from tap t of the range that ends at uhi: densities into the path sum
// R, T times the rows' increments into the compensated sum (acc, ac).  LAST:
// taps at or past uhi take the address of tap uhi - 1, path length 0 and T =
// 0.  Their table entries are read all the same (a cone's taps are followed by
// kTapPad unused ones), so the chunk's entries come in wide scalar loads; one
// load each, with the index held below uhi, cost 3 to 6 % of the gather.
template <bool LAST, int N>
__device__ __forceinline__ void rad_chunk(const char* rho, uint32_t voff,
                                          uint32_t toff, const c_i32* ml,
                                          const c_f64* ms,
                                          const double* s_cum, int t, int uhi,
                                          double& R, double& cprev,
                                          float& acc, float& ac)
{
    static_assert(N <= kTapPad, "entries read past the range");
    float v[N], y[N];
    int idx[N];
    const int32_t last = LAST ? ml[uhi - 1] : 0;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int32_t o = ml[t + u];
        const int32_t tap = LAST && t + u >= uhi ? last : o;
        v[u] = tap_load(rho, tap, voff);
        y[u] = tap_load(rho, tap, toff);
    }
    // For x = 100 R >= 5 the subtraction of 5 is exact (the difference is a
    // multiple of ulp(x) below x), so the slot |floor(x - 5)| + 5, clamped,
    // is min(trunc(x), kMaxIndex + 5); a chunk with a tap below 5 (or NaN,
    // which truncates to 0) takes rad_index_of for all its taps.
    const double R0 = R;
    int least = kMaxIndex;
    int any = 0;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        if (LAST)
            y[u] = t + u < uhi ? y[u] : 0.0f;
        any |= __float_as_int(y[u]);
        const double g = ms[t + u];
        R = R + (double)v[u] * (LAST && t + u >= uhi ? 0.0 : g);
        idx[u] = min(trunc_sat(R * 100.0), kMaxIndex + kRadLead);
        least = min(least, idx[u]);
    }
    const bool lit = __builtin_amdgcn_ballot_w64(any != 0) != 0;
    if (__builtin_amdgcn_ballot_w64(least < kRadLead) != 0) {
        // a real branch: R passes through an empty asm here, so the compiler
        // cannot hoist this work onto every chunk
        double r = R0;
        asm volatile("" : "+v"(r));
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const double g = ms[t + u];
            r = r + (double)v[u] * (LAST && t + u >= uhi ? 0.0 : g);
            idx[u] = rad_index_of(r * 100.0) + kRadLead;
        }
    }
    if (!lit) {
        cprev = s_cum[idx[N - 1]];
        return;
    }
    float some = 0.0f;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const double cv = s_cum[idx[u]];
        const float k = (float)(cv - cprev);
        cprev = cv;
        some = fmaf(k, y[u], some);
    }
    rad_kahan(acc, ac, some);
}

// R along N taps, those at or past the end without length (LAST).
template <bool LAST, int N>
__device__ __forceinline__ void rad_path(const char* rho, uint32_t voff,
                                         const c_i32* ml, const c_f64* ms,
                                         int t, int end, double& R)
{
    float v[N];
    double g[N];
    const int32_t last = LAST ? ml[end - 1] : 0;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int32_t o = ml[t + u];
        const double s = ms[t + u];
        v[u] = tap_load(rho, LAST && t + u >= end ? last : o, voff);
        g[u] = LAST && t + u >= end ? 0.0 : s;
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
        R = R + (double)v[u] * g[u];
}

constexpr int kRadAhead = 2;   // chunks of densities in flight
constexpr int kRadTail = 4;    // taps per chunk at the end of a range
constexpr int kRadStage = (kRadRow + 64 * kRadWaves - 1) / (64 * kRadWaves);

// The lane's sum over every kernel row (all wavefronts of the workgroup call
// it; work: the tile has something to do).
__device__ __forceinline__ void rad_rows(const RadJob& j, double* s_cum,
                                          bool work, int x, int y0, int yl,
                                          int z0, int zl, const int (&lo)[3],
                                          const int (&hi)[3], uint32_t voff,
                                          uint32_t toff, float& sum,
                                          float& comp)
{
    const int lane = threadIdx.x & 63;
    const char* rho = (const char*)j.grids;
    const c_i32* lin = (const c_i32*)j.lin;
    const c_f64* seg = (const c_f64*)j.seg;
    sum = comp = 0.0f;
    const int part = blockIdx.y;
    const int row_end = j.n_rows * (part + 1) / j.n_parts;
    for (int row = j.n_rows * part / j.n_parts; row < row_end; ++row) {
        __syncthreads();
        const double* src = j.cum + (size_t)row * j.row_len;
        // every load of the row first, then the stores
        double v[kRadStage];
#pragma unroll
        for (int q = 0; q < kRadStage; ++q) {
            const int i = threadIdx.x + q * 64 * kRadWaves;
            if (i < kRadRow)
                v[q] = src[i];
        }
#pragma unroll
        for (int q = 0; q < kRadStage; ++q) {
            const int i = threadIdx.x + q * 64 * kRadWaves;
            if (i < kRadRow)
                s_cum[i + kRadLead] = v[q];
        }
        __syncthreads();
        if (!work)
            continue;
        const int cb = j.row_begin[row], ce = j.row_begin[row + 1];
        for (int q = cb; q < ce; q += 64) {
            // lane l: the tile's union range of cone perm[q + l]
            int r_lo = 0, r_hi = 0, r_tb = 0;
            if (q + lane < ce) {
                const int c = j.perm[q + lane];
                const ConeMeta* m = j.meta + c;
                const int n = j.n_cones;
                const int32_t* f0 = j.ftT;
                const int32_t* f1 = j.ftT + ftab_t_base(1, j.X, j.Y, n);
                const int32_t* f2 = j.ftT + ftab_t_base(2, j.X, j.Y, n);
                int ax, bx, ay1, by1, ay2, by2, az1, bz1, az2, bz2;
                vrange_t(x, lo[0], hi[0], m->step[0], f0, j.X + 2, n, c, ax,
                         bx);
                vrange_t(y0, lo[1], hi[1], m->step[1], f1, j.Y + 2, n, c, ay1,
                         by1);
                vrange_t(yl, lo[1], hi[1], m->step[1], f1, j.Y + 2, n, c, ay2,
                         by2);
                vrange_t(z0, lo[2], hi[2], m->step[2], f2, j.Z + 2, n, c, az1,
                         bz1);
                vrange_t(zl, lo[2], hi[2], m->step[2], f2, j.Z + 2, n, c, az2,
                         bz2);
                r_lo = max(max(ax, min(ay1, ay2)), min(az1, az2));
                r_hi = min(min(bx, max(by1, by2)), max(bz1, bz2));
                r_tb = m->tap_begin;
            }
            const int nc = min(64, ce - q);
            for (int i = 0; i < nc; ++i) {
                const int ulo = __builtin_amdgcn_readlane(r_lo, i);
                const int uhi = __builtin_amdgcn_readlane(r_hi, i);
                if (ulo >= uhi)
                    continue;
                const int tb = __builtin_amdgcn_readlane(r_tb, i);
                const c_i32* ml = lin + tb;
                const c_f64* ms = seg + tb;
                // the path from the receiving voxel up to the union range:
                // densities only (every source there is outside the box)
                double R = 0.0;
                int t = 0;
                constexpr int far = kRadAhead * kUnroll;
                for (; t + far <= ulo; t += far)
                    rad_path<false, far>(rho, voff, ml, ms, t, ulo, R);
                if (t + kUnroll <= ulo) {
                    rad_path<false, kUnroll>(rho, voff, ml, ms, t, ulo, R);
                    t += kUnroll;
                }
                for (; t < ulo; t += kRadTail)
                    rad_path<true, kRadTail>(rho, voff, ml, ms, t, ulo, R);
                double cprev = ulo > 0 ? rad_at(s_cum, R) : 0.0;
                float acc = 0.0f, ac = 0.0f;
                for (t = ulo; t + kUnroll <= uhi; t += kUnroll)
                    rad_chunk<false, kUnroll>(rho, voff, toff, ml, ms, s_cum,
                                              t, uhi, R, cprev, acc, ac);
                for (; t < uhi; t += kRadTail)
                    rad_chunk<true, kRadTail>(rho, voff, toff, ml, ms, s_cum,
                                              t, uhi, R, cprev, acc, ac);
                rad_kahan(sum, comp, acc);
            }
        }
    }
}

__global__ __launch_bounds__(64 * kRadWaves, 6) void gather_rad(RadJob j)
{
    __shared__ double s_cum[kRadRow + kRadLead];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int gz = (j.ntz + j.wz - 1) / j.wz, gy = (j.nty + j.wy - 1) / j.wy;
    const int g = blockIdx.x, gxy = g / gz, wxy = wave / j.wx;
    const int xw = gxy / gy * j.wx + wave % j.wx;
    const int ty = gxy % gy * j.wy + wxy % j.wy;
    const int tz = g % gz * j.wz + wxy / j.wy;
    const bool live = xw < j.X && ty < j.nty && tz < j.ntz;
    const int x = live ? xw : 0;
    const int y0 = live ? ty * kRadTY : 0, z0 = live ? tz * kRadTZ : 0;
    const int yl = min(y0 + kRadTY - 1, j.Y - 1);
    const int zl = min(z0 + kRadTZ - 1, j.Z - 1);
    const int y = y0 + lane / kRadTZ;
    const int z = z0 + lane % kRadTZ;
    const int Zp = j.Z + 2 * kZPad;
    const int Yp = j.Y + 2 * kYPad;

    int lo[3] = {0, 0, 0}, hi[3] = {j.X - 1, j.Y - 1, j.Z - 1};
    if (j.box) {
        const c_i32* b = (const c_i32*)j.box;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = max(lo[a], b[a]);
            hi[a] = min(hi[a], b[3 + a]);
        }
    }
    const bool work =
        live && lo[0] <= hi[0] && lo[1] <= hi[1] && lo[2] <= hi[2];
    const uint32_t voff =
        (uint32_t)((x * Yp + y + kYPad) * Zp + z + kZPad) * 4u;
    const uint32_t toff = voff + (uint32_t)(j.X * Yp * Zp) * 4u;
    float sum, comp;
    rad_rows(j, s_cum, work, x, y0, yl, z0, zl, lo, hi, voff, toff, sum,
             comp);
    if (live && y <= yl && z <= zl && j.n_parts > 1) {
        const int64_t n = (int64_t)j.X * j.Y * j.Z;
        j.parts[blockIdx.y * n + ((int64_t)x * j.Y + y) * j.Z + z] =
            (double)sum - (double)comp;
    } else if (live && y <= yl && z <= zl) {
        float* d = j.dose + ((size_t)x * j.Y + y) * j.Z + z;
        *d = (j.accumulate ? *d : 0.0f) + sum;
    }
}

// dose (+)= the sum of the parts, in FP64.
__global__ __launch_bounds__(256) void rad_sum(const double* parts,
                                               int n_parts, int64_t n,
                                               float* dose, int accumulate)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    double v = 0.0;
    for (int p = 0; p < n_parts; ++p)
        v += parts[p * n + i];
    dose[i] = (accumulate ? dose[i] : 0.0f) + (float)v;
}

// The tiles of a workgroup in x, y and z, by the tiles along z: 2 x 1 x 4
// where they fill groups of four to within an eighth, 2 x 2 x 2 where there
// are two, 4 x 2 x 1 elsewhere, 2 x 4 x 1 for grids of at most 12 slices (us,
// 144 cones, the last 72; gantry 0 but where given; consecutive: the eight
// tiles along z, then y, of range-checked loads and whole rows that this
// replaced):
//                          here   4 x 2 x 1  consecutive
//   128^3                  3040   3783       3448
//   101 x 83 x 120         1233              1236
//   64^3                    420    482        529
//   96^3, 20 degrees              1928       2498
//   128 x 128 x 20         1028   1210       999
//   64 x 64 x 30            281    369        548
//   128 x 128 x 10          712    772        701
//   64 x 200 x 24           894    975        926
// One contiguous eighth of the workgroups per XCD: 2371 for 1976 at 96^3, the
// XCDs' shares are too uneven.
static void rad_tiles(RadJob& j)
{
    const bool flat = (j.ntz + 3) / 4 * 4 * 8 <= j.ntz * 9;
    const bool thin = j.Z <= 12;
    j.wx = flat || j.ntz == 2 || thin ? 2 : 4;
    j.wy = flat ? 1 : thin ? 4 : 2;
    j.wz = flat ? 4 : j.ntz == 2 ? 2 : 1;
}

// Parts of the kernel rows, each a grid of workgroups of its own: a launch
// of a few workgroups per slot ends in a round of partly idle compute units
// (and a small grid never fills them), so the rows are split until there are
// four per slot (us at two, four and eight, before the tails of ranges took
// chunks of four: 96^3 voxels 2265, 2147, 2145, 101 x 83 x 120 1375, 1215,
// 1239, 128^3 3255, 3249, 3697).  Grids two tiles deep that fill the slots
// keep their rows whole: walks are short there, and a part costs more than
// the idle slots (128 x 128 x 20 1028 us whole, 1072 in two parts, 1118 in
// three).  A slot is a third of a compute unit: the row in LDS.
static int rad_parts(const RadJob& j, unsigned blocks)
{
    const unsigned slots = 3u * (unsigned)num_cus();
    if (j.wz == 2 && blocks >= slots)
        return 1;
    const unsigned parts = (4 * slots + blocks - 1) / blocks;
    return (int)std::max(1u, std::min(parts, (unsigned)j.n_rows));
}

}  // namespace ch

using namespace ch;

extern "C" {

ch_status ch_convolve_rad(const ch_plan* plan, const float* d_terma,
                          const float* d_density, float* d_dose,
                          const int32_t* d_box, int32_t accumulate,
                          void* stream)
{
    CH_REQUIRE(plan && d_terma && d_density && d_dose,
               "ch_convolve_rad: null pointer");
    CH_REQUIRE(plan->semantics == CH_SEM_RADIOLOGICAL,
               "ch_convolve_rad: the plan was built with semantics %d, not "
               "CH_SEM_RADIOLOGICAL",
               plan->semantics);
    CH_REQUIRE(plan->d_cum && plan->d_perm && plan->d_row_begin &&
                   plan->row_len >= kRadRow,
               "ch_convolve_rad: plan has no kernel rows");
    hipStream_t s = (hipStream_t)stream;
    RadJob j;
    j.X = plan->shape[0];
    j.Y = plan->shape[1];
    j.Z = plan->shape[2];
    j.n_rows = plan->n_rows;
    j.nty = (plan->shape[1] + kRadTY - 1) / kRadTY;
    j.ntz = (plan->shape[2] + kRadTZ - 1) / kRadTZ;
    rad_tiles(j);
    const int64_t groups =
        (int64_t)((plan->shape[0] + j.wx - 1) / j.wx) *
        ((j.nty + j.wy - 1) / j.wy) * ((j.ntz + j.wz - 1) / j.wz);
    CH_REQUIRE(groups * kRadWaves < INT_MAX / 2,
               "ch_convolve_rad: too many tiles");
    const unsigned blocks = (unsigned)groups;
    j.n_parts = rad_parts(j, blocks);
    ch_status st = pad_rad(plan, d_terma, d_density, &j.n_parts, s, &j.grids,
                           &j.parts);
    if (st != CH_OK)
        return st;
    capture_pin(s, plan);
    j.dose = d_dose;
    j.box = d_box;
    j.lin = plan->d_lin;
    j.seg = plan->d_k64;
    j.ftT = plan->d_ftT;
    j.meta = plan->d_meta;
    j.perm = plan->d_perm;
    j.row_begin = plan->d_row_begin;
    j.cum = plan->d_cum;
    j.row_len = plan->row_len;
    j.n_cones = plan->n_cones;
    j.accumulate = accumulate;
    LaunchTimer timer(s);
    timer.launch(gather_rad, dim3(blocks, j.n_parts), dim3(64 * kRadWaves), 0,
                 j);
    CH_HIP(hipGetLastError());
    if (j.n_parts > 1) {
        const int64_t n = (int64_t)j.X * j.Y * j.Z;
        timer.launch(rad_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     j.parts, j.n_parts, n, d_dose, accumulate);
        CH_HIP(hipGetLastError());
    }
    timer.stop();
    return CH_OK;
}

}  // extern "C"
