// Grid-to-grid resampling (nearest / trilinear / cubic B-spline) for the activity
// <-> kernel resolution round trip of the dose path.  Linear and cubic interpolation
// are separable: a workgroup interpolates the input along x once into LDS and writes a
// tile of output rows from it (resample_linear, resample_cubic); nearest, and outputs much
// coarser than the input, gather each output's neighbours (resample_kernel).  Coordinates are formed
// in FP64 so that equal spacings map every output voxel exactly onto an input voxel.
// The cubic B-spline coefficients come from a separable mirror-boundary prefilter
// (two launches: x, then y and z).
#include "pvd_internal.h"
#include "../../include/pvd_resample.h"

#include <algorithm>
#include <cmath>

namespace {

struct ResampleArgs {
    const float *in;
    float *out;
    int n[3], m[3];
    double ratio[3];   // out_spacing / in_spacing
    float scale;
    int interp;
};

// Index i (any integer) of a whole-sample symmetric (mirror) extension of [0, n).
__device__ __forceinline__ int mirror_index(int i, int n) {
    if (n == 1) return 0;
    const int p = 2 * (n - 1);
    int m = i % p;
    if (m < 0) m += p;
    return m < n ? m : p - m;
}

// Cubic B-spline weights of the 4 neighbours floor(c)-1 .. floor(c)+2 at fraction t.
__device__ __forceinline__ void bspline3_weights(float t, float w[4]) {
    const float t2 = t * t, t3 = t2 * t, u = 1.0f - t;
    w[0] = u * u * u * (1.0f / 6.0f);
    w[1] = (3.0f * t3 - 6.0f * t2 + 4.0f) * (1.0f / 6.0f);
    w[2] = (-3.0f * t3 + 3.0f * t2 + 3.0f * t + 1.0f) * (1.0f / 6.0f);
    w[3] = t3 * (1.0f / 6.0f);
}

// An output: stored past the last-level cache where the whole output is larger than it.
// 512x512x400 linear 124 -> 83-98 us, 512x512x512 nearest 285 -> 206, cubic 309 -> 273; 333x333x333
// (148 MB) would take 54 us instead of 43.
template <bool NT>
__device__ __forceinline__ void put(float *p, float v) {
    if (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// continuous index -> (lower neighbour, weight of the upper one); false if outside
__device__ __forceinline__ bool axis_pos(double c, int n, int &i0, float &f) {
    if (!(c >= -0.5 && c < n - 0.5)) return false;
    const double fl = floor(c);
    i0 = (int)fl;
    f = (float)(c - fl);
    return true;
}

// One workgroup per output row (i, j): the x/y neighbours and weights are
// uniform across the row, the threads stride along z.  Workgroups are handed
// to the 8 XCDs round-robin, so block b works on row chunk (b % 8) * G/8 + b / 8:
// each XCD walks a contiguous band of rows and neighbouring output rows find
// their shared input rows in that XCD's L2.
template <bool NT>
__global__ __launch_bounds__(256) void resample_kernel(ResampleArgs a) {
    const int rows = a.m[0] * a.m[1];
    const int G = gridDim.x;
    const int b = (G % 8 == 0) ? (int)(blockIdx.x % 8) * (G / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    for (int row = b; row < rows; row += G) {
        const int i = row / a.m[1], j = row - i * a.m[1];
        float *orow = a.out + (long long)row * a.m[2];
        int b0, b1;
        float f0, f1;
        const bool in_xy = axis_pos(i * a.ratio[0], a.n[0], b0, f0) && axis_pos(j * a.ratio[1], a.n[1], b1, f1);
        if (!in_xy) {
            for (int k = threadIdx.x; k < a.m[2]; k += blockDim.x) orow[k] = 0.0f;
            continue;
        }
        if (a.interp == PVD_INTERP_CUBIC) {
            // 4 x 4 neighbour rows (mirrored indices) with their x/y weights, uniform over the row
            float wx[4], wy[4];
            bspline3_weights(f0, wx);
            bspline3_weights(f1, wy);
            const float *rowp[16];
            float wxy[16];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int x = mirror_index(b0 - 1 + u, a.n[0]), y = mirror_index(b1 - 1 + v, a.n[1]);
                    rowp[u * 4 + v] = a.in + ((long long)x * a.n[1] + y) * a.n[2];
                    wxy[u * 4 + v] = wx[u] * wy[v];
                }
            for (int k = threadIdx.x; k < a.m[2]; k += blockDim.x) {
                int b2;
                float f2;
                float v = 0.0f;
                if (axis_pos(k * a.ratio[2], a.n[2], b2, f2)) {
                    float wz[4];
                    bspline3_weights(f2, wz);
                    int z[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) z[q] = mirror_index(b2 - 1 + q, a.n[2]);
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float *p = rowp[r];
                        const float s = fmaf(wz[0], p[z[0]], fmaf(wz[1], p[z[1]], fmaf(wz[2], p[z[2]], wz[3] * p[z[3]])));
                        v = fmaf(wxy[r], s, v);
                    }
                }
                put<NT>(orow + k, a.scale * v);
            }
            continue;
        }
        if (a.interp == PVD_INTERP_NEAREST) {
            const int x = min(max(b0 + (f0 >= 0.5f), 0), a.n[0] - 1);
            const int y = min(max(b1 + (f1 >= 0.5f), 0), a.n[1] - 1);
            const float *p = a.in + ((long long)x * a.n[1] + y) * a.n[2];
            for (int k = threadIdx.x; k < a.m[2]; k += blockDim.x) {
                int b2;
                float f2;
                float v = 0.0f;
                if (axis_pos(k * a.ratio[2], a.n[2], b2, f2)) v = p[min(max(b2 + (f2 >= 0.5f), 0), a.n[2] - 1)];
                put<NT>(orow + k, a.scale * v);
            }
            continue;
        }
        const int x0 = max(b0, 0), x1 = min(b0 + 1, a.n[0] - 1);
        const int y0 = max(b1, 0), y1 = min(b1 + 1, a.n[1] - 1);
        const float *p00 = a.in + ((long long)x0 * a.n[1] + y0) * a.n[2];
        const float *p01 = a.in + ((long long)x0 * a.n[1] + y1) * a.n[2];
        const float *p10 = a.in + ((long long)x1 * a.n[1] + y0) * a.n[2];
        const float *p11 = a.in + ((long long)x1 * a.n[1] + y1) * a.n[2];
        for (int k = threadIdx.x; k < a.m[2]; k += blockDim.x) {
            int b2;
            float f2;
            float v = 0.0f;
            if (axis_pos(k * a.ratio[2], a.n[2], b2, f2)) {
                const int z0 = max(b2, 0), z1 = min(b2 + 1, a.n[2] - 1);
                const float c00 = fmaf(f2, p00[z1] - p00[z0], p00[z0]);
                const float c01 = fmaf(f2, p01[z1] - p01[z0], p01[z0]);
                const float c10 = fmaf(f2, p10[z1] - p10[z0], p10[z0]);
                const float c11 = fmaf(f2, p11[z1] - p11[z0], p11[z0]);
                const float e0 = fmaf(f1, c01 - c00, c00);
                const float e1 = fmaf(f1, c11 - c10, c10);
                v = fmaf(f0, e1 - e0, e0);
            }
            put<NT>(orow + k, a.scale * v);
        }
    }
}

// ---------------------------------------------------------------------------------
// Separable form of the linear and cubic interpolation.  A workgroup writes a tile of
// TJ output rows (i, j0 .. j0 + TJ - 1) times KT outputs along z:
//   1. S[y][z] = the input interpolated along x, for the input rows and columns that
//      the tile reads (coalesced loads, W per element, shared by the whole tile);
//   2. cubic only: T[j][z] = S interpolated along y;
//   3. every output from 2 x 2 values of S (linear) or 4 of T (cubic) in LDS.
// The gather form above issues 8 (linear) or 64 (cubic) loads per output and is bound
// by them; here a tile costs W loads per input element it spans, so the cost follows
// the input samples per output and the pass goes to the HBM stores.  Gather -> staged:
// 251x251x196 -> 512x512x400 linear 321 -> 83-98 us by box (88 at the copy rate), cubic 2139
// -> 209; 301x301x233 -> 206x206x160 linear 51 -> 25 us, cubic 283 -> 41 (22).
constexpr int kRsBlock = 256;      // threads
constexpr int kRsU = 5;            // linear: columns per lane in flight in step 1
constexpr int kRsSpan = 64 * kRsU; // input columns of a tile (at most)
constexpr int kRsK = 8;            // linear: outputs along z per lane
constexpr int kRsCubicU = 4, kRsCubicSpan = 256;   // cubic: the same two
constexpr int kRsRows = 8;         // output rows of a tile (at most)
constexpr int kRsPlanes = 4;       // linear: output planes of a workgroup (at most)

struct StagedArgs {
    ResampleArgs a;
    int tj, kt;                    // output rows and columns of a tile
    int ti;                        // output planes of a workgroup
    int njt, nkc;                  // tiles along y and z
    int span, rows;                // LDS extents: input columns, input rows
    long long tiles;
    long long first;               // tile of this launch's first workgroup
};

// Workgroups of a launch (at most): a launch has fewer than 2^32 threads, so larger outputs take
// several.
constexpr long long kRsGrid = 1 << 21;

// Linear: an output takes the bilinear product of y and z from 2 x 2 values of S.  The
// wave issue rate bound the tile-per-output-plane form (an FP64 coordinate, a row lookup and
// a branch per output): a workgroup now keeps a lane's z positions over kRsPlanes output
// planes and gives each wave whole rows, about 12 instructions an output.
// 251x251x196 -> 512x512x400, through the cache, 150 -> 124 us (past it 83-98), 400x300x350 ->
// half 32.6 -> 29.7; eight planes a workgroup with 64 VGPRs 170.
template <bool NT>
__global__ __launch_bounds__(kRsBlock) void resample_linear(StagedArgs q) {
    extern __shared__ float rs_lds[];
    __shared__ float s_wy[kRsRows];
    __shared__ int s_ry[kRsRows][2];     // input rows of an output row (relative to ylo); < 0: outside
    const ResampleArgs &a = q.a;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    constexpr int NW = kRsBlock / 64;
    // XCD-contiguous bands of tiles (neighbouring tiles share input rows in one L2)
    const long long G = gridDim.x;
    const long long t = q.first + (long long)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
    if (t >= q.tiles) return;
    const int kc = (int)(t % q.nkc);
    const long long ij = t / q.nkc;
    const int jt = (int)(ij % q.njt), i0 = (int)(ij / q.njt) * q.ti, i1 = min(i0 + q.ti, a.m[0]);
    const int j0 = jt * q.tj, nj = min(q.tj, a.m[1] - j0);
    const int k0 = kc * q.kt, nk = min(q.kt, a.m[2] - k0);
    // first and last input row the tile can touch, 0-filled tiles aside
    const double cy1 = (j0 + nj - 1) * a.ratio[1];
    const int ylo = min(max((int)floor(fmin(j0 * a.ratio[1], 2.0e9)), 0), a.n[1] - 1);
    const int yb1 = (int)fmin(floor(cy1), (double)(a.n[1] - 1));
    const int yhi = min(yb1 + 1, a.n[1] - 1);
    const int ny = min(yhi - ylo + 1, q.rows);
    const bool in_y = j0 * a.ratio[1] < a.n[1] - 0.5;
    if (tid < nj) {
        int b = 0;
        float f = 0.0f;
        const bool in = axis_pos((j0 + tid) * a.ratio[1], a.n[1], b, f);
        s_ry[tid][0] = in ? max(b, 0) - ylo : -1;
        s_ry[tid][1] = min(b + 1, a.n[1] - 1) - ylo;
        s_wy[tid] = f;
    }
    // LDS column c is the input column zlo + c, clamped, so an output reads two consecutive
    // columns.
    const int zlo = (int)floor(fmin(k0 * a.ratio[2], 2.0e9));
    int zc[kRsU];
#pragma unroll
    for (int c = 0; c < kRsU; ++c) {
        zc[c] = min(zlo + lane + 64 * c, a.n[2] - 1);
    }
    // this lane's outputs k0 + lane + 64 u: first column (< 0: outside), fraction
    int ko[kRsK];
    float kf[kRsK];
#pragma unroll
    for (int u = 0; u < kRsK; ++u) {
        int b = 0;
        float f = 0.0f;
        const bool in = axis_pos((k0 + lane + 64 * u) * a.ratio[2], a.n[2], b, f);
        ko[u] = in ? min(b - zlo, q.span - 2) : -1;
        kf[u] = f;
    }
    float *S = rs_lds;
    for (int i = i0; i < i1; ++i) {
        int bx;
        float fx;
        const bool in_xy = axis_pos(i * a.ratio[0], a.n[0], bx, fx) && in_y;       // uniform
        if (in_xy) {
            // 1. x: the planes and weights are uniform over the workgroup
            const float *plane[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
                plane[u] = a.in + ((long long)min(max(bx + u, 0), a.n[0] - 1) * a.n[1] + ylo) * a.n[2];
            for (int y = wave; y < ny; y += NW) {
                const long long r0 = (long long)y * a.n[2];
                float v[kRsU][2];
#pragma unroll
                for (int c = 0; c < kRsU; ++c) {
                    if (64 * c >= q.span) break;
#pragma unroll
                    for (int u = 0; u < 2; ++u) v[c][u] = plane[u][r0 + zc[c]];
                }
#pragma unroll
                for (int c = 0; c < kRsU; ++c) {
                    if (64 * c >= q.span) break;
                    if (lane + 64 * c < q.span) S[y * q.span + lane + 64 * c] = fmaf(fx, v[c][1] - v[c][0], v[c][0]);
                }
            }
        }
        lds_barrier();
        // 2. y and z, and the stores: a row per wave
        for (int jj = wave; jj < nj; jj += NW) {
            float *o = a.out + ((long long)i * a.m[1] + j0 + jj) * a.m[2] + k0 + lane;
            const int r0 = in_xy ? s_ry[jj][0] : -1;                   // uniform
            if (r0 < 0) {
                for (int u = 0; u < kRsK; ++u)
                    if (lane + 64 * u < nk) o[64 * u] = 0.0f;
                continue;
            }
            const float *p = S + r0 * q.span, *p1 = S + s_ry[jj][1] * q.span;
            const float fy = s_wy[jj];
#pragma unroll
            for (int u = 0; u < kRsK; ++u) {
                if (lane + 64 * u >= nk) break;
                const int c = max(ko[u], 0);
                const float e0 = fmaf(fy, p1[c] - p[c], p[c]);
                const float e1 = fmaf(fy, p1[c + 1] - p[c + 1], p[c + 1]);
                const float x = fmaf(kf[u], e1 - e0, e0);
                put<NT>(o + 64 * u, a.scale * (ko[u] < 0 ? 0.0f : x));
            }
        }
        lds_barrier();       // S is read
    }
}

// Cubic: T[j][z] = S interpolated along y, then 4 values of T an output; an output plane per
// workgroup.  (The linear kernel's form held 135 VGPRs here and took 120x250x250 @3.3 ->
// 1.5 mm from 181 to 255 us.)
template <bool NT>
__global__ __launch_bounds__(kRsBlock) void resample_cubic(StagedArgs q) {
    constexpr int W = 4, B = 3;          // neighbours, and the furthest of them past the base index
    extern __shared__ float rs_lds[];
    __shared__ float s_wy[kRsRows][4];
    __shared__ int s_ry[kRsRows][4];     // input rows of an output row (relative to ylo); < 0: outside
    const ResampleArgs &a = q.a;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // XCD-contiguous bands of tiles (neighbouring tiles share input rows in one L2)
    const long long G = gridDim.x;
    const long long t = q.first + (long long)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
    if (t >= q.tiles) return;
    const int kc = (int)(t % q.nkc);
    const long long ij = t / q.nkc;
    const int jt = (int)(ij % q.njt), i = (int)(ij / q.njt);
    const int j0 = jt * q.tj, nj = min(q.tj, a.m[1] - j0);
    const int k0 = kc * q.kt, nk = min(q.kt, a.m[2] - k0);
    float *orow = a.out + ((long long)i * a.m[1] + j0) * a.m[2] + k0;
    int bx;
    float fx;
    // first and last input row and column the tile can touch (mirrored and clamped
    // neighbours lie within 3 of the base index), 0-filled tiles aside
    const double cy1 = (j0 + nj - 1) * a.ratio[1], cz1 = (k0 + nk - 1) * a.ratio[2];
    const int ylo = min(max((int)floor(fmin(j0 * a.ratio[1], 2.0e9)) - 2, 0), a.n[1] - 1);
    const int yb1 = (int)fmin(floor(cy1), (double)(a.n[1] - 1));
    const int yhi = min(yb1 + B, a.n[1] - 1);
    const int zlo = min(max((int)floor(fmin(k0 * a.ratio[2], 2.0e9)) - 2, 0), a.n[2] - 1);
    const int zhi = min((int)fmin(floor(cz1), (double)(a.n[2] - 1)) + B, a.n[2] - 1);
    const int ny = min(yhi - ylo + 1, q.rows), nz = min(zhi - zlo + 1, q.span);
    if (!axis_pos(i * a.ratio[0], a.n[0], bx, fx) || !(j0 * a.ratio[1] < a.n[1] - 0.5)) {
        for (int jj = 0; jj < nj; ++jj)
            for (int k = tid; k < nk; k += kRsBlock) orow[(long long)jj * a.m[2] + k] = 0.0f;
        return;
    }
    if (tid < nj) {
        int b = 0;
        float f = 0.0f;
        const bool in = axis_pos((j0 + tid) * a.ratio[1], a.n[1], b, f);
        float w[4];
        bspline3_weights(f, w);
#pragma unroll
        for (int v = 0; v < W; ++v) {
            const int y = mirror_index(b - 1 + v, a.n[1]);
            s_ry[tid][v] = in ? y - ylo : -1;
            s_wy[tid][v] = w[v];
        }
    }
    // 1. x: the planes and weights are uniform over the workgroup
    const float *plane[W];
    float wx[4];
    bspline3_weights(fx, wx);
#pragma unroll
    for (int u = 0; u < W; ++u) {
        const int x = mirror_index(bx - 1 + u, a.n[0]);
        plane[u] = a.in + (long long)x * a.n[1] * a.n[2];
    }
    float *S = rs_lds, *T = rs_lds + (size_t)q.rows * q.span;
    for (int y = wave; y < ny; y += kRsBlock / 64) {
        const long long r0 = (long long)(ylo + y) * a.n[2] + zlo;
        for (int z0 = lane; z0 < nz; z0 += 64 * kRsCubicU) {
            float v[kRsCubicU][W];
#pragma unroll
            for (int c = 0; c < kRsCubicU; ++c)
#pragma unroll
                for (int u = 0; u < W; ++u) v[c][u] = plane[u][r0 + min(z0 + 64 * c, nz - 1)];
#pragma unroll
            for (int c = 0; c < kRsCubicU; ++c) {
                if (z0 + 64 * c < nz)
                    S[y * q.span + z0 + 64 * c] =
                        fmaf(wx[3], v[c][3], fmaf(wx[2], v[c][2], fmaf(wx[1], v[c][1], wx[0] * v[c][0])));
            }
        }
    }
    __syncthreads();
    // 2. y
    for (int jj = wave; jj < nj; jj += kRsBlock / 64) {
        if (s_ry[jj][0] < 0) continue;
        const float *s0 = S + s_ry[jj][0] * q.span, *s1 = S + s_ry[jj][1] * q.span;
        const float *s2 = S + s_ry[jj][2] * q.span, *s3 = S + s_ry[jj][3] * q.span;
        const float w0 = s_wy[jj][0], w1 = s_wy[jj][1], w2 = s_wy[jj][2], w3 = s_wy[jj][3];
        for (int z = lane; z < nz; z += 64)
            T[jj * q.span + z] = fmaf(w3, s3[z], fmaf(w2, s2[z], fmaf(w1, s1[z], w0 * s0[z])));
    }
    __syncthreads();
    // 3. z, and the stores
    for (int k = tid; k < nk; k += kRsBlock) {
        int b = 0;
        float f = 0.0f;
        const bool inz = axis_pos((k0 + k) * a.ratio[2], a.n[2], b, f);
        float wz[4];
        int z[W];
        bspline3_weights(f, wz);
#pragma unroll
        for (int v = 0; v < W; ++v) {
            z[v] = inz ? mirror_index(b - 1 + v, a.n[2]) - zlo : 0;
        }
        for (int jj = 0; jj < nj; ++jj) {
            float x = 0.0f;
            if (inz && s_ry[jj][0] >= 0) {
                const float *p = T + jj * q.span;
                x = fmaf(wz[3], p[z[3]], fmaf(wz[2], p[z[2]], fmaf(wz[1], p[z[1]], wz[0] * p[z[0]])));
            }
            put<NT>(orow + (long long)jj * a.m[2] + k, a.scale * x);
        }
    }
}

// Largest extent of input indices, past + 1 beyond the last base index, that `cnt`
// consecutive outputs span (any start).
int staged_extent(double ratio, int cnt, int past) {
    // (one more than the real numbers need: the products are rounded)
    return (int)std::min(1.0e9, std::floor((cnt - 1) * ratio)) + 3 + past;
}

// Coarsest output / input spacing (along y and z) that takes the staged form: beyond it
// a tile spans more input than its outputs use and the gather is faster.  512x512x400
// inputs, gather / staged us: linear 102 / 97 at 2.04, 38 / 52 at 3.0; cubic 225 / 110 at
// 3.0, 99 / 72 at 4.5, 32 / 34 at 8.3.
constexpr double kStagedLinear = 2.5, kStagedCubic = 8.0;

bool streamed(const ResampleArgs &a) { return 4LL * a.m[0] * a.m[1] * a.m[2] > PVD_STREAM_BYTES; }

template <typename Kernel>
hipError_t launch_staged(Kernel kernel, StagedArgs &q, int tj, hipStream_t st) {
    const size_t lds = sizeof(float) * q.span * (size_t)(q.rows + tj);
    if (q.span > kRsSpan || lds > 48 * 1024) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    for (q.first = 0; q.first < q.tiles && e == hipSuccess; q.first += kRsGrid) {
        const long long grid = (std::min(q.tiles - q.first, kRsGrid) + 7) / 8 * 8;
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kRsBlock), lds, st, q);
        e = hipGetLastError();
    }
    return e;
}

hipError_t launch_linear(const ResampleArgs &a, hipStream_t st) {
    StagedArgs q{};
    q.a = a;
    // outputs along z that a row's lanes and a tile's input columns hold, in equal tiles
    q.kt = std::min(a.m[2], 64 * kRsK);
    if (staged_extent(a.ratio[2], q.kt, 1) > kRsSpan)
        q.kt = std::max(1, std::min(q.kt, (int)((kRsSpan - 9) / a.ratio[2])));
    q.nkc = (a.m[2] + q.kt - 1) / q.kt;
    q.kt = (a.m[2] + q.nkc - 1) / q.nkc;
    q.nkc = (a.m[2] + q.kt - 1) / q.kt;
    q.span = staged_extent(a.ratio[2], q.kt, 1);
    q.tj = kRsRows;
    while (q.tj > 1 && staged_extent(a.ratio[1], q.tj, 1) > 32) q.tj /= 2;
    q.rows = std::min(staged_extent(a.ratio[1], q.tj, 1), a.n[1]);
    q.njt = (a.m[1] + q.tj - 1) / q.tj;
    // planes per workgroup: fewer while that leaves less than eight workgroups a CU
    q.ti = kRsPlanes;
    const long long per = (long long)q.njt * q.nkc;
    while (q.ti > 1 && per * ((a.m[0] + q.ti - 1) / q.ti) < 2048) q.ti /= 2;
    q.tiles = per * ((a.m[0] + q.ti - 1) / q.ti);
    return streamed(a) ? launch_staged(resample_linear<true>, q, 0, st)
                       : launch_staged(resample_linear<false>, q, 0, st);
}

hipError_t launch_cubic(const ResampleArgs &a, hipStream_t st) {
    StagedArgs q{};
    q.a = a;
    const auto extent = [&](int d, int cnt) { return std::min(staged_extent(a.ratio[d], cnt, 5), a.n[d]); };
    // outputs along z whose input columns fit a tile
    q.kt = a.m[2];
    if (extent(2, q.kt) > kRsCubicSpan) {
        q.kt = std::max(1, std::min(a.m[2], (int)((kRsCubicSpan - 9) / a.ratio[2])));
        const int nt = (a.m[2] + q.kt - 1) / q.kt;     // equal tiles
        q.kt = (a.m[2] + nt - 1) / nt;
    }
    q.kt = std::min(q.kt, 2048);
    q.span = extent(2, q.kt);
    q.tj = kRsRows;
    while (q.tj > 1 && extent(1, q.tj) > 32) q.tj /= 2;
    q.rows = extent(1, q.tj);
    q.ti = 1;
    q.njt = (a.m[1] + q.tj - 1) / q.tj;
    q.nkc = (a.m[2] + q.kt - 1) / q.kt;
    q.tiles = (long long)a.m[0] * q.njt * q.nkc;
    return streamed(a) ? launch_staged(resample_cubic<true>, q, q.tj, st)
                       : launch_staged(resample_cubic<false>, q, q.tj, st);
}

// Cubic B-spline prefilter: c[i] = sum_k sqrt(3) z^|k| w[i + k], z = sqrt(3) - 2, as one
// recursion from each side over a window of the line (Unser's factorisation of the
// inverse).  A window starts and ends kBsK samples beyond its outputs, mirrored at the
// volume's ends: the tail left out is below z^15 = 2.6e-9 of a sample.
constexpr int kBsK = 14;
constexpr float kBsZ0 = (float)(1.7320508075688772935 - 2.0), kBsGain = 1.7320508075688772935f;

// R outputs from the R + 28 samples get(0) ..: p and m are the sums over k <= 0 and k > 0.
// A recursion never forgets an infinity or a NaN, which may reach 14 samples and no
// further: a window that ends with one takes the 29-tap sum of each output.
template <int R, typename Get>
__device__ __forceinline__ void bs_line(const Get &get, float (&c)[R]) {
    float w[R + 2 * kBsK];
#pragma unroll
    for (int i = 0; i < R + 2 * kBsK; ++i) w[i] = get(i);
    float p = 0.0f, m = 0.0f;
#pragma unroll
    for (int i = 0; i < R + kBsK; ++i) {
        p = fmaf(kBsZ0, p, w[i]);
        if (i >= kBsK) c[i - kBsK] = p;
    }
#pragma unroll
    for (int i = R + 2 * kBsK - 1; i >= kBsK; --i) {
        if (i < R + kBsK) c[i - kBsK] = kBsGain * fmaf(kBsZ0, m, c[i - kBsK]);
        m = fmaf(kBsZ0, m, w[i]);
    }
    if (!isfinite(p) || !isfinite(m)) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            float h = kBsGain, acc = h * get(i + kBsK);
            for (int k = 1; k <= kBsK; ++k) {
                h *= kBsZ0;
                acc = fmaf(h, get(i + kBsK - k) + get(i + kBsK + k), acc);
            }
            c[i] = acc;
        }
    }
}

// The prefilter runs along x in one launch and along y and z in a second.  A thread owns
// one column of R consecutive outputs along the filtered axis: R + 28 loads, all issued
// before the first is used, and four operations an output (43 as a 29-tap FIR).
// 301x301x233: x 52 us, yz 104 -> 86, the call 184 -> 170 (32 each at the copy rate: the 28 samples a thread reads
// beyond its outputs, and the yz launch's three barriers with 20 waves per CU; 32 or 40
// rows a tile took fewer samples but fewer waves, and 180 us for the whole call instead
// of 173).
constexpr int kBsX = 32;           // outputs per thread along x
constexpr int kBsY = 24;           // outputs per thread along y (rows of the z tile)
constexpr int kBsZ = 27;           // outputs per unit along z (odd: neighbouring units in other LDS banks)
constexpr int kBsCols = 17 * kBsZ + 2 * kBsK;      // columns of a z tile (at most): 487

__global__ __launch_bounds__(256) void bspline_x(const float *__restrict__ src, float *__restrict__ dst, int n0,
                                                 long long plane, unsigned gx, unsigned first) {
    const unsigned b = first + blockIdx.x, bx = b / gx;
    const long long p = (b - bx * gx) * 256LL + threadIdx.x;
    const int x0 = (int)bx * kBsX;
    const long long pc = p < plane ? p : plane - 1;
    float c[kBsX];
    bs_line([&](int i) { return src[(long long)mirror_index(min(x0 + i - kBsK, n0 - 1 + kBsK), n0) * plane + pc]; }, c);
    if (p >= plane) return;
#pragma unroll
    for (int i = 0; i < kBsX; ++i)
        if (x0 + i < n0) dst[(long long)(x0 + i) * plane + p] = c[i];
}

// y in registers, then z through LDS: column c of a tile holds z = mirror(z0 - 14 + c),
// kBsY rows; phase 2 takes units of kBsZ consecutive outputs of a row (one per thread,
// kBsZ + 28 LDS words), puts the results back into the tile and stores whole rows.
__global__ __launch_bounds__(512) void bspline_yz(const float *__restrict__ src, float *__restrict__ dst, int n1,
                                                  int n2, int zt, int ld, int nzt, int nyt, long long tiles) {
    extern __shared__ float tile[];
    const int tid = threadIdx.x;
    const int cols = zt + 2 * kBsK;
    const int upr = zt / kBsZ;                       // units per row
    const bool unit = tid < kBsY * upr;              // at most blockDim (host)
    float *row = tile + (unit ? tid / upr * ld + tid % upr * kBsZ : 0);
    for (long long t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int z0 = (int)(t % nzt) * zt, y0 = (int)(t / nzt % nyt) * kBsY;
        const long long base = t / nzt / nyt * n1 * n2;
        if (tid < cols) {
            const int z = mirror_index(min(z0 + tid - kBsK, n2 - 1 + kBsK), n2);
            const float *col = src + base + z;
            float c[kBsY];
            bs_line([&](int i) { return col[(long long)mirror_index(min(y0 + i - kBsK, n1 - 1 + kBsK), n1) * n2]; }, c);
#pragma unroll
            for (int i = 0; i < kBsY; ++i) tile[i * ld + tid] = c[i];
        }
        __syncthreads();
        float c[kBsZ];
        if (unit) bs_line([&](int i) { return row[i]; }, c);
        __syncthreads();
        if (unit) {
#pragma unroll
            for (int i = 0; i < kBsZ; ++i) row[i] = c[i];
        }
        __syncthreads();
        const int nz = min(zt, n2 - z0), rows = min(kBsY, n1 - y0);
        for (int i = 0; i < rows; ++i)
            for (int k = tid; k < nz; k += blockDim.x) dst[base + (long long)(y0 + i) * n2 + z0 + k] = tile[i * ld + k];
        __syncthreads();
    }
}

}  // namespace

extern "C" int pvd_bspline_prefilter(const float *in, int n0, int n1, int n2, float *coef, float *tmp,
                                     void *stream) {
    if (!in || !coef || !tmp) return pvd_set_error(PVD_EINVAL, "null argument");
    if (n0 < 1 || n1 < 1 || n2 < 1) return pvd_set_error(PVD_EINVAL, "grid extents must be >= 1");
    if (coef == in || tmp == in || coef == tmp) return pvd_set_error(PVD_EINVAL, "coef, tmp and in must differ");
    const long long plane = (long long)n1 * n2;
    const long long gx = (plane + 255) / 256, blocks_x = gx * ((n0 + (long long)kBsX - 1) / kBsX);
    if (blocks_x > 0xffffffffLL) return pvd_set_error(PVD_ENOTSUP, "grid too large");     // 4e12 bytes and more
    const int nyt = (n1 + kBsY - 1) / kBsY;
    // z tiles of equal width, a multiple of the unit; a thread per column
    const int nt = (n2 + kBsCols - 2 * kBsK - 1) / (kBsCols - 2 * kBsK);
    const int zt = ((n2 + nt - 1) / nt + kBsZ - 1) / kBsZ * kBsZ;
    const int block = (std::max(zt + 2 * kBsK, kBsY * (zt / kBsZ)) + 63) / 64 * 64;
    const int ld = zt + 2 * kBsK + 1;
    hipStream_t st = (hipStream_t)stream;
    hipError_t e = hipSuccess;
    for (long long first = 0; first < blocks_x; first += kRsGrid) {
        hipLaunchKernelGGL(bspline_x, dim3((unsigned)std::min(blocks_x - first, kRsGrid)), dim3(256), 0, st, in, tmp, n0,
                           plane, (unsigned)gx, (unsigned)first);
        e = hipGetLastError();
        if (e != hipSuccess) return pvd_hip_error(e, "launch B-spline prefilter");
    }
    const int nzt = (n2 + zt - 1) / zt;
    const long long tiles = (long long)n0 * nyt * nzt;
    hipLaunchKernelGGL(bspline_yz, dim3((unsigned)std::min(tiles, kRsGrid)), dim3(block),
                       sizeof(float) * kBsY * ld, st, (const float *)tmp, coef, n1, n2, zt, ld, nzt, nyt, tiles);
    e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch B-spline prefilter");
}

extern "C" int pvd_resample(const float *in, int n0, int n1, int n2, const double *in_spacing, float *out, int m0,
                            int m1, int m2, const double *out_spacing, int interp, double scale, void *stream) {
    if (!in || !out || !in_spacing || !out_spacing) return pvd_set_error(PVD_EINVAL, "null argument");
    if (n0 < 1 || n1 < 1 || n2 < 1 || m0 < 1 || m1 < 1 || m2 < 1)
        return pvd_set_error(PVD_EINVAL, "grid extents must be >= 1");
    if (interp != PVD_INTERP_NEAREST && interp != PVD_INTERP_LINEAR && interp != PVD_INTERP_CUBIC)
        return pvd_set_error(PVD_EINVAL, "interp must be PVD_INTERP_NEAREST, PVD_INTERP_LINEAR or PVD_INTERP_CUBIC");
    ResampleArgs a{};
    a.in = in;
    a.out = out;
    a.n[0] = n0; a.n[1] = n1; a.n[2] = n2;
    a.m[0] = m0; a.m[1] = m1; a.m[2] = m2;
    for (int d = 0; d < 3; ++d) {
        if (!(in_spacing[d] > 0.0) || !(out_spacing[d] > 0.0))
            return pvd_set_error(PVD_EINVAL, "spacings must be > 0");
        a.ratio[d] = out_spacing[d] / in_spacing[d];
    }
    a.scale = (float)scale;
    a.interp = interp;
    if ((long long)m0 * m1 > 0x7fffffffLL) return pvd_set_error(PVD_ENOTSUP, "too many output rows");
    long long g = (long long)m0 * m1;
    if (g > 65536) g = 65536;
    hipError_t e;
    if (interp == PVD_INTERP_LINEAR && a.ratio[2] <= kStagedLinear && a.ratio[1] <= kStagedLinear) {
        e = launch_linear(a, (hipStream_t)stream);
    } else if (interp == PVD_INTERP_CUBIC && a.ratio[2] <= kStagedCubic && a.ratio[1] <= kStagedCubic) {
        e = launch_cubic(a, (hipStream_t)stream);
    } else {
        if (streamed(a)) hipLaunchKernelGGL(resample_kernel<true>, dim3((unsigned)g), dim3(256), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL(resample_kernel<false>, dim3((unsigned)g), dim3(256), 0, (hipStream_t)stream, a);
        e = hipGetLastError();
    }
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch resample");
}
