// HU -> (metal fill) -> class bits and mass density, one pass over the CT.
//
// The reference (tissue/composition.py:72-94) marks metal (HU > 2000), sets it
// to NaN, smooths nan_to_num(image) with scipy.ndimage.gaussian_filter (sigma
// 1, 'reflect', truncate 4) and writes the smoothed values back into the metal
// voxels only.  The smoothing is needed at metal voxels alone, so this kernel
// evaluates the separable Gaussian there as a direct (2r+1)^3 weighted sum in
// FP64 (per-axis reflected indices: the same linear map as three 1-D passes)
// and streams every other voxel straight through.  The pass is HBM-bound:
// 4 B read and up to 9 B written per voxel.
#include "pvd_internal.h"
#include "../../include/pvd_tissue.h"

#include <cfloat>
#include <cmath>

namespace {

struct TissueArgs {
    const float *ct;
    float *corrected;
    unsigned char *bits;
    float *density;
    int n0, n1, n2;
    int radius;
    int handle;
    float metal;
    int ncls;
    int nmat;
    float clo[PVD_TISSUE_MAX_CLASSES];
    float chi[PVD_TISSUE_MAX_CLASSES];
    float mlo[PVD_TISSUE_MAX_MATERIALS];
    float mden[PVD_TISSUE_MAX_MATERIALS];
    double w[2 * PVD_TISSUE_MAX_RADIUS + 1];
};

// scipy.ndimage 'reflect' (half-sample symmetric: d c b a | a b c d | d c b a),
// folded as often as needed when the radius exceeds the extent.
__device__ __forceinline__ int reflect(int i, int n) {
    const int p = 2 * n;
    i %= p;
    if (i < 0) i += p;
    return i < n ? i : p - 1 - i;
}

// nan_to_num of the image whose metal voxels were set to NaN (float32 data).
__device__ __forceinline__ double fill_source(float c, float metal) {
    if (c > metal || c != c) return 0.0;
    if (c == -INFINITY) return -(double)FLT_MAX;
    return (double)c;
}

// Smoothed values of V consecutive voxels of one z-row (x, y, z0 .. z0+V-1), for the voxels
// flagged in `which`, at the run-time radius.  For each of the (2r+1)^2 (dx, dy) rows the lane
// issues all V+2r reflected z-loads of that row before using them, so a metal voxel costs
// (2r+1)^2 load round trips, shared by the V voxels.
template <int V>
__device__ void metal_fill_row(const TissueArgs &a, int x, int y, int z0, unsigned which, float *h) {
    const int r = a.radius, side = 2 * r + 1;
    constexpr int W = V + 2 * PVD_TISSUE_MAX_RADIUS;
    double acc[V];
#pragma unroll
    for (int k = 0; k < V; ++k) acc[k] = 0.0;
    for (int dx = -r; dx <= r; ++dx) {
        const long long px = (long long)reflect(x + dx, a.n0) * a.n1;
        for (int dy = -r; dy <= r; ++dy) {
            const float *row = a.ct + (px + reflect(y + dy, a.n1)) * a.n2;
            const double wxy = a.w[dx + r] * a.w[dy + r];
            float win[W];
#pragma unroll
            for (int j = 0; j < W; ++j)
                if (j < V + 2 * r) win[j] = row[reflect(z0 - r + j, a.n2)];
#pragma unroll
            for (int k = 0; k < V; ++k) {
                if (!(which & (1u << k))) continue;
                double s = 0.0;
                for (int dz = 0; dz < side; ++dz) s += a.w[dz] * fill_source(win[k + dz], a.metal);
                acc[k] += wxy * s;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < V; ++k)
        if (which & (1u << k)) h[k] = (float)acc[k];
}

// Class bits and density of one HU value.  The loops have compile-time trip
// counts (NM materials, all PVD_TISSUE_MAX_CLASSES classes; the host pads unused
// entries with bounds that never match) so the table stays in scalar registers.
template <int NM>
__device__ __forceinline__ void classify(const TissueArgs &a, float v, unsigned char &bits, float &dens) {
    unsigned b = 0;
#pragma unroll
    for (int c = 0; c < PVD_TISSUE_MAX_CLASSES; ++c) b |= (unsigned)(v >= a.clo[c] && v <= a.chi[c]) << c;
    bits = (unsigned char)b;
    float d = a.mden[0];
#pragma unroll
    for (int i = 1; i < NM; ++i) d = (v >= a.mlo[i]) ? a.mden[i] : d;
    dens = (v == v) ? d : v;
}

// Voxels are streamed V per lane (V = 4 with 16-byte aligned maps, whatever the extents: an
// item of four voxels may span two z-rows, which only its fill has to know).  Each lane issues the loads of kItems grid-stride
// items before using any, so a wavefront keeps kItems x 64 x 4V bytes in flight.
// Lanes whose voxels hold metal do not fill them in place (81 dependent load rounds for
// radius 4, while a rod along z puts 40 such lanes into one wave): they list their items in
// LDS, and the workgroup fills the listed items together, a wave per item.  512x512x400 with
// a plate and a rod of 22,000 metal voxels: 505 -> 329 us (294 without implants: 4.6 TB/s,
// the copy rate is 5.0); 511x300x401 580 -> 181, 200^3 with two implants 233 -> 37.  Volumes
// within the last-level cache and without metal pay for the list: 200^3 23.1 -> 28.1, 256x256x200
// 36.8 -> 39.5.
constexpr int kItems = 4;
constexpr int kTissueGrid = 2048;       // workgroups (at most)
constexpr int kTissueBlock = 512;
// Consecutive items a workgroup takes at once: 512 bytes of each map, half a wave.  Fewer
// spread an implant's metal over more workgroups, more keep the stream's bursts long.
// 512x512x400 with no, one, two implants, us: 64 items 311 / 329 / 372, 32 items 303 / 325 /
// 351, 16 items 332 / 363 / 368.
constexpr int kTissueChunk = 32;
// Chunks a workgroup has before there are more than kTissueFew workgroups (a CU each): a
// chunk each costs 64^3 12.1 us without metal, this rule 4.2 (100^3 13.4 -> 6.8, 128^3 14.6 ->
// 11.1).  With two implants 64^3 18.8 -> 15.1, 128^3 19.0 -> 20.6; 32 chunks 26.4 there.
constexpr int kTissuePer = 16, kTissueFew = 256;
// A workgroup with at least kTissueDense items of metal, kTissuePerSpan or more of them to each
// span of kSpan voxels that holds any, fills whole spans: a third of the instructions an item
// where most items are listed.  200^3, single items -> spans: its first two thirds metal 2640 ->
// 486 us, random 30 % 3175 -> 725, random 10 % (4 items a span) 1557 -> 700; random 2 % (1.5)
// would take 500 instead of 453.
constexpr int kTissueDense = 16, kTissuePerSpan = 3;

template <int NM>
__device__ __forceinline__ void tissue_store1(const TissueArgs &a, long long v, float h) {
    unsigned char b;
    float d;
    classify<NM>(a, h, b, d);
    if (a.corrected) a.corrected[v] = h;
    if (a.bits) a.bits[v] = b;
    if (a.density) a.density[v] = d;
}

// Maps that do not fit the last-level cache are stored past it: 512x512x400 with no, one, two
// implants 303 / 325 / 352 -> 295 / 315 / 338 us, 512x300x401 with none 184 -> 149.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned char u8x4 __attribute__((ext_vector_type(4)));
template <int V, int NM, bool NT>
__device__ __forceinline__ void tissue_store(const TissueArgs &a, long long i, const float *h) {
    if constexpr (V == 4) {
        unsigned char b[V];
        float d[V];
#pragma unroll
        for (int k = 0; k < V; ++k) classify<NM>(a, h[k], b[k], d[k]);
        const f32x4 h4 = {h[0], h[1], h[2], h[3]}, d4 = {d[0], d[1], d[2], d[3]};
        const u8x4 b4 = {b[0], b[1], b[2], b[3]};
        if constexpr (NT) {
            if (a.corrected) __builtin_nontemporal_store(h4, reinterpret_cast<f32x4 *>(a.corrected) + i);
            if (a.bits) __builtin_nontemporal_store(b4, reinterpret_cast<u8x4 *>(a.bits) + i);
            if (a.density) __builtin_nontemporal_store(d4, reinterpret_cast<f32x4 *>(a.density) + i);
        } else {
            if (a.corrected) reinterpret_cast<f32x4 *>(a.corrected)[i] = h4;
            if (a.bits) reinterpret_cast<u8x4 *>(a.bits)[i] = b4;
            if (a.density) reinterpret_cast<f32x4 *>(a.density)[i] = d4;
        }
    } else {
        tissue_store1<NM>(a, i, h[0]);
    }
}

template <int V>
__device__ __forceinline__ void tissue_load(const TissueArgs &a, long long i, float *h) {
    if constexpr (V == 4) {
        const float4 q = reinterpret_cast<const float4 *>(a.ct)[i];
        h[0] = q.x;
        h[1] = q.y;
        h[2] = q.z;
        h[3] = q.w;
    } else {
        h[0] = a.ct[i];
    }
}

template <int V>
__device__ __forceinline__ unsigned metal_of(const TissueArgs &a, const float *h) {
    unsigned which = 0;
#pragma unroll
    for (int k = 0; k < V; ++k) which |= (unsigned)(h[k] > a.metal) << k;
    return which;
}

// The lane, opaque: what the fills derive from it (rows, columns, weights' places) is computed
// where it is used and not kept in registers over the streaming loop.
__device__ __forceinline__ int fill_lane() {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    return lane;
}

// Fill of the cnt <= V voxels of item i by a wave, radius 4 (sw: the nine weights in LDS):
// lane (g, j) sums wxy * source over the rows (dx, dy) g, g + G, ... at z = z0 - 4 + j (W
// consecutive floats of a row per group: coalesced), the groups are added, and the outputs
// take the z weights of the W sums.  An item that spans two z-rows takes a turn for each.
template <int V, int NM>
__device__ __forceinline__ void metal_fill_wave(const TissueArgs &a, const double *sw, long long i, int cnt) {
    constexpr int R = 4, W = V + 2 * R, G = 64 / W, ROWS = 81, PER = (ROWS + G - 1) / G;
    const int lane = fill_lane(), g = lane / W, j = lane - g * W;
    auto fold = [](int k, int n) { return k < 0 || k >= n ? reflect(k, n) : k; };
    long long xy = i * V / a.n2;
    int z0 = (int)(i * V - xy * a.n2);
#pragma unroll 1
    for (int done = 0; done < cnt;) {
        const int run = min(cnt - done, a.n2 - z0);
        const int x = (int)(xy / a.n1), y = (int)(xy - (long long)x * a.n1);
        const int z = fold(z0 - R + j, a.n2);
        double acc = 0.0;
#pragma unroll 6
        for (int t = 0; t < PER; ++t) {
            const int row = g + G * t;
            const bool on = g < G && row < ROWS;
            const int dx = on ? row / 9 : R, dy = on ? row % 9 : R;
            const float c = a.ct[((long long)fold(x + dx - R, a.n0) * a.n1 + fold(y + dy - R, a.n1)) * a.n2 + z];
            acc += (on ? sw[dx] * sw[dy] : 0.0) * fill_source(c, a.metal);
        }
        double sum = 0.0;                        // lane j < W: all rows at z0 - 4 + j
#pragma unroll
        for (int q = 0; q < G; ++q) sum += __shfl(acc, (j + q * W) & 63);
        double out = 0.0;                        // lane k < run
#pragma unroll
        for (int dz = 0; dz < 2 * R + 1; ++dz) out += sw[dz] * __shfl(sum, (lane + dz) & 63);
        if (lane < run) {                        // each of these lanes writes its voxel
            const long long v = xy * a.n2 + z0 + lane;
            const float c = a.ct[v];
            tissue_store1<NM>(a, v, c > a.metal ? (float)out : c);
        }
        done += run;
        z0 = 0;
        ++xy;
    }
}

// Fill of `run` <= kSpan consecutive voxels of a z-row by a wave, radius 4: a lane per column
// z0 - 4 + lane sums it over the 81 rows.  Voxels without metal keep their value.  (The offsets
// of a plane's nine rows lie in lanes 0..8: as uniform addresses they took the scalar registers
// of the streaming loop's tables, 511x300x401 without metal 150 -> 161 us.)
constexpr int kSpan = 48;                // a third of a chunk's voxels at most, with 8 more columns
template <int NM>
__device__ __forceinline__ void metal_fill_span(const TissueArgs &a, const double *sw, int x, int y, int z0, int run) {
    constexpr int R = 4;
    const int lane = fill_lane();
    auto fold = [](int k, int n) { return k < 0 || k >= n ? reflect(k, n) : k; };
    const int z = fold(z0 - R + lane, a.n2);
    const long long yo = (long long)fold(y + min(lane, 2 * R) - R, a.n1) * a.n2;
    double sum = 0.0;
#pragma unroll 1
    for (int dx = 0; dx <= 2 * R; ++dx) {
        const float *col = a.ct + (long long)fold(x + dx - R, a.n0) * a.n1 * a.n2 + z;
        float c[2 * R + 1];
#pragma unroll
        for (int dy = 0; dy <= 2 * R; ++dy) c[dy] = col[__shfl(yo, dy)];
        double row = 0.0;
#pragma unroll
        for (int dy = 0; dy <= 2 * R; ++dy) row += sw[dy] * fill_source(c[dy], a.metal);
        sum += sw[dx] * row;
    }
    double out = 0.0;
#pragma unroll
    for (int dz = 0; dz <= 2 * R; ++dz) out += sw[dz] * __shfl(sum, (lane + dz) & 63);
    if (lane < run) {
        const long long v = ((long long)x * a.n1 + y) * a.n2 + z0 + lane;
        const float c = a.ct[v];
        tissue_store1<NM>(a, v, c > a.metal ? (float)out : c);
    }
}

// (More than 16 materials: held to 128 registers, two workgroups a CU; 200^3 51 -> 37 us.)
template <bool VEC, int NM, bool NT = false>
__global__ __launch_bounds__(kTissueBlock) __attribute__((amdgpu_waves_per_eu(NM == 32 ? 4 : 1))) void tissue_map(TissueArgs a, long long nitems, long long n) {
    constexpr int V = VEC ? 4 : 1;
    __shared__ unsigned short list[kItems * kTissueBlock];
    __shared__ int count;
    __shared__ double sw[9];
    constexpr int kChunks = kItems * kTissueBlock / kTissueChunk;
    constexpr int kUnits = (kTissueChunk * V + kSpan - 1) / kSpan;
    __shared__ unsigned flags[kChunks];
    const int tid = threadIdx.x;
    // Chunks of items are dealt round the workgroups, so an implant (whose metal sits in
    // neighbouring rows) is spread over many of them.
    const long long stride = (long long)gridDim.x * kTissueBlock;
    auto item = [&](long long b0, int e) {                   // e = u * kTissueBlock + thread
        return b0 + ((long long)(e / kTissueChunk) * gridDim.x + blockIdx.x) * kTissueChunk + e % kTissueChunk;
    };
    if (tid == 0) count = 0;
    if (tid < 9) sw[tid] = a.w[tid];
    lds_barrier();
    const long long whole = n / V;                           // items of V voxels; one more if n % V
    for (long long b0 = 0; b0 + blockIdx.x * (long long)kTissueChunk < nitems; b0 += kItems * stride) {
        float h[kItems][V];
        unsigned which[kItems];
#pragma unroll
        for (int u = 0; u < kItems; ++u)                      // (clamped, so that no branch splits the loads)
            tissue_load<V>(a, min(item(b0, u * kTissueBlock + tid), whole - 1), h[u]);
        int mine = 0;
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const long long i = item(b0, u * kTissueBlock + tid);
            // (without artefact handling the metal threshold is infinite); the last n % V
            // voxels go through the list as well
            which[u] = i < whole ? metal_of<V>(a, h[u]) : i < nitems ? 1u : 0u;
            mine += which[u] ? 1 : 0;
            if (i < whole && !which[u]) tissue_store<V, NM, NT>(a, i, h[u]);
        }
        int at = mine ? atomicAdd(&count, mine) : 0;
#pragma unroll
        for (int u = 0; u < kItems; ++u)
            if (which[u]) list[at++] = (unsigned short)(u * kTissueBlock + tid);
        lds_barrier();
        const int m = count;
        lds_barrier();
        if (m == 0) continue;                            // uniform
        if (tid == 0) count = 0;
        bool spans = false;
        if (m >= kTissueDense) {
            static_assert(kTissueChunk == 32 && kChunks == 64, "a word of flags per chunk, a lane per word");
            if (tid < kChunks) flags[tid] = 0u;
            lds_barrier();
            for (int k = tid; k < m; k += kTissueBlock) atomicOr(&flags[list[k] >> 5], 1u << (list[k] & 31));
            lds_barrier();
            const unsigned f = flags[tid & 63];
            constexpr unsigned part = kUnits == 1 ? ~0u : (1u << (kSpan / V) % 32) - 1u;
            int units = 0;                               // spans that hold metal
#pragma unroll
            for (int q = 0; q < kUnits; ++q) units += __popcll(__ballot(((f >> (q * (kSpan / V))) & part) != 0u));
            spans = m >= kTissuePerSpan * units;
        }
        if (!spans) {
            for (int k = tid >> 6; k < m; k += kTissueBlock / 64) {
                const long long i = item(b0, list[k]);
                metal_fill_wave<V, NM>(a, sw, i, (int)min((long long)V, n - i * V));
            }
        } else {
            for (int u = tid >> 6; u < kChunks * kUnits; u += kTissueBlock / 64) {
                const int c = u / kUnits;
                const unsigned on = flags[c];
                const long long v0 = item(b0, c * kTissueChunk) * V;
                int p = (u - c * kUnits) * kSpan;
                const int end = (int)min((long long)min(p + kSpan, kTissueChunk * V), n - v0);
                while (p < end) {
                    const unsigned rest = on >> (p / V);
                    if (!rest) break;
                    if (!(rest & 1u)) {                  // to the next item with metal
                        p = (p / V + __ffs(rest) - 1) * V;
                        continue;
                    }
                    const long long xy = (v0 + p) / a.n2;
                    const int z0 = (int)(v0 + p - xy * a.n2), x = (int)(xy / a.n1);
                    const int run = min(end - p, a.n2 - z0);
                    metal_fill_span<NM>(a, sw, x, (int)(xy - (long long)x * a.n1), z0, run);
                    p += run;
                }
            }
        }
        lds_barrier();                                   // list and count are free again
    }
}

// Any other radius: a lane holding metal fills it in place (VEC: n2 % 4 == 0, so an item lies in
// one z-row).  Workgroups of 256 threads over consecutive items: the window of a run-time radius
// takes 140-156 registers, which leave one workgroup of 512 on a CU (512x512x200 at sigma 0.6
// with no, two implants 191, 308 us; in workgroups of 512 with the chunks above 511, 708).
constexpr int kRowBlock = 256, kRowGrid = 4096;
template <bool VEC, int NM>
__global__ __launch_bounds__(kRowBlock) void tissue_map_rows(TissueArgs a, long long nitems) {
    constexpr int V = VEC ? 4 : 1;
    const long long stride = (long long)gridDim.x * kRowBlock;
    for (long long i0 = blockIdx.x * (long long)kRowBlock + threadIdx.x; i0 < nitems; i0 += kItems * stride) {
        float h[kItems][V];
#pragma unroll
        for (int u = 0; u < kItems; ++u)
            if (i0 + u * stride < nitems) tissue_load<V>(a, i0 + u * stride, h[u]);
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const long long i = i0 + u * stride;
            if (i >= nitems) continue;
            const unsigned which = metal_of<V>(a, h[u]);
            if (which) {
                const long long v0 = i * V, xy = v0 / a.n2;
                metal_fill_row<V>(a, (int)(xy / a.n1), (int)(xy % a.n1), (int)(v0 % a.n2), which, h[u]);
            }
            tissue_store<V, NM, false>(a, i, h[u]);
        }
    }
}

bool aligned(const void *p, uintptr_t k) { return (reinterpret_cast<uintptr_t>(p) & (k - 1)) == 0; }

}  // namespace

extern "C" int pvd_tissue_map(const pvd_tissue_params *p, const float *ct, int n0, int n1, int n2, float *corrected,
                              unsigned char *class_bits, float *density, void *stream) {
    if (!p || !ct) return pvd_set_error(PVD_EINVAL, "null parameters or CT");
    if (n0 < 1 || n1 < 1 || n2 < 1) return pvd_set_error(PVD_EINVAL, "grid extents must be >= 1");
    if (p->n_classes < 0 || p->n_classes > PVD_TISSUE_MAX_CLASSES)
        return pvd_set_error(PVD_EINVAL, "n_classes must be 0..%d", PVD_TISSUE_MAX_CLASSES);
    if (p->n_materials < 1 || p->n_materials > PVD_TISSUE_MAX_MATERIALS)
        return pvd_set_error(PVD_EINVAL, "n_materials must be 1..%d", PVD_TISSUE_MAX_MATERIALS);
    for (int i = 1; i < p->n_materials; ++i)
        if (!(p->mat_lo[i] > p->mat_lo[i - 1])) return pvd_set_error(PVD_EINVAL, "mat_lo must be ascending");
    TissueArgs a{};
    a.ct = ct;
    a.corrected = corrected;
    a.bits = class_bits;
    a.density = density;
    a.n0 = n0;
    a.n1 = n1;
    a.n2 = n2;
    a.handle = p->handle_artifacts ? 1 : 0;
    a.metal = a.handle ? p->metal_hu : INFINITY;
    a.ncls = p->n_classes;
    a.nmat = p->n_materials;
    for (int c = 0; c < PVD_TISSUE_MAX_CLASSES; ++c) {          // unused classes never match
        a.clo[c] = c < a.ncls ? p->class_lo[c] : INFINITY;
        a.chi[c] = c < a.ncls ? p->class_hi[c] : -INFINITY;
    }
    for (int i = 0; i < PVD_TISSUE_MAX_MATERIALS; ++i) {        // unused materials are never reached
        a.mlo[i] = i < a.nmat ? p->mat_lo[i] : INFINITY;
        a.mden[i] = p->mat_density[i < a.nmat ? i : a.nmat - 1];   // +inf HU keeps the last material
    }
    if (a.handle) {
        if (!(p->sigma > 0.0) || !(p->truncate >= 0.0))
            return pvd_set_error(PVD_EINVAL, "sigma must be > 0 and truncate >= 0");
        const int r = (int)(p->truncate * p->sigma + 0.5);   // scipy: int(truncate * sd + 0.5)
        if (r > PVD_TISSUE_MAX_RADIUS)
            return pvd_set_error(PVD_ENOTSUP, "Gaussian radius %d exceeds %d", r, PVD_TISSUE_MAX_RADIUS);
        a.radius = r;
        double sum = 0.0;
        for (int k = -r; k <= r; ++k) sum += (a.w[k + r] = std::exp(-0.5 / (p->sigma * p->sigma) * k * k));
        for (int k = 0; k <= 2 * r; ++k) a.w[k] /= sum;
    }
    const long long n = (long long)n0 * n1 * n2;
    const bool nt = n * ((corrected ? 4 : 0) + (density ? 4 : 0) + (class_bits ? 1 : 0)) > PVD_STREAM_BYTES;
    hipStream_t st = (hipStream_t)stream;
    const bool r4 = a.radius == 4 || !a.handle;   // sigma 1, truncate 4: the reference's filter
    // (other radii fill in place, four voxels of one z-row at a time)
    const bool vec = (r4 ? n >= 4 : n2 % 4 == 0) && aligned(ct, 16) && (!corrected || aligned(corrected, 16)) &&
                     (!density || aligned(density, 16)) && (!class_bits || aligned(class_bits, 4));
    const bool few = a.nmat <= 16;
    if (r4) {
        const long long items = vec ? (n + 3) / 4 : n, chunks = (items + kTissueChunk - 1) / kTissueChunk;
        const long long g = std::min<long long>(
            {chunks, kTissueGrid, std::max<long long>(kTissueFew, (chunks + kTissuePer - 1) / kTissuePer)});
        const auto kernel = vec ? nt ? few ? tissue_map<true, 16, true> : tissue_map<true, 32, true>
                                     : few ? tissue_map<true, 16> : tissue_map<true, 32>
                                : few ? tissue_map<false, 16> : tissue_map<false, 32>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)g), dim3(kTissueBlock), 0, st, a, items, n);
    } else {
        const long long items = vec ? n / 4 : n;
        const long long g = std::min<long long>((items + kRowBlock - 1) / kRowBlock, kRowGrid);
        const auto kernel = vec ? few ? tissue_map_rows<true, 16> : tissue_map_rows<true, 32>
                                : few ? tissue_map_rows<false, 16> : tissue_map_rows<false, 32>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)g), dim3(kRowBlock), 0, st, a, items);
    }
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return pvd_hip_error(e, "launch tissue map");
    return PVD_OK;
}
