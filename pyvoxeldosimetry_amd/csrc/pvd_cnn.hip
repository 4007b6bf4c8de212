// 3-D residual CNN kernels on the gfx950 matrix cores (BF16 in, FP32 accumulate).
//
// Layout: activations channels-last BF16 [n0][n1][n2][C] (n2 % 32 == 0), weights
// BF16 [27][32 cout][cin] with tap = (dx+1)*9 + (dy+1)*3 + (dz+1).
//
// conv_march residual layers on whole volumes (see there); conv_fwd the other layers and
//           region lists:
// conv_fwd  implicit GEMM per output row of 32 voxels along z:
//           D[32 voxels][32 cout] += A[32 voxels][16 cin] * B[16 cin][32 cout]
//           with v_mfma_f32_32x32x16_bf16, K-loop over 27 taps x cin/16.
//           Persistent workgroups (8 waves) keep all weights in LDS and stage a
//           halo of 2x4 output rows; voxel/cout strides are padded by 16 bytes so
//           the 16-byte fragment reads of 8 consecutive lanes hit distinct banks.
// wgrad     D[32 cout][32 cin] per tap += A[32 cout][16 voxels] * B[16 voxels][32 cin]
//           from channels-last LDS tiles by transposing LDS reads.  Each wave owns a
//           fixed subset of taps; per-workgroup partial sums are reduced in a fixed
//           order (deterministic).
#include <algorithm>

#include "pvd_internal.h"

#include "../../include/pvd_learned.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

// row of accumulator i held by `lane` in the 32x32 MFMA output; its column is lane % 32
__device__ __forceinline__ int mfma_row(int i, int lane) { return ((i >> 2) << 3) + ((lane >> 5) << 2) + (i & 3); }

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// round to nearest even; NaN stays NaN
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ bf16x8 lds_frag(const char *p) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return __builtin_bit_cast(bf16x8, v);
}

struct ConvArgs {
    const uint16_t *x;
    const uint16_t *w;
    const float *bias;
    const uint16_t *resid;
    uint16_t *y;
    uint16_t *act;
    float *y32;
    int n0, n1, n2;
    const int *list;          // blocks to compute (NULL: every block)
    const int *list_n;        // number of entries of list (device)
    uint32_t *mask;           // ReLU mask, one word per voxel (bit = channel), or NULL
};

constexpr int FWD_BX = 2, FWD_BY = 4, FWD_THREADS = 512;
constexpr int HX = FWD_BX + 2, HY = FWD_BY + 2, HZ = 34;

// per-wave staging of one 32 x 32 BF16 output tile (32 voxels x 32 channels)
constexpr int FWD_STAGE = 32 * 32 * 2;

template <int CIN>
constexpr size_t fwd_lds_bytes() {
    return (size_t)27 * 32 * (CIN * 2 + 16) + (size_t)HX * HY * HZ * (CIN * 2 + 16) +
           (size_t)(FWD_THREADS / 64) * FWD_STAGE;
}

// MASK (a residual layer in training): a.mask instead of a.act.
template <int CIN, int EPI, bool MASK = false>
__global__ __launch_bounds__(FWD_THREADS) void cnn_conv_fwd(ConvArgs a) {
    extern __shared__ uint4 lds_u4[];
    char *lds = reinterpret_cast<char *>(lds_u4);
    constexpr int VS = CIN * 2 + 16;   // bytes per halo voxel
    constexpr int WS = CIN * 2 + 16;   // bytes per (tap, cout) weight row
    constexpr int C8 = CIN / 8;        // 16-byte chunks per voxel
    char *wl = lds;
    char *hl = lds + 27 * 32 * WS;
    const int tid = threadIdx.x;
    char *stg = hl + HX * HY * HZ * VS + (tid >> 6) * FWD_STAGE;   // this wave's output staging
    for (int i = tid; i < 27 * 32 * C8; i += FWD_THREADS) {
        const int row = i / C8, c8 = i - row * C8;
        *reinterpret_cast<uint4 *>(wl + row * WS + c8 * 16) = reinterpret_cast<const uint4 *>(a.w)[i];
    }
    const int nbx = (a.n0 + FWD_BX - 1) / FWD_BX, nby = (a.n1 + FWD_BY - 1) / FWD_BY, nbz = a.n2 >> 5;
    // blocks to compute: the list's entries (a region of the volume) or all of them
    const int total = a.list ? *a.list_n : nbx * nby * nbz;
    auto block_of = [&](int i) { return a.list ? a.list[i] : i; };
    const int wave = tid >> 6, lane = tid & 63;
    const int wx = wave / FWD_BY, wy = wave % FWD_BY;
    const int m = lane & 31, kh = lane >> 5;
    // this lane's output-channel bias, loaded once: a global load in the epilogue
    // would wait (in-order counter) for the next block's halo prefetch
    const float bco = a.bias ? a.bias[m] : 0.0f;
    // The halo of the next block is fetched into registers while this block's
    // MFMA loop runs (all loads in flight at once), then written to LDS.
    constexpr int HALO = HX * HY * HZ * C8;
    constexpr int PER_T = (HALO + FWD_THREADS - 1) / FWD_THREADS;
    uint4 pf[PER_T];
    auto fetch = [&](int b) {
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * FWD_BX, y0 = by * FWD_BY, z0 = bz * 32;
#pragma unroll
        for (int u = 0; u < PER_T; ++u) {
            const int i = tid + u * FWD_THREADS;
            const int c8 = i % C8, vox = i / C8;
            const int hz = vox % HZ, hy = (vox / HZ) % HY, hx = vox / (HZ * HY);
            const int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
            pf[u] = make_uint4(0u, 0u, 0u, 0u);
            if (i < HALO && gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2)
                pf[u] = reinterpret_cast<const uint4 *>(a.x + (((long long)gx * a.n1 + gy) * a.n2 + gz) * CIN)[c8];
        }
    };
    auto put_halo = [&]() {
#pragma unroll
        for (int u = 0; u < PER_T; ++u) {
            const int i = tid + u * FWD_THREADS;
            if (i < HALO) *reinterpret_cast<uint4 *>(hl + (i / C8) * VS + (i % C8) * 16) = pf[u];
        }
    };
    // Per block: MFMA loop, the skip values out of the halo, barrier, the next block's
    // halo into LDS, then the epilogue, whose output stores overlap the next block's
    // MFMAs.  (The wait for the prefetched halo registers counts every earlier vector
    // memory operation; the latest stores are then a block old.)
    if ((int)blockIdx.x < total) {
        fetch(block_of(blockIdx.x));
        put_halo();
    }
    for (int bi = blockIdx.x; bi < total; bi += gridDim.x) {
        const int b = block_of(bi);
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * FWD_BX, y0 = by * FWD_BY, z0 = bz * 32;
        // LDS-only barriers: the previous block's output stores stay in flight (a
        // full __syncthreads would wait for them)
        lds_barrier();     // weights and this block's halo visible
        const int ox = x0 + wx, oy = y0 + wy;
        const bool live = ox < a.n0 && oy < a.n1;    // wave-uniform
        const long long vrow = ((long long)ox * a.n1 + oy) * a.n2 + z0;
        // skip term of a residual layer: a layer whose skip input is its own input
        // (resid == x, 32 channels) reads it from the centre of the halo in LDS;
        // any other tensor is loaded here, before the next halo, so the epilogue
        // waits for these loads only
        const bool resid_lds = EPI == PVD_CNN_EPI_RESID_RELU && CIN == 32 && a.resid == a.x;
        uint16_t rs[16];
        if (EPI == PVD_CNN_EPI_RESID_RELU && !resid_lds && live) {
#pragma unroll
            for (int i = 0; i < 16; ++i) rs[i] = a.resid[(vrow + mfma_row(i, lane)) * 32 + m];
        }
        if (bi + (int)gridDim.x < total) fetch(block_of(bi + gridDim.x));
        // one accumulation chain in tap order; the fragments of tap t + 1 are read
        // before the MFMAs of tap t (two register sets), so each LDS round trip
        // overlaps the previous tap's MFMAs
        f32x16 acc = {};
        if (live) {
            constexpr int KC = CIN / 16;
            bf16x8 fa[2][KC], fb[2][KC];
            auto read_tap = [&](int tap, bf16x8 *ta, bf16x8 *tb) {
                const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
                const char *hrow = hl + (((wx + dx + 1) * HY + (wy + dy + 1)) * HZ + (m + dz + 1)) * VS + kh * 16;
                const char *wrow = wl + (tap * 32 + m) * WS + kh * 16;
#pragma unroll
                for (int cc = 0; cc < KC; ++cc) {
                    ta[cc] = lds_frag(hrow + cc * 32);
                    tb[cc] = lds_frag(wrow + cc * 32);
                }
            };
            read_tap(0, fa[0], fb[0]);
#pragma unroll
            for (int tap = 0; tap < 27; ++tap) {
                const int cur = tap & 1;
                if (tap + 1 < 27) read_tap(tap + 1, fa[cur ^ 1], fb[cur ^ 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int cc = 0; cc < KC; ++cc)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[cur][cc], fb[cur][cc], acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (resid_lds) {   // halo voxel (wx + 1, wy + 1, z + 1), channel m
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    rs[i] = *reinterpret_cast<const uint16_t *>(
                        hl + (((wx + 1) * HY + (wy + 1)) * HZ + mfma_row(i, lane) + 1) * VS + m * 2);
            }
        }
        lds_barrier();     // every wave finished with this block's halo
        // unconditional, so that no path leaves the prefetch loads outstanding (they
        // would be waited for, with the epilogue's stores, at the next fetch); after
        // the last block it rewrites values that nothing reads
        put_halo();
        if (!live) continue;
        const int co = m;
        if (EPI == PVD_CNN_EPI_RELU || EPI == PVD_CNN_EPI_RESID_RELU) {
            // The wave's output tile (voxels z0..z0+31 of one column, 32 channels) is
            // 2 KB contiguous in y: stage it in the wave's LDS slot as [row][channel],
            // then write it as two 16-byte stores per lane (in place of 16 two-byte
            // stores).  One wave reads only what it wrote, in program order.
            uint16_t *sy = reinterpret_cast<uint16_t *>(stg);
            const uint4 *src = reinterpret_cast<const uint4 *>(stg);
            if constexpr (MASK) {
                // a voxel's 32 channels are a half wave: one ballot has the words of two voxels
                uint32_t word = 0;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const unsigned long long on = __ballot(f2bf(fmaxf(acc[i] + bco, 0.0f)) != 0);
                    if (m == i) word = (uint32_t)(kh ? on >> 32 : on);
                }
                if (m < 16) a.mask[vrow + mfma_row(m, lane)] = word;
            } else if (a.act) {                  // the activations first
#pragma unroll
                for (int i = 0; i < 16; ++i) sy[mfma_row(i, lane) * 32 + co] = f2bf(fmaxf(acc[i] + bco, 0.0f));
                uint4 *dst = reinterpret_cast<uint4 *>(a.act + vrow * 32);
                dst[lane] = src[lane];
                dst[lane + 64] = src[lane + 64];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float av = fmaxf(acc[i] + bco, 0.0f);
                uint16_t h;
                if (EPI == PVD_CNN_EPI_RELU) {
                    h = f2bf(av);
                } else {
                    h = f2bf(bf2f(rs[i]) + av);
                }
                sy[mfma_row(i, lane) * 32 + co] = h;
            }
            uint4 *dst = reinterpret_cast<uint4 *>(a.y + vrow * 32);
            dst[lane] = src[lane];
            dst[lane + 64] = src[lane + 64];
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const long long v = vrow + mfma_row(i, lane);
                if (EPI == PVD_CNN_EPI_LINEAR_F32) {
                    if (co == 0) a.y32[v] = acc[i] + bco;
                } else {
                    a.y32[v * 32 + co] += acc[i];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// Residual layer (32 -> 32, y = x + relu(conv(x) + b)) on whole volumes.  A workgroup owns
// a column of 8 y-rows x 32 z-voxels and marches along x, one plane of outputs per step (a
// row per wave), over a ring of four input planes in LDS: planes p - 1, p, p + 1 are read
// while p + 2 arrives, so a step costs one barrier and the waves may drift by a step (one
// wave's epilogue beside another's MFMAs), and each input plane is read once per column
// (1.33 times over the volume, against 3.2 for 2 x 4-row blocks).  The weights of MR_REG
// of the 27 taps stay in registers (two waves per SIMD leave room for them), the others in
// LDS: MFMAs take fewer LDS reads than the two fragments each would need.
// Operands are swapped against the kernel above: the weights are A and the voxels B, so a
// lane holds one voxel's channels in groups of four and the epilogue moves 8 bytes at a
// time; the accumulation order is the same (same bits).
// LDS: 16-byte chunk c of weight row R sits in slot c ^ (R >> 2) & 3 of its 64 bytes, of
// halo voxel (row, hz) in slot c ^ (hz >> 2) & 3: 8 consecutive lanes hit distinct banks
// without padding, and a fragment address is a lane constant plus an immediate.
// 128^3 layer 176 -> 115-125 us, 256x256x224 1090 -> 790 us (812 GFLOP at 1.03 PFLOP/s; the
// one-row kernel above waits at its two barriers a block and for its LDS reads).  Measured
// at 256x256x224: no tap in registers 842, 9 taps 809, 21 taps 816, 18 taps 790 (reading
// one or three taps ahead the same); 4 x 4-row blocks, two rows per wave sharing fragments,
// all weights in LDS 863.
constexpr int MR_Y = 8, MR_HY = MR_Y + 2;                            // rows of a column, with halo
constexpr int MR_PITCH = HZ * 64, MR_PLANE = MR_HY * MR_PITCH;       // bytes of a halo row, a plane
constexpr int MR_WBYTES = 27 * 32 * 64;
constexpr size_t MR_LDS = (size_t)MR_WBYTES + 4 * MR_PLANE + 8 * FWD_STAGE + 128;
// The same march runs the input gradient (MR_GRAD*: x is dz, the weights are flipped):
//   dh' = dh + conv(dz),  dz' = bf16(dh' where the ReLU mask is set),  sum of dz' before
// rounding per channel, so the ReLU gradient of the layer below costs no pass of its own
// over dh (128^3: accumulating convolution 360 us + ReLU gradient 165 us before, 128 us
// now, 106 without a dh input).  Its epilogue needs registers for the dh tile: fewer taps'
// weights stay there.  The forward writes the ReLU masks (4 bytes a voxel) in place of the
// activations (64 bytes).
enum { MR_FWD = 0, MR_MASK, MR_GRAD_FIRST, MR_GRAD, MR_GRAD_LAST };   // MASK: forward and mask;
                                                                     // FIRST: dh = 0; LAST: dh' not stored
constexpr int MR_DEPTH = 2;                                              // taps read ahead
constexpr int mr_regs(int mode) { return mode == MR_FWD ? 18 : mode == MR_MASK ? 15 : 12; }   // taps in registers
constexpr bool mr_in_reg(int t, int nr) { return t * nr / 27 != (t + 1) * nr / 27; }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ u32x4 g_zero_row[64];        // what a halo row outside the volume reads

// two floats to BF16, round to nearest even, in one word
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}

struct MarchArgs {
    ConvArgs c;
    int nby, nbz, seg;        // columns along y and z, planes per segment
    int nseg;
    const float *dh_in;       // gradient modes: c.x = dz, c.y = dz', c.mask = the mask
    float *dh_out;
    float *part;              // [column][32] sums of dz'
};

template <int MODE>
__global__ __launch_bounds__(FWD_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void cnn_conv_march(MarchArgs q) {
    constexpr int NR = mr_regs(MODE);
    constexpr bool FWD = MODE == MR_FWD || MODE == MR_MASK;
    constexpr bool IN = MODE == MR_GRAD || MODE == MR_GRAD_LAST, OUT = MODE == MR_GRAD_FIRST || MODE == MR_GRAD;
    extern __shared__ uint4 lds_u4[];
    const ConvArgs &a = q.c;
    char *lds = reinterpret_cast<char *>(lds_u4);
    char *wl = lds, *ring = lds + MR_WBYTES;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char *stg = ring + 4 * MR_PLANE + wave * FWD_STAGE;
    float *bl = reinterpret_cast<float *>(ring + 4 * MR_PLANE + 8 * FWD_STAGE);
    for (int i = tid; i < 27 * 32 * 4; i += FWD_THREADS) {
        const int row = i >> 2, c = i & 3;
        reinterpret_cast<uint4 *>(wl)[row * 4 + (c ^ ((row >> 2) & 3))] = reinterpret_cast<const uint4 *>(a.w)[i];
    }
    if (tid < 32) bl[tid] = a.bias ? a.bias[tid] : 0.0f;
    const int m = lane & 31, kh = lane >> 5;
    // Columns: XCD x (workgroups x, x + 8, ...) takes the x-th eighth of them in (segment,
    // y, z) order, so neighbouring columns share their halo rows in one L2.
    const int cols = q.nby * q.nbz * q.nseg, per = gridDim.x / 8;
    const int col = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (col >= cols) return;
    const int bz = col % q.nbz, by = col / q.nbz % q.nby, x0 = col / (q.nbz * q.nby) * q.seg;
    const int x1 = min(x0 + q.seg, a.n0), y0 = by * MR_Y, z0 = bz * 32;
    // A plane's halo: 20 units of 16 voxels (half rows, wave-uniform), waves 0..7 units w and
    // w + 8, waves 0..3 also 16 + w; then 80 lanes of waves 4 and 5 the rows' end voxels.
    u32x4 pf[3];
    const long long plane = (long long)a.n1 * a.n2 * 4;           // 16-byte chunks
    const u32x4 *xb = reinterpret_cast<const u32x4 *>(a.x);
    auto unit_off = [&](int u, bool &in) -> long long {
        const int gy = y0 - 1 + (u >> 1);
        in = gy >= 0 && gy < a.n1;
        return ((long long)gy * a.n2 + z0 + (u & 1) * 16) * 4;
    };
    auto fetch = [&](int p) {
        const bool px = p >= 0 && p < a.n0;
        const u32x4 *xp = xb + p * plane;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            bool in;
            const long long o = unit_off(wave + 8 * j, in);
            const u32x4 *s = px && in ? xp + o : g_zero_row;
            pf[j] = s[lane];
        }
        if (wave < 4) {
            bool in;
            const long long o = unit_off(wave + 16, in);
            const u32x4 *s = px && in ? xp + o : g_zero_row;
            pf[2] = s[lane];
        } else {
            const int e = tid - 256, gy = y0 - 1 + (e >> 3), gz = z0 + (e & 4 ? 32 : -1);
            const bool in = px && e < MR_HY * 8 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
            const u32x4 *s = in ? xp + ((long long)gy * a.n2 + gz) * 4 + (e & 3) : g_zero_row;
            pf[2] = *s;
        }
    };
    const int hzp = 1 + (wave & 1) * 16 + (lane >> 2);
    const int put0 = (wave >> 1) * MR_PITCH + hzp * 64 + (((lane & 3) ^ ((hzp >> 2) & 3)) << 4);
    int put2;
    if (wave < 4) {
        put2 = put0 + 8 * MR_PITCH;
    } else {
        const int e = tid - 256, he = e & 4 ? 33 : 0;
        put2 = (e >> 3) * MR_PITCH + he * 64 + (((e & 3) ^ ((he >> 2) & 3)) << 4);
    }
    auto put = [&](int slot) {
        char *d = ring + slot * MR_PLANE;
        *reinterpret_cast<u32x4 *>(d + put0) = pf[0];
        *reinterpret_cast<u32x4 *>(d + put0 + 4 * MR_PITCH) = pf[1];
        if (wave < 4 || tid < 256 + MR_HY * 8) *reinterpret_cast<u32x4 *>(d + put2) = pf[2];
    };
    for (int p = x0 - 1; p <= x0 + 1; ++p) {
        fetch(p);
        put(p & 3);
    }
    lds_barrier();
    // lane constants of the fragment addresses, and the register-resident weights
    int wa[2], xa[3][2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        wa[c] = m * 64 + (((c * 2 + kh) ^ ((m >> 2) & 3)) << 4);
#pragma unroll
        for (int dz = 0; dz < 3; ++dz) {
            const int hz = m + dz;
            xa[dz][c] = wave * MR_PITCH + hz * 64 + (((c * 2 + kh) ^ ((hz >> 2) & 3)) << 4);
        }
    }
    bf16x8 WR[NR][2];
#pragma unroll
    for (int t = 0; t < 27; ++t)
        if (mr_in_reg(t, NR)) {
            WR[t * NR / 27][0] = lds_frag(wl + wa[0] + t * 2048);
            WR[t * NR / 27][1] = lds_frag(wl + wa[1] + t * 2048);
        }
    const int oy = y0 + wave;
    const bool live = oy < a.n1;         // wave-uniform
    const long long row0 = (long long)min(oy, a.n1 - 1) * a.n2 + z0, pvox = (long long)a.n1 * a.n2;
    u32x4 *yb = reinterpret_cast<u32x4 *>(a.y) + row0 * 4;
    float bs[FWD ? 1 : 16] = {};
    for (int p = x0; p < x1; ++p) {
        // plane p + 1 written by every wave; slot (p + 2) & 3 (plane p - 2) read by every wave
        if (p > x0) lds_barrier();
        if (p + 1 < x1) fetch(p + 2);
        f32x16 acc = {};
        uint2 rs[4];
        f32x4 dh[4];                       // this lane's voxel: channels 8 g + 4 kh ..
        const long long vox = p * pvox + row0 + m;
        uint32_t mk = 0;
        if constexpr (!FWD) {
            mk = a.mask[vox];
#pragma unroll
            for (int g = 0; g < 4; ++g)
                dh[g] = IN ? reinterpret_cast<const f32x4 *>(q.dh_in)[vox * 8 + 2 * g + kh] : f32x4{};
        }
        {
            constexpr int NS = MR_DEPTH + 1;
            bf16x8 X[NS][2], W[NS][2];
            const char *pl[3] = {ring + ((p - 1) & 3) * MR_PLANE, ring + (p & 3) * MR_PLANE, ring + ((p + 1) & 3) * MR_PLANE};
            auto read = [&](int t) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    X[t % NS][c] = lds_frag(pl[t / 9] + xa[t % 3][c] + t / 3 % 3 * MR_PITCH);
                    if (!mr_in_reg(t, NR)) W[t % NS][c] = lds_frag(wl + wa[c] + t * 2048);
                }
            };
#pragma unroll
            for (int t = 0; t < MR_DEPTH; ++t) read(t);
#pragma unroll
            for (int t = 0; t < 27; ++t) {
                if (t + MR_DEPTH < 27) read(t + MR_DEPTH);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mr_in_reg(t, NR) ? WR[t * NR / 27][c] : W[t % NS][c],
                                                                  X[t % NS][c], acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (FWD) {
                // skip values: the centre voxel, 4 channels at a time
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int hz = m + 1;
                    rs[g] = *reinterpret_cast<const uint2 *>(pl[1] + (wave + 1) * MR_PITCH + hz * 64 +
                                                             ((g ^ ((hz >> 2) & 3)) << 4) + kh * 8);
                }
            }
        }
        put((p + 2) & 3);      // (after the last plane it rewrites values that nothing reads)
        // the row's 32 voxels x 32 channels through the wave's staging, stored as 2 KB
        uint32_t bits = 0;
        if (!FWD) mk = live ? mk >> (4 * kh) : 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float v[4];
            if constexpr (FWD) {
                const float4 bb = *reinterpret_cast<const float4 *>(bl + 8 * g + 4 * kh);
                const float b4[4] = {bb.x, bb.y, bb.z, bb.w};
                const uint32_t r2[2] = {rs[g].x, rs[g].y};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float av = fmaxf(acc[4 * g + j] + b4[j], 0.0f);
                    v[j] = bf2f((uint16_t)(r2[j >> 1] >> (16 * (j & 1)))) + av;
                    if (MODE == MR_MASK) bits |= av > 0x1p-134f ? 1u << (8 * g + j) : 0u;      // BF16 of av is not 0
                }
            } else {
                f32x4 d = dh[g];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    d[j] += acc[4 * g + j];
                    v[j] = (mk >> (8 * g + j)) & 1u ? d[j] : 0.0f;
                    bs[4 * g + j] += v[j];
                }
                if (OUT && live) reinterpret_cast<f32x4 *>(q.dh_out)[vox * 8 + 2 * g + kh] = d;
            }
            *reinterpret_cast<uint2 *>(stg + m * 64 + ((g ^ ((m >> 2) & 3)) << 4) + kh * 8) =
                make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        }
        if constexpr (MODE == MR_MASK) {
            bits <<= 4 * kh;
            bits |= __shfl_xor(bits, 32);
            if (live && kh == 0) a.mask[vox] = bits;
        }
        if (live) {
            u32x4 *dst = yb + p * plane;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int v = h * 16 + (lane >> 2);
                dst[h * 64 + lane] = *reinterpret_cast<const u32x4 *>(stg + v * 64 + (((lane & 3) ^ ((v >> 2) & 3)) << 4));
            }
        }
    }
    if constexpr (!FWD) {
        // channel sums: over the 32 voxels of a lane half, then over the waves in order
        float *red = reinterpret_cast<float *>(ring + 4 * MR_PLANE);
        lds_barrier();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v = bs[i];
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o);
            if (m == 0) red[wave * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)] = v;
        }
        lds_barrier();
        if (tid < 32) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; ++w) v += red[w * 32 + tid];
            q.part[(size_t)col * 32 + tid] = v;
        }
    }
}

// ---------------------------------------------------------------------------------
// Input layer with four live channels (the packer's activity, density and plain dose,
// and a zero) in a 16-channel BF16 input whose channels 4..15 are zero, ReLU epilogue.
// K of each MFMA packs 4 taps x 4 channels: 7 MFMAs per 32-voxel row (taps 24..27, the
// last zero) in place of 27 with 13 of 16 channels zero.  The packed weights
// wp[c][co][k] = w[4c + k/4][co][k%4] are built in LDS from the [27][32][16] layout;
// the halo holds the four channels (8 bytes a voxel).  Blocks, region lists, the
// next-halo prefetch and the epilogue are cnn_conv_fwd's.
constexpr int IN_CHUNKS = 7;
constexpr int IN_WS = 16 * 2 + 16;                              // bytes per (chunk, cout) row
template <int BX, int BY>
constexpr int in_halo() { return (BX + 2) * (BY + 2) * HZ; }
template <int BX, int BY>
constexpr size_t in_lds_bytes() {
    return (size_t)IN_CHUNKS * 32 * IN_WS + (size_t)in_halo<BX, BY>() * 8 + (size_t)(FWD_THREADS / 64) * FWD_STAGE;
}

// the network's inputs as FP32 maps (rows of n2 voxels `pitch` floats apart) and the device
// maxima that scale the activity and the plain dose
struct InMaps {
    const float *map[3];               // activity, density, plain dose
    const float *amax, *dmax;
    long long pitch;
};

__device__ __forceinline__ float inv_scale(const float *m) { return 1.0f / fmaxf(*m, 1e-30f); }

// the packer's four channels of one voxel
__device__ __forceinline__ uint2 pack_input(float act, float dens, float dose, float sa, float sd) {
    return make_uint2((uint32_t)f2bf(act * sa) | (uint32_t)f2bf(dens) << 16, (uint32_t)f2bf(dose * sd));
}

// BX x BY rows per block (2 x 4: the blocks of region lists; 4 x 4 for whole volumes,
// less halo per output); each of the 8 waves computes BX * BY / 8 rows.  MAPS: the halo
// comes from the FP32 maps and is packed on its way into LDS (the same bits): 12 bytes a
// voxel instead of a pack pass (12 in, 32 out) and 32 bytes of which 8 are live.  128^3:
// pack 14.5 + 40.5 us -> 45.0, 512x256x224: 288 + 546 -> 556.  What is left is each block's
// two barriers and its epilogue (134 MB of y at 3 TB/s); twice the workgroups per CU (128
// VGPRs) measured 45.0 and 669.
template <int BX, int BY, bool MAPS>
__global__ __launch_bounds__(FWD_THREADS) void cnn_conv_in(ConvArgs a, InMaps mp) {
    constexpr int IN_HALO = in_halo<BX, BY>(), HYL = BY + 2, NR = BX * BY / 8;
    static_assert(NR * 8 == BX * BY, "whole rows per wave");
    extern __shared__ uint4 lds_u4[];
    char *lds = reinterpret_cast<char *>(lds_u4);
    char *wl = lds;
    char *hl = lds + IN_CHUNKS * 32 * IN_WS;
    const int tid = threadIdx.x;
    char *stg = hl + IN_HALO * 8 + (tid >> 6) * FWD_STAGE;
    for (int i = tid; i < IN_CHUNKS * 32 * 16; i += FWD_THREADS) {
        const int c = i >> 9, co = (i >> 4) & 31, k = i & 15;
        const int tap = 4 * c + (k >> 2), ch = k & 3;
        const uint16_t v = tap < 27 ? a.w[((size_t)tap * 32 + co) * 16 + ch] : (uint16_t)0;
        *reinterpret_cast<uint16_t *>(wl + (c * 32 + co) * IN_WS + k * 2) = v;
    }
    const int nbx = (a.n0 + BX - 1) / BX, nby = (a.n1 + BY - 1) / BY, nbz = a.n2 >> 5;
    const int total = a.list ? *a.list_n : nbx * nby * nbz;
    auto block_of = [&](int i) { return a.list ? a.list[i] : i; };
    const int wave = tid >> 6, lane = tid & 63;
    const int m = lane & 31, kh = lane >> 5;
    float bias4[4][4];         // channels 8 g + 4 kh + j
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) bias4[g][j] = a.bias ? a.bias[8 * g + 4 * kh + j] : 0.0f;
    constexpr int PER_T = (IN_HALO + FWD_THREADS - 1) / FWD_THREADS;
    uint2 pf[MAPS ? 1 : PER_T];
    float pm[MAPS ? PER_T : 1][3];
    uint32_t inside = 0;                 // MAPS: bit u, voxel u of this thread lies in the volume
    const float sa = MAPS ? inv_scale(mp.amax) : 0.0f, sd = MAPS ? inv_scale(mp.dmax) : 0.0f;
    auto fetch = [&](int b) {
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * BX, y0 = by * BY, z0 = bz * 32;
        inside = 0;
#pragma unroll
        for (int u = 0; u < PER_T; ++u) {
            const int vox = tid + u * FWD_THREADS;
            const int hz = vox % HZ, hy = (vox / HZ) % HYL, hx = vox / (HZ * HYL);
            const int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
            const bool in = vox < IN_HALO && gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
            if constexpr (MAPS) {
                // (read at voxel 0 where outside and masked when packed)
                const long long o = in ? ((long long)gx * a.n1 + gy) * mp.pitch + gz : 0;
                inside |= (uint32_t)in << u;
#pragma unroll
                for (int c = 0; c < 3; ++c) pm[u][c] = mp.map[c][o];
            } else {
                pf[u] = make_uint2(0u, 0u);
                if (in) pf[u] = *reinterpret_cast<const uint2 *>(a.x + (((long long)gx * a.n1 + gy) * a.n2 + gz) * 16);
            }
        }
    };
    if ((int)blockIdx.x < total) fetch(block_of(blockIdx.x));
    for (int bi = blockIdx.x; bi < total; bi += gridDim.x) {
        const int b = block_of(bi);
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * BX, y0 = by * BY, z0 = bz * 32;
        lds_barrier();     // weights visible / previous block finished with the halo
#pragma unroll
        for (int u = 0; u < PER_T; ++u) {
            const int vox = tid + u * FWD_THREADS;
            if (vox < IN_HALO) {
                if constexpr (MAPS) {
                    const uint2 v = pack_input(pm[u][0], pm[u][1], pm[u][2], sa, sd);
                    *reinterpret_cast<uint2 *>(hl + vox * 8) = (inside >> u) & 1u ? v : make_uint2(0u, 0u);
                } else {
                    *reinterpret_cast<uint2 *>(hl + vox * 8) = pf[u];
                }
            }
        }
        lds_barrier();
        if (bi + (int)gridDim.x < total) fetch(block_of(bi + gridDim.x));
#pragma unroll
        for (int r = 0; r < NR; ++r) {
        const int wx = (wave + 8 * r) / BY, wy = (wave + 8 * r) % BY;
        const int ox = x0 + wx, oy = y0 + wy;
        const bool live = ox < a.n0 && oy < a.n1;    // wave-uniform
        const long long vrow = ((long long)ox * a.n1 + oy) * a.n2 + z0;
        if (!live) continue;
        f32x16 acc0 = {}, acc1 = {};
#pragma unroll
        for (int c = 0; c < IN_CHUNKS; ++c) {
            uint2 h[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int tap = 4 * c + 2 * kh + j;
                const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
                h[j] = tap < 27 ? *reinterpret_cast<const uint2 *>(
                                      hl + (((wx + dx + 1) * HYL + (wy + dy + 1)) * HZ + (m + dz + 1)) * 8)
                                : make_uint2(0u, 0u);
            }
            const bf16x8 fa = __builtin_bit_cast(bf16x8, make_uint4(h[0].x, h[0].y, h[1].x, h[1].y));
            const bf16x8 fb = lds_frag(wl + (c * 32 + m) * IN_WS + kh * 16);
            // weights as A, voxels as B: a lane holds one voxel's channels in groups of four
            if ((c & 1) == 0) acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb, fa, acc0, 0, 0, 0);
            else acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb, fa, acc1, 0, 0, 0);
        }
        const f32x16 acc = acc0 + acc1;
        // the output tile (32 voxels x 32 channels) through the wave's LDS slot (16-byte
        // chunk g of voxel v in slot g ^ (v >> 2) & 3), stored as two 16-byte pieces per lane
        uint32_t bits = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = fmaxf(acc[4 * g + j] + bias4[g][j], 0.0f);
            const uint32_t lo = pack_bf16(v[0], v[1]), hi = pack_bf16(v[2], v[3]);
            bits |= ((lo & 0xffffu ? 1u : 0u) | (lo >> 16 ? 2u : 0u) | (hi & 0xffffu ? 4u : 0u) | (hi >> 16 ? 8u : 0u))
                    << (8 * g);
            *reinterpret_cast<uint2 *>(stg + m * 64 + ((g ^ ((m >> 2) & 3)) << 4) + kh * 8) = make_uint2(lo, hi);
        }
        if (a.mask) {
            bits <<= 4 * kh;
            bits |= __shfl_xor(bits, 32);
            if (kh == 0) a.mask[vrow + m] = bits;
        }
        uint4 *dst = reinterpret_cast<uint4 *>(a.y + vrow * 32);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int v = h * 16 + (lane >> 2);
            dst[h * 64 + lane] = *reinterpret_cast<const uint4 *>(stg + v * 64 + (((lane & 3) ^ ((v >> 2) & 3)) << 4));
        }
        }
    }
}

// ---------------------------------------------------------------------------------
// Output layer (32 channels in, channel 0 out, FP32, + bias[0]), by taps:
//   Y[u][t] = sum_ci W[t][0][ci] x[u][ci]   for every voxel u of the block's halo, t < 27
//   y[v]    = sum_t Y[v + tap(t)][t] + bias[0]
// The first is a GEMM of the halo (32 voxels per MFMA row block, 32 channels) with the
// 32 x 27 weight columns (taps padded to 32), so the matrix cores do 27 useful columns of
// 32 instead of 1 of the 32 output channels a full layer computes; the second is a
// 27-term sum per output voxel from LDS, in tap order.  Blocks and the region list are
// those of cnn_conv_fwd (2 x 4 rows of 32 voxels along z).
constexpr int OUT_YS = 28;                                     // floats per halo voxel of Y
template <int BX, int BY>
constexpr size_t out_lds_bytes() { return (size_t)(BX + 2) * (BY + 2) * HZ * OUT_YS * 4; }

// BX x BY rows per block: 2 x 4 (816 halo voxels, 26 row blocks of 32) for region lists;
// one thread per output voxel in the sums.
template <int BX, int BY>
__global__ __launch_bounds__(FWD_THREADS) void cnn_conv_out(ConvArgs a) {
    constexpr int HYL = BY + 2;
    constexpr int OUT_HALO = (BX + 2) * HYL * HZ;
    constexpr int OUT_GROUPS = (OUT_HALO + 31) / 32;
    static_assert(BX * BY * 32 <= FWD_THREADS, "one thread per output voxel");
    extern __shared__ uint4 lds_u4[];
    float *ys = reinterpret_cast<float *>(lds_u4);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int m = lane & 31, kh = lane >> 5;
    constexpr int NW = FWD_THREADS / 64;
    constexpr int GPW = (OUT_GROUPS + NW - 1) / NW;            // row blocks per wave (at most)
    // B: column n = tap (zero past 26), rows = input channels; both K halves of 16
    bf16x8 bw[2];
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (m < 27) v = *reinterpret_cast<const uint4 *>(a.w + ((size_t)m * 32 * 32 + cc * 16 + kh * 8));
        bw[cc] = __builtin_bit_cast(bf16x8, v);
    }
    const float b0 = a.bias ? a.bias[0] : 0.0f;
    const int nbx = (a.n0 + BX - 1) / BX, nby = (a.n1 + BY - 1) / BY, nbz = a.n2 >> 5;
    const int total = a.list ? *a.list_n : nbx * nby * nbz;
    for (int bi = blockIdx.x; bi < total; bi += gridDim.x) {
        const int b = a.list ? a.list[bi] : bi;
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * BX, y0 = by * BY, z0 = bz * 32;
        // A fragments of this wave's row blocks, all loads issued before the MFMAs
        uint4 av[GPW][2];
#pragma unroll
        for (int j = 0; j < GPW; ++j) {
            const int u = (wave + j * NW) * 32 + m;
            const int hz = u % HZ, hy = (u / HZ) % HYL, hx = u / (HZ * HYL);
            const int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
            const bool in = u < OUT_HALO && gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
            const uint4 *src = reinterpret_cast<const uint4 *>(
                a.x + (in ? (((long long)gx * a.n1 + gy) * a.n2 + gz) * 32 : 0));
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                const uint4 v = src[cc * 2 + kh];
                av[j][cc] = in ? v : make_uint4(0u, 0u, 0u, 0u);
            }
        }
        lds_barrier();      // the previous block's sums have read Y
#pragma unroll
        for (int j = 0; j < GPW; ++j) {
            const int g = wave + j * NW;
            if (g >= OUT_GROUPS) continue;           // wave-uniform
            f32x16 acc = {};
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[j][0]), bw[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[j][1]), bw[1], acc, 0, 0, 0);
            if (m < 27) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int u = g * 32 + mfma_row(i, lane);
                    if (u < OUT_HALO) ys[u * OUT_YS + m] = acc[i];
                }
            }
        }
        lds_barrier();
        if (tid < BX * BY * 32) {
            const int ox = tid / (BY * 32), oy = (tid >> 5) % BY, z = tid & 31;
            if (x0 + ox < a.n0 && y0 + oy < a.n1) {
                float sum = 0.0f;
                for (int t = 0; t < 27; ++t) {
                    const int dx = t / 9 - 1, dy = (t / 3) % 3 - 1, dz = t % 3 - 1;
                    sum += ys[(((ox + dx + 1) * HYL + (oy + dy + 1)) * HZ + (z + dz + 1)) * OUT_YS + t];
                }
                a.y32[((long long)(x0 + ox) * a.n1 + (y0 + oy)) * a.n2 + z0 + z] = sum + b0;
            }
        }
    }
}

// Whole volumes: the output layer marching along x.  A workgroup owns 8 y-rows x 32
// z-voxels of one segment of planes; each input plane's halo (10 x 34 voxels) goes through
// the tap GEMM once and its 27 values per voxel are added to the three output planes they
// reach, whose sums a thread carries (the taps of a voxel are added plane after plane, in
// tap order: the bits of the block form).  Y lies tap by tap (pitch 356 words: 16-byte
// stores of 4 voxels and reads along z meet every bank once), in two buffers, with one
// barrier a plane; the next two planes' loads are in flight during it.
// Bound by the reads of h: 1.33 (y, z halo) x 1.13 (segments of 16) of 134 MB at 128^3.
// 128^3 61 -> 31 us, 176x150x160 134 -> 61, 256x256x224 452 -> 219 (5.4 TB/s of h), against
// 4 x 4-row blocks with two barriers a block, Y voxel by voxel (4-way bank conflicts) and no
// load in flight over the sums; 64^3 and smaller the same.  A mask applied to a fetched
// plane at once, instead of before its MFMAs, waits for the load: 44 us.
constexpr int OM_Y = 8, OM_THREADS = 256, OM_HALO = (OM_Y + 2) * HZ, OM_GROUPS = (OM_HALO + 31) / 32, OM_PITCH = 356;
constexpr size_t OM_LDS = 2 * (size_t)27 * OM_PITCH * 4;
static_assert(OM_PITCH >= OM_GROUPS * 32 && OM_PITCH % 8 == 4, "a tap's row holds every group; odd in 16 bytes");

__global__ __launch_bounds__(OM_THREADS) void cnn_conv_out_march(ConvArgs a, int seg, int nby, int nbz) {
    extern __shared__ uint4 lds_u4[];
    float *lds = reinterpret_cast<float *>(lds_u4);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int m = lane & 31, kh = lane >> 5;
    constexpr int NW = OM_THREADS / 64, GPW = (OM_GROUPS + NW - 1) / NW;
    bf16x8 bw[2];
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (m < 27) v = *reinterpret_cast<const uint4 *>(a.w + ((size_t)m * 32 * 32 + cc * 16 + kh * 8));
        bw[cc] = __builtin_bit_cast(bf16x8, v);
    }
    const float b0 = a.bias ? a.bias[0] : 0.0f;
    const int bz = blockIdx.x % nbz, by = blockIdx.x / nbz % nby, sx = blockIdx.x / (nbz * nby);
    const int x0 = sx * seg, x1 = min(x0 + seg, a.n0), y0 = by * OM_Y, z0 = bz * 32;
    const long long plane = (long long)a.n1 * a.n2;
    // this lane's halo voxels: offset in a plane, or none
    long long off[GPW];
    bool in[GPW];
#pragma unroll
    for (int j = 0; j < GPW; ++j) {
        const int u = (wave + j * NW) * 32 + m;
        const int gy = y0 + u / HZ - 1, gz = z0 + u % HZ - 1;
        in[j] = u < OM_HALO && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
        off[j] = in[j] ? ((long long)gy * a.n2 + gz) * 32 + kh * 8 : kh * 8;
    }
    uint4 ring[2][GPW][2];                           // the two planes ahead
    auto fetch = [&](int gx, uint4 (*av)[2]) {
        const uint16_t *src = a.x + min(max(gx, 0), a.n0 - 1) * plane * 32;
#pragma unroll
        for (int j = 0; j < GPW; ++j)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) av[j][cc] = *reinterpret_cast<const uint4 *>(src + off[j] + cc * 16);
    };
    const int oy = tid >> 5, oz = tid & 31;
    float s0 = 0.0f, s1 = 0.0f;                      // sums of planes p - 1 and p before plane p
    auto step = [&](int p, uint4 (*av)[2], float *ys) {
        const bool ix = p >= 0 && p < a.n0;
#pragma unroll
        for (int j = 0; j < GPW; ++j) {
            const int g = wave + j * NW;
            if (g >= OM_GROUPS) continue;            // wave-uniform
            // (masked here, not when loaded: a use would wait for the load)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
                if (!(ix && in[j])) av[j][cc] = make_uint4(0u, 0u, 0u, 0u);
            f32x16 acc = {};
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[j][0]), bw[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[j][1]), bw[1], acc, 0, 0, 0);
            if (m < 27) {
#pragma unroll
                for (int i = 0; i < 16; i += 4)      // rows mfma_row(i ..): 4 consecutive voxels
                    *reinterpret_cast<float4 *>(ys + m * OM_PITCH + g * 32 + mfma_row(i, lane)) =
                        make_float4(acc[i], acc[i + 1], acc[i + 2], acc[i + 3]);
            }
        }
        if (p + 2 <= x1) fetch(p + 2, av);
        lds_barrier();       // Y of plane p; the other buffer's readers are past the previous one
        const float *yr = ys + oy * HZ + oz;
        float t0 = s0, t1 = s1, t2 = 0.0f;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int o = t / 3 * HZ + t % 3;
            t2 += yr[t * OM_PITCH + o];              // dx = -1: plane p + 1
            t1 += yr[(9 + t) * OM_PITCH + o];
            t0 += yr[(18 + t) * OM_PITCH + o];       // dx = +1: plane p - 1, now complete
        }
        if (p > x0 && y0 + oy < a.n1)
            a.y32[(p - 1) * plane + (long long)(y0 + oy) * a.n2 + z0 + oz] = t0 + b0;
        s0 = t1;
        s1 = t2;
    };
    fetch(x0 - 1, ring[0]);
    fetch(x0, ring[1]);
    for (int p = x0 - 1; p <= x1; p += 2) {
        step(p, ring[0], lds);
        if (p + 1 <= x1) step(p + 1, ring[1], lds + 27 * OM_PITCH);
    }
}

// ---------------------------------------------------------------------------------
struct WgradArgs {
    const uint16_t *x;
    const uint16_t *dz;
    float *work;
    int n0, n1, n2;
};

// Blocks of 2 x 4 rows of 32 voxels.  Both operands of D[co][ci] += dz^T x need 8
// consecutive voxels of one channel per lane while the tensors are channels-last, so the
// block's input halo and output gradient sit in LDS as they are in HBM and the fragments
// are read with the transposing LDS loads (ds_read_b64_tr_b16: 16 lanes read 4 voxels x
// 16 channels, lane j receives channel j of the 4 voxels).  The z taps share one read:
// a lane's window of 12 voxels serves dz = -1 (elements 0..7), 0 (1..8, by alignbit) and
// +1 (2..9).  Wave w owns the three taps of (dx, dy) = group w for all 8 rows, and row w
// of the ninth group (reduced over the waves at the end), so every wave issues 54 MFMAs
// per block: 2.5 KB of LDS reads per three MFMAs.  Two LDS buffers, one barrier per block;
// the next block's loads are in flight during the MFMAs.
// (Before: 2 x 2 blocks, 2-byte LDS stores into three dz-shifted channel-major copies, and
// 2 KB of fragment reads per MFMA: 355 us per 128^3 layer;
// now 120 us, 116 GFLOP at 0.97 PFLOP/s.)
constexpr int WG_BX = 2, WG_BY = 4, WG_THREADS = 512;
constexpr int WHX = WG_BX + 2, WHY = WG_BY + 2, WROWS = WG_BX * WG_BY;
constexpr int WG_HALO = WHX * WHY * HZ;                    // halo voxels
template <int CIN>
constexpr int wg_buf() { return WG_HALO * CIN * 2 + WROWS * 32 * 64; }   // one buffer: halo, gradient
constexpr int WG_RED = 8 * 3 * 1024 * 4;                   // the ninth group's partial sums
template <int CIN>
constexpr size_t wg_lds() { return 2 * wg_buf<CIN>() > WG_RED ? 2 * wg_buf<CIN>() : WG_RED; }
constexpr int WG_MAX_BLOCKS = 256;

typedef short s16x4 __attribute__((ext_vector_type(4)));
// 4 voxels of this lane's channel: `p` is the lane's own 8 bytes of the 16-lane group's
// 4 x 16 block (voxel (lane & 15) / 4, channels 4 (lane & 3) ..)
__device__ __forceinline__ uint2 lds_read_tr(const char *p) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) s16x4 *)(void *)const_cast<char *>(p)));
#else
    return uint2{};
#endif
}
__device__ __forceinline__ bf16x8 frag4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(bf16x8, make_uint4(a, b, c, d));
}
// bytes 2..5 of the pair (lo, hi): one 16-bit element further along
__device__ __forceinline__ uint32_t shift_elem(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_alignbit(hi, lo, 16); }

template <int CIN>
__global__ __launch_bounds__(WG_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void cnn_wgrad(WgradArgs a) {
    extern __shared__ uint4 lds_u4[];
    char *lds = reinterpret_cast<char *>(lds_u4);
    constexpr int VS = CIN * 2, C8 = CIN / 8, BUF = wg_buf<CIN>(), XB = WG_HALO * VS;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int m = lane & 31;
    const int nbx = (a.n0 + WG_BX - 1) / WG_BX, nby = (a.n1 + WG_BY - 1) / WG_BY, nbz = a.n2 >> 5;
    const int total = nbx * nby * nbz;
    // this lane's part of a transposing read: voxel within the 8 of its K half, channels
    const int tv = (lane >> 5) * 8 + ((lane & 15) >> 2), tc = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    const int xoff = tv * VS + (CIN == 32 ? tc : tc & 15) * 2, doff = tv * 64 + tc * 2;
    constexpr int NX = (WG_HALO * C8 + WG_THREADS - 1) / WG_THREADS, ND = WROWS * 32 * 4 / WG_THREADS;
    uint4 px[NX], pd[ND];
    auto fetch = [&](int b) {
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * WG_BX, y0 = by * WG_BY, z0 = bz * 32;
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            const int i = tid + u * WG_THREADS;
            const int c8 = i % C8, vox = i / C8;
            const int hz = vox % HZ, hy = (vox / HZ) % WHY, hx = vox / (HZ * WHY);
            const int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
            px[u] = make_uint4(0u, 0u, 0u, 0u);
            if (i < WG_HALO * C8 && gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2)
                px[u] = reinterpret_cast<const uint4 *>(a.x + (((long long)gx * a.n1 + gy) * a.n2 + gz) * CIN)[c8];
        }
#pragma unroll
        for (int u = 0; u < ND; ++u) {
            const int i = tid + u * WG_THREADS;
            const int c8 = i & 3, z = (i >> 2) & 31, r = i >> 7;
            const int ox = x0 + r / WG_BY, oy = y0 + r % WG_BY;
            pd[u] = make_uint4(0u, 0u, 0u, 0u);
            if (ox < a.n0 && oy < a.n1)
                pd[u] = reinterpret_cast<const uint4 *>(a.dz + (((long long)ox * a.n1 + oy) * a.n2 + z0 + z) * 32)[c8];
        }
    };
    auto put = [&](char *buf) {
#pragma unroll
        for (int u = 0; u < NX; ++u)
            if (tid + u * WG_THREADS < WG_HALO * C8) reinterpret_cast<uint4 *>(buf)[tid + u * WG_THREADS] = px[u];
#pragma unroll
        for (int u = 0; u < ND; ++u) reinterpret_cast<uint4 *>(buf + XB)[tid + u * WG_THREADS] = pd[u];
    };
    f32x16 acc[6];                   // taps of group `wave`, taps of the ninth group
#pragma unroll
    for (int j = 0; j < 6; ++j) acc[j] = f32x16{};
    const int grow = (wave / 3) * WHY + wave % 3;            // halo row of output row 0 for this group
    if ((int)blockIdx.x < total) {
        fetch(blockIdx.x);
        put(lds);
    }
    int cur = 0;
    for (int b = blockIdx.x; b < total; b += gridDim.x, cur ^= 1) {
        lds_barrier();     // this block's buffer written; the other one read by every wave
        const char *xs = lds + cur * BUF + xoff, *ds = lds + cur * BUF + XB + doff;
        if (b + (int)gridDim.x < total) fetch(b + gridDim.x);
        uint2 A[2][2][2], X[2][2][3];                        // [set][K chunk][4 voxels]
        auto read_d = [&](int r, uint2 (*d)[2]) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int q = 0; q < 2; ++q) d[c][q] = lds_read_tr(ds + (r * 32 + c * 16 + q * 4) * 64);
        };
        // (the last read of a row reaches two voxels past it: never used elements)
        auto read_x = [&](int hrow, uint2 (*x)[3]) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int q = 0; q < 3; ++q) x[c][q] = lds_read_tr(xs + (hrow * HZ + c * 16 + q * 4) * VS);
        };
        auto taps = [&](const uint2 (*d)[2], const uint2 (*x)[3], f32x16 *t) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16x8 f = frag4(d[c][0].x, d[c][0].y, d[c][1].x, d[c][1].y);
                const uint32_t w0 = x[c][0].x, w1 = x[c][0].y, w2 = x[c][1].x, w3 = x[c][1].y, w4 = x[c][2].x;
                t[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, frag4(w0, w1, w2, w3), t[0], 0, 0, 0);
                t[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, frag4(w1, w2, w3, w4), t[2], 0, 0, 0);
                t[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    f, frag4(shift_elem(w0, w1), shift_elem(w1, w2), shift_elem(w2, w3), shift_elem(w3, w4)), t[1], 0, 0, 0);
            }
        };
        read_d(0, A[0]);
        read_x(grow, X[0]);
#pragma unroll
        for (int r = 0; r < WROWS; ++r) {
            const int s = r & 1;
            if (r + 1 < WROWS) {
                read_d(r + 1, A[s ^ 1]);
                read_x(grow + (r + 1) / WG_BY * WHY + (r + 1) % WG_BY, X[s ^ 1]);
            } else {                                         // the ninth group's row
                read_d(wave, A[s ^ 1]);
                read_x((wave / WG_BY + 2) * WHY + wave % WG_BY + 2, X[s ^ 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
            taps(A[s], X[s], acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        taps(A[WROWS & 1], X[WROWS & 1], acc + 3);
        if (b + (int)gridDim.x < total) put(lds + (cur ^ 1) * BUF);
    }
    // partial dW of this workgroup: work[blockIdx][tap][co][ci], ci < CIN
    float *out = a.work + (size_t)blockIdx.x * 27 * 32 * CIN;
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (m < CIN) {
#pragma unroll
            for (int i = 0; i < 16; ++i) out[((size_t)(wave * 3 + j) * 32 + mfma_row(i, lane)) * CIN + m] = acc[j][i];
        }
    // the ninth group: sum over the waves, in wave order
    float *red = reinterpret_cast<float *>(lds_u4);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) red[(wave * 3 + j) * 1024 + mfma_row(i, lane) * 32 + m] = acc[3 + j][i];
    __syncthreads();
    for (int e = tid; e < 3 * 1024; e += WG_THREADS) {
        const int ci = e & 31;
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) sum += red[w * 3 * 1024 + e];
        if (ci < CIN) out[((size_t)24 * 32 + (e >> 5)) * CIN + ci] = sum;
    }
}

// ---------------------------------------------------------------------------------
// Gradients of the output layer.  Its dL/dr has one channel, kept as BF16 [n] rather than
// channel 0 of 32 (the kernels above would compute 31 channels of zeros on 134 MB of them).
//
// Weights: dw[t][ci] = sum_u x[u][ci] dr[u - d(t)], one GEMM of the 27 taps (32 rows)
// against the 32 channels instead of a GEMM per tap; x is read once, without a halo.  A
// tile is 8 rows of 32 voxels, a row per wave: x channels-last as in cnn_wgrad (transposing
// reads), the dr halo in three copies shifted by one voxel so that a tap's 8 voxels are one
// aligned read.  Bound by reading x: 128^3 123 us (cnn_wgrad on 32 channels of dr) -> 30
// (134 MB at 4.5 TB/s).
constexpr int OW_Y = 8, OW_ROW = 80, OW_HALO = 3 * (OW_Y + 2) * HZ;      // bytes of a dr row, halo voxels
constexpr int OW_XB = OW_Y * 32 * 64, OW_PL = (OW_Y + 2) * OW_ROW, OW_COPY = 3 * OW_PL, OW_BUF = OW_XB + 3 * OW_COPY;
constexpr int OW_RED = 8 * 27 * 32 * 4;
constexpr size_t OW_LDS = 2 * OW_BUF > OW_RED ? 2 * OW_BUF : OW_RED;
constexpr int OW_BLOCKS_PER_CU = 3;

__global__ __launch_bounds__(WG_THREADS) void cnn_out_wgrad(WgradArgs a) {
    extern __shared__ uint4 lds_u4[];
    char *lds = reinterpret_cast<char *>(lds_u4);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int m = lane & 31, kh = lane >> 5;
    const int nby = (a.n1 + OW_Y - 1) / OW_Y, nbz = a.n2 >> 5, total = a.n0 * nby * nbz;
    const int tv = (lane >> 5) * 8 + ((lane & 15) >> 2), tc = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    const int tap = min(m, 26), dx = tap / 9 - 1, dy = tap / 3 % 3 - 1, dz = tap % 3 - 1;
    const int aoff = OW_XB + (1 - dz) * OW_COPY + (1 - dx) * OW_PL + (wave + 1 - dy) * OW_ROW + kh * 16;
    const int boff = wave * 32 * 64 + tv * 64 + tc * 2;
    constexpr int NX = OW_Y * 32 * 4 / WG_THREADS, ND = (OW_HALO + WG_THREADS - 1) / WG_THREADS;
    uint4 px[NX];
    uint16_t pd[ND];
    uint32_t xin = 0, din = 0;             // which of them lie in the volume
    auto fetch = [&](int b) {
        const int z0 = b % nbz * 32, y0 = b / nbz % nby * OW_Y, x0 = b / (nbz * nby);
        xin = din = 0;
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            const int i = tid + u * WG_THREADS, oy = y0 + (i >> 7);
            xin |= (uint32_t)(oy < a.n1) << u;
            px[u] = reinterpret_cast<const uint4 *>(
                a.x + (((long long)x0 * a.n1 + min(oy, a.n1 - 1)) * a.n2 + z0 + ((i >> 2) & 31)) * 32)[i & 3];
        }
#pragma unroll
        for (int u = 0; u < ND; ++u) {
            const int e = tid + u * WG_THREADS, hz = e % HZ, row = e / HZ % (OW_Y + 2), pl = e / (HZ * (OW_Y + 2));
            const int gx = x0 + pl - 1, gy = y0 + row - 1, gz = z0 + hz - 1;
            const bool in = e < OW_HALO && gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
            din |= (uint32_t)in << u;
            pd[u] = a.dz[in ? ((long long)gx * a.n1 + gy) * a.n2 + gz : 0];
        }
    };
    auto put = [&](char *buf) {
#pragma unroll
        for (int u = 0; u < NX; ++u)
            reinterpret_cast<uint4 *>(buf)[tid + u * WG_THREADS] = (xin >> u) & 1u ? px[u] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int u = 0; u < ND; ++u) {
            const int e = tid + u * WG_THREADS, hz = e % HZ, row = e / HZ % (OW_Y + 2), pl = e / (HZ * (OW_Y + 2));
            if (e >= OW_HALO) continue;
            const uint16_t v = (din >> u) & 1u ? pd[u] : (uint16_t)0;
#pragma unroll
            for (int c = 0; c < 3; ++c)
                if (hz >= c && hz - c < 32)
                    *reinterpret_cast<uint16_t *>(buf + OW_XB + c * OW_COPY + pl * OW_PL + row * OW_ROW + (hz - c) * 2) = v;
        }
    };
    f32x16 acc[2] = {f32x16{}, f32x16{}};
    if ((int)blockIdx.x < total) {
        fetch(blockIdx.x);
        put(lds);
    }
    int cur = 0;
    for (int b = blockIdx.x; b < total; b += gridDim.x, cur ^= 1) {
        lds_barrier();     // this tile's buffer written; the other one read by every wave
        const char *buf = lds + cur * OW_BUF;
        if (b + (int)gridDim.x < total) fetch(b + gridDim.x);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            uint4 f = *reinterpret_cast<const uint4 *>(buf + aoff + c * 32);
            if (m >= 27) f = make_uint4(0u, 0u, 0u, 0u);
            const uint2 b0 = lds_read_tr(buf + boff + c * 16 * 64), b1 = lds_read_tr(buf + boff + (c * 16 + 4) * 64);
            acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f), frag4(b0.x, b0.y, b1.x, b1.y),
                                                             acc[c], 0, 0, 0);
        }
        if (b + (int)gridDim.x < total) put(lds + (cur ^ 1) * OW_BUF);
    }
    // work[blockIdx][tap][ci]: the waves' sums in wave order
    float *red = reinterpret_cast<float *>(lds_u4);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int t = mfma_row(i, lane);
        if (t < 27) red[(wave * 27 + t) * 32 + m] = acc[0][i] + acc[1][i];
    }
    __syncthreads();
    for (int e = tid; e < 27 * 32; e += WG_THREADS) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) sum += red[w * 27 * 32 + e];
        a.work[(size_t)blockIdx.x * 27 * 32 + e] = sum;
    }
}

// Input: dh[v][ci] = sum_t dr[v + d(t)] w[26 - t][0][ci], the 27 taps as one K of 32 (two
// MFMAs per 32 voxels instead of 54), with the epilogue of cnn_conv_march's first gradient
// layer (dh, ReLU mask, dz', channel sums) and its columns; dr planes (8 + 2 rows) go round a ring of four.  Bound by storing dh and dz'
// (402 MB at 128^3): 106 us (cnn_conv_march on 32 channels of dr) -> 85; 98 with that
// kernel's segments, one workgroup a CU.
constexpr int OG_ROW = 36, OG_PLANE = (MR_Y + 2) * OG_ROW;               // voxels of a dr row, a plane
constexpr size_t OG_LDS = 4 * OG_PLANE * 2 + 8 * FWD_STAGE;

__global__ __launch_bounds__(FWD_THREADS) void cnn_out_grad(MarchArgs q) {
    extern __shared__ uint4 lds_u4[];
    const ConvArgs &a = q.c;
    char *stage = reinterpret_cast<char *>(lds_u4);
    uint16_t *ring = reinterpret_cast<uint16_t *>(stage + 8 * FWD_STAGE);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char *stg = stage + wave * FWD_STAGE;
    const int m = lane & 31, kh = lane >> 5;
    const int cols = q.nby * q.nbz * q.nseg, per = gridDim.x / 8;
    const int col = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (col >= cols) return;
    const int bz = col % q.nbz, by = col / q.nbz % q.nby, x0 = col / (q.nbz * q.nby) * q.seg;
    const int x1 = min(x0 + q.seg, a.n0), y0 = by * MR_Y, z0 = bz * 32;
    const long long pvox = (long long)a.n1 * a.n2;
    // weights: row ci = m, K = tap
    bf16x8 wf[2];
    int toff[2][8], tdx[2][8];             // this lane half's taps: offset in a plane, plane
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        uint32_t w2[4];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int t = c * 16 + kh * 8 + j, tt = min(t, 26);
            const uint32_t v = t < 27 ? a.w[(size_t)(26 - tt) * 32 * 32 + m] : 0u;
            w2[j >> 1] = j & 1 ? w2[j >> 1] | v << 16 : v;
            tdx[c][j] = tt / 9 - 1;
            toff[c][j] = (wave + tt / 3 % 3) * OG_ROW + m + tt % 3;
        }
        wf[c] = frag4(w2[0], w2[1], w2[2], w2[3]);
    }
    // one halo voxel of a plane per thread
    const int hy = tid / HZ, hz = tid % HZ, gy = y0 + hy - 1, gz = z0 + hz - 1;
    const bool mine = tid < (MR_Y + 2) * HZ, in = mine && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
    const long long goff = in ? (long long)gy * a.n2 + gz : 0;
    auto fetch = [&](int p) { return a.x[(p >= 0 && p < a.n0 ? p : 0) * pvox + goff]; };
    auto put = [&](int p, uint16_t v) {
        if (mine) ring[(p & 3) * OG_PLANE + hy * OG_ROW + hz] = in && p >= 0 && p < a.n0 ? v : (uint16_t)0;
    };
    for (int p = x0 - 1; p <= x0 + 1; ++p) put(p, fetch(p));
    lds_barrier();
    const int oy = y0 + wave;
    const bool live = oy < a.n1;           // wave-uniform
    const long long row0 = (long long)min(oy, a.n1 - 1) * a.n2 + z0;
    u32x4 *yb = reinterpret_cast<u32x4 *>(a.y) + row0 * 4;
    float bs[16] = {};
    for (int p = x0; p < x1; ++p) {
        if (p > x0) lds_barrier();         // plane p + 1 written; slot (p + 2) & 3 read by every wave
        const uint16_t next = fetch(p + 2);
        const long long vox = p * pvox + row0 + m;
        uint32_t mk = a.mask[vox];
        f32x16 acc = {};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            uint32_t f[4];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                // (zeros past the last tap: an infinite dr times a zero weight is not 0)
                const uint32_t v = c * 16 + kh * 8 + j < 27 ? ring[((p + tdx[c][j]) & 3) * OG_PLANE + toff[c][j]] : 0u;
                f[j >> 1] = j & 1 ? f[j >> 1] | v << 16 : v;
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[c], frag4(f[0], f[1], f[2], f[3]), acc, 0, 0, 0);
        }
        put(p + 2, next);
        mk = live ? mk >> (4 * kh) : 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4 d;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                d[j] = acc[4 * g + j];
                v[j] = (mk >> (8 * g + j)) & 1u ? d[j] : 0.0f;
                bs[4 * g + j] += v[j];
            }
            if (live) reinterpret_cast<f32x4 *>(q.dh_out)[vox * 8 + 2 * g + kh] = d;
            *reinterpret_cast<uint2 *>(stg + m * 64 + ((g ^ ((m >> 2) & 3)) << 4) + kh * 8) =
                make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        }
        if (live) {
            u32x4 *dst = yb + p * pvox * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int v = h * 16 + (lane >> 2);
                dst[h * 64 + lane] = *reinterpret_cast<const u32x4 *>(stg + v * 64 + (((lane & 3) ^ ((v >> 2) & 3)) << 4));
            }
        }
    }
    float *red = reinterpret_cast<float *>(lds_u4);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float v = bs[i];
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (m == 0) red[wave * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)] = v;
    }
    lds_barrier();
    if (tid < 32) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) v += red[w * 32 + tid];
        q.part[(size_t)col * 32 + tid] = v;
    }
}

// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void cnn_flip(const uint16_t *w, uint16_t *wt) {
    const int i = blockIdx.x * 256 + threadIdx.x;     // over 27*32*32
    if (i >= 27 * 32 * 32) return;
    const int ci = i & 31, co = (i >> 5) & 31, tap = i >> 10;
    // wt[tap][ci][co] = w[26 - tap][co][ci]  (stored with the second index as "cout")
    wt[((size_t)tap * 32 + ci) * 32 + co] = w[((size_t)(26 - tap) * 32 + co) * 32 + ci];
}

__global__ __launch_bounds__(256) void cnn_relu_grad(const float *__restrict__ dh, const uint16_t *__restrict__ act,
                                                     uint16_t *__restrict__ dz, float *__restrict__ part,
                                                     long long n) {
    __shared__ float red[8][32];
    const int c = threadIdx.x & 31, vo = threadIdx.x >> 5;
    float sum = 0.0f;
    const long long base = (long long)blockIdx.x * 1024;
    for (int k = 0; k < 128; ++k) {
        const long long v = base + k * 8 + vo;
        if (v < n) {
            const long long idx = v * 32 + c;
            const uint16_t av = act[idx];
            const float g = ((av & 0x8000u) == 0 && av != 0) ? dh[idx] : 0.0f;
            dz[idx] = f2bf(g);
            sum += g;
        }
    }
    red[vo][c] = sum;
    __syncthreads();
    if (threadIdx.x < 32) {
        float s = 0.0f;
        for (int j = 0; j < 8; ++j) s += red[j][threadIdx.x];
        part[(size_t)blockIdx.x * 32 + threadIdx.x] = s;
    }
}

// ROWS: dr as channel 0 of 32 (the layout of pvd_cnn_wgrad and pvd_cnn_layer_grad); else
// [n].  Four voxels' loads in flight a thread: 128^3 with rows 56 us (64 bytes stored a
// voxel), without 14.
template <bool ROWS>
__global__ __launch_bounds__(256) void cnn_loss(const float *__restrict__ r, const float *__restrict__ dp,
                                                const float *__restrict__ dt, const float *__restrict__ mk,
                                                long long n, float inv_count, uint16_t *__restrict__ dr,
                                                float *__restrict__ part) {
    __shared__ float red[3][256];
    float se = 0.0f, sw = 0.0f, sg = 0.0f;
    const long long step = (long long)gridDim.x * 256;
    constexpr int U = 4;
    for (long long v0 = blockIdx.x * 256LL + threadIdx.x; v0 < n; v0 += U * step) {
        float xw[U], xp[U], xr[U], xt[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long v = v0 + u * step < n ? v0 + u * step : v0;
            xw[u] = mk[v];
            xp[u] = dp[v];
            xr[u] = r[v];
            xt[u] = dt[v];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long v = v0 + u * step;
            if (v >= n) break;
            const float w = xw[u];
            const float e = xp[u] * xr[u] - (xt[u] - xp[u]);
            se += w * e * e;
            sw += w;
            const uint16_t g = f2bf(2.0f * w * e * xp[u] * inv_count);
            sg += bf2f(g);
            if (ROWS) {
                uint4 *row = reinterpret_cast<uint4 *>(dr + v * 32);
                row[0] = make_uint4((uint32_t)g, 0u, 0u, 0u);
                row[1] = make_uint4(0u, 0u, 0u, 0u);
                row[2] = make_uint4(0u, 0u, 0u, 0u);
                row[3] = make_uint4(0u, 0u, 0u, 0u);
            } else {
                dr[v] = g;
            }
        }
    }
    red[0][threadIdx.x] = se;
    red[1][threadIdx.x] = sw;
    red[2][threadIdx.x] = sg;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] += red[1][threadIdx.x + s];
            red[2][threadIdx.x] += red[2][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x < 3) part[3 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void cnn_adam(float *p, const float *g, float *m, float *v, uint16_t *pb, long long n,
                                                float lr, float b1, float b2, float eps, float c1, float c2) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float pi = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
        p[i] = pi;
        if (pb) pb[i] = f2bf(pi);
    }
}

// Column sums of part[rows][cols] in a fixed order: a workgroup takes 32 columns, its 32
// row groups each sum rows g, g + 32, ... (8 loads in flight), then a pairwise sum over
// the groups in LDS.  (A thread per column walking all rows is one serial chain of loads
// on cols / 256 blocks: the 2048 x 32 bias partials of a 128^3 layer took about 460 us and
// the 256 x 27648 weight partials 61 us; both now take 4-6 us.)
constexpr int RED_COLS = 32, RED_GROUPS = 32;
constexpr int RED_GRID = 1 << 20;      // workgroups (at most; a launch has fewer than 2^32 threads)
__global__ __launch_bounds__(RED_COLS * RED_GROUPS) void reduce_rows(const float *__restrict__ part, unsigned rows,
                                                                     unsigned cols, float *__restrict__ out,
                                                                     int accumulate, int pitch) {
    __shared__ float red[RED_GROUPS][RED_COLS + 1];
    const unsigned l = threadIdx.x & (RED_COLS - 1), g = threadIdx.x / RED_COLS;
    for (unsigned b = blockIdx.x; b * RED_COLS < cols; b += gridDim.x) {       // (rows, cols < 2^31)
        const unsigned c = b * RED_COLS + l;
        const float *p = part + (c < cols ? c : cols - 1);
        float s = 0.0f;
        for (unsigned r0 = g; r0 < rows; r0 += 8 * RED_GROUPS) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[(size_t)min(r0 + u * RED_GROUPS, rows - 1) * cols];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += r0 + u * RED_GROUPS < rows ? v[u] : 0.0f;
        }
        if (b != blockIdx.x) __syncthreads();                                  // red is free again
        red[g][l] = s;
        __syncthreads();
#pragma unroll
        for (int h = RED_GROUPS / 2; h > 0; h >>= 1) {
            if (g < (unsigned)h) red[g][l] += red[g + h][l];
            __syncthreads();
        }
        float *o = out + (size_t)b * pitch + l;                  // `pitch` floats per 32 columns
        if (g == 0 && c < cols) *o = accumulate ? *o + red[0][l] : red[0][l];
    }
}

__global__ __launch_bounds__(256) void cnn_pack(const float *__restrict__ a, const float *__restrict__ d,
                                                const float *__restrict__ dp, const float *__restrict__ amax,
                                                const float *__restrict__ dmax, uint16_t *__restrict__ x,
                                                long long n) {
    const float sa = inv_scale(amax), sd = inv_scale(dmax);
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < n; v += (long long)gridDim.x * 256) {
        const uint2 c = pack_input(a[v], d[v], dp[v], sa, sd);
        uint4 *row = reinterpret_cast<uint4 *>(x + v * 16);
        row[0] = make_uint4(c.x, c.y, 0u, 0u);
        row[1] = make_uint4(0u, 0u, 0u, 0u);
    }
}

__global__ __launch_bounds__(256) void cnn_apply(const float *__restrict__ dp, const float *__restrict__ r,
                                                 float bound, const float *__restrict__ dmax, float region_frac,
                                                 float apply_frac, float *__restrict__ out,
                                                 unsigned long long *__restrict__ counts, long long n) {
    __shared__ unsigned red[2][256];
    const float region_min = region_frac * *dmax;
    const float apply_min = apply_frac * *dmax;
    unsigned ex = 0, reg = 0;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < n; v += (long long)gridDim.x * 256) {
        const float d = dp[v];
        const bool applied = d >= apply_min;     // r is read (and defined) only there
        const float rv = applied ? r[v] : 0.0f;
        const bool ok = fabsf(rv) <= bound;      // NaN fails too
        out[v] = (ok && applied) ? d * (1.0f + rv) : d;
        const bool in_region = d >= region_min;
        ex += (!ok && in_region) ? 1u : 0u;
        reg += in_region ? 1u : 0u;
    }
    red[0][threadIdx.x] = ex;
    red[1][threadIdx.x] = reg;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] += red[1][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (red[0][0]) atomicAdd(&counts[0], (unsigned long long)red[0][0]);
        if (red[1][0]) atomicAdd(&counts[1], (unsigned long long)red[1][0]);
    }
}

// Maxima of the activity and of the plain dose (the network input's scales) in one pass:
// per-block maxima into part[2 * block + {0, 1}], then one block reduces them into
// out[0], out[1].  A maximum is exact, whatever the order.
constexpr int MAX2_BLOCKS = (PVD_CNN_MAXIMA_FLOATS - 2) / 2;   // partial maxima per call

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

__global__ __launch_bounds__(256) void cnn_max2_part(const float *__restrict__ a, const float *__restrict__ b,
                                                     long long n, float *__restrict__ part) {
    __shared__ float red[2][4];
    float ma = -INFINITY, mb = -INFINITY;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < n; v += (long long)gridDim.x * 256) {
        ma = fmaxf(ma, a[v]);
        mb = fmaxf(mb, b[v]);
    }
    ma = wave_max(ma);
    mb = wave_max(mb);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = ma;
        red[1][threadIdx.x >> 6] = mb;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const float *r = red[threadIdx.x];
        part[2 * blockIdx.x + threadIdx.x] = fmaxf(fmaxf(r[0], r[1]), fmaxf(r[2], r[3]));
    }
}

__global__ __launch_bounds__(256) void cnn_max2_final(const float *__restrict__ part, int nb, float *__restrict__ out) {
    __shared__ float red[2][4];
    float ma = -INFINITY, mb = -INFINITY;
    for (int i = threadIdx.x; i < nb; i += 256) {
        ma = fmaxf(ma, part[2 * i]);
        mb = fmaxf(mb, part[2 * i + 1]);
    }
    ma = wave_max(ma);
    mb = wave_max(mb);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = ma;
        red[1][threadIdx.x >> 6] = mb;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const float *r = red[threadIdx.x];
        out[threadIdx.x] = fmaxf(fmaxf(r[0], r[1]), fmaxf(r[2], r[3]));
    }
}

// Whole-volume fallback decided on the device from cnn_apply's counts: out = dp when
// counts[1] > 0 and counts[0] > max_exceed_frac * counts[1]; otherwise every block
// returns at once.
__global__ __launch_bounds__(256) void cnn_fallback(const float *__restrict__ dp,
                                                    const unsigned long long *__restrict__ counts,
                                                    double max_exceed_frac, float *__restrict__ out, long long n) {
    const unsigned long long ex = counts[0], reg = counts[1];
    if (!(reg > 0 && (double)ex > max_exceed_frac * (double)reg)) return;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < n; v += (long long)gridDim.x * 256) out[v] = dp[v];
}

// Region blocks of the forward kernel (FWD_BX x FWD_BY x 32 output voxels):
// flag[b] = 1 if block b holds a voxel with dp >= frac * max; count reset.
__global__ __launch_bounds__(256) void cnn_block_flags(const float *__restrict__ dp, int n0, int n1, int n2,
                                                       const float *__restrict__ dmax, float frac,
                                                       int *__restrict__ flag, int *__restrict__ count) {
    const int nby = (n1 + FWD_BY - 1) / FWD_BY, nbz = n2 >> 5;
    const int b = blockIdx.x;
    const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
    const float thr = frac * *dmax;
    const int t = threadIdx.x;                       // 256 = FWD_BX * FWD_BY * 32 voxels
    const int z = bz * 32 + (t & 31), y = by * FWD_BY + ((t >> 5) % FWD_BY), x = bx * FWD_BX + (t >> 5) / FWD_BY;
    const bool hit = x < n0 && y < n1 && dp[((long long)x * n1 + y) * n2 + z] >= thr;
    const int any = __syncthreads_or(hit ? 1 : 0);
    if (t == 0) flag[b] = any ? 1 : 0;
    if (b == 0 && t == 0) *count = 0;
}

// list the blocks within (3, 2, 1) blocks (6 voxels, the network's receptive field)
// of a flagged block; the order follows the atomic slots (the outputs do not depend on it)
__global__ __launch_bounds__(256) void cnn_block_list(const int *__restrict__ flag, int nbx, int nby, int nbz,
                                                      int *__restrict__ list, int *__restrict__ count) {
    const int total = nbx * nby * nbz;
    for (int b = blockIdx.x * 256 + threadIdx.x; b < total; b += gridDim.x * 256) {
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        bool near = false;
        for (int i = max(bx - 3, 0); i <= min(bx + 3, nbx - 1) && !near; ++i)
            for (int j = max(by - 2, 0); j <= min(by + 2, nby - 1) && !near; ++j)
                for (int k = max(bz - 1, 0); k <= min(bz + 1, nbz - 1); ++k)
                    if (flag[(i * nby + j) * nbz + k]) { near = true; break; }
        if (near) list[atomicAdd(count, 1)] = b;
    }
}

int g_num_cus = 0;

int num_cus() {
    if (g_num_cus == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            g_num_cus = v;
        else
            g_num_cus = 256;
    }
    return g_num_cus;
}

template <int CIN, int EPI, bool MASK = false>
hipError_t launch_fwd(const ConvArgs &a, int blocks, hipStream_t st) {
    static pvd_device_once once;
    if (hipError_t e = pvd_lds_limit(once, cnn_conv_fwd<CIN, EPI, MASK>, fwd_lds_bytes<CIN>()); e != hipSuccess) return e;
    hipLaunchKernelGGL((cnn_conv_fwd<CIN, EPI, MASK>), dim3(blocks), dim3(FWD_THREADS), fwd_lds_bytes<CIN>(), st, a);
    return hipGetLastError();
}

// Segments along x of the marching kernel: the count that minimises the rounds of
// workgroups times a segment's steps (its planes and about two for the start).
void march_plan(MarchArgs *q, int n0, int n1, int n2) {
    q->nby = (n1 + MR_Y - 1) / MR_Y;
    q->nbz = n2 >> 5;
    const long long cols = (long long)q->nby * q->nbz;
    long long best = -1;
    for (int s = 1; s <= n0 && s <= 1024; ++s) {
        const int seg = (n0 + s - 1) / s, nseg = (n0 + seg - 1) / seg;
        const long long cost = (cols * nseg + num_cus() - 1) / num_cus() * (seg + 2);
        if (best < 0 || cost < best) {
            best = cost;
            q->seg = seg;
            q->nseg = nseg;
        }
    }
}

// cnn_out_grad: segments half as long, for two workgroups a CU (a segment's halo is two planes
// of one-channel dr)
void out_grad_plan(MarchArgs *q, int n0, int n1, int n2) {
    march_plan(q, n0, n1, n2);
    q->seg = (q->seg + 1) / 2;
    q->nseg = (n0 + q->seg - 1) / q->seg;
}

template <int MODE>
hipError_t launch_march(MarchArgs &q, hipStream_t st) {
    static pvd_device_once once;
    if (hipError_t e = pvd_lds_limit(once, cnn_conv_march<MODE>, MR_LDS); e != hipSuccess) return e;
    march_plan(&q, q.c.n0, q.c.n1, q.c.n2);
    const long long grid = ((long long)q.nby * q.nbz * q.nseg + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(cnn_conv_march<MODE>, dim3((unsigned)grid), dim3(FWD_THREADS), MR_LDS, st, q);
    return hipGetLastError();
}

hipError_t launch_layer(const ConvArgs &a, hipStream_t st) {
    MarchArgs q{};
    q.c = a;
    return a.mask ? launch_march<MR_MASK>(q, st) : launch_march<MR_FWD>(q, st);
}

template <int BX, int BY, bool MAPS>
hipError_t launch_in_as(const ConvArgs &a, const InMaps &mp, int blocks, hipStream_t st) {
    static pvd_device_once once;
    constexpr size_t lds = in_lds_bytes<BX, BY>();
    if (hipError_t e = pvd_lds_limit(once, cnn_conv_in<BX, BY, MAPS>, lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((cnn_conv_in<BX, BY, MAPS>), dim3(blocks), dim3(FWD_THREADS), lds, st, a, mp);
    return hipGetLastError();
}

template <int BX, int BY>
hipError_t launch_in(const ConvArgs &a, const InMaps *mp, int blocks, hipStream_t st) {
    return mp ? launch_in_as<BX, BY, true>(a, *mp, blocks, st) : launch_in_as<BX, BY, false>(a, InMaps{}, blocks, st);
}

template <int BX, int BY>
hipError_t launch_out(const ConvArgs &a, int blocks, hipStream_t st) {
    static pvd_device_once once;
    constexpr size_t lds = out_lds_bytes<BX, BY>();
    if (hipError_t e = pvd_lds_limit(once, cnn_conv_out<BX, BY>, lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((cnn_conv_out<BX, BY>), dim3(blocks), dim3(FWD_THREADS), lds, st, a);
    return hipGetLastError();
}

hipError_t launch_out_march(const ConvArgs &a, hipStream_t st) {
    static pvd_device_once once;
    if (hipError_t e = pvd_lds_limit(once, cnn_conv_out_march, OM_LDS); e != hipSuccess) return e;
    // two workgroups a CU (77 KB of LDS each), segments of at least 4 planes
    const int nby = (a.n1 + OM_Y - 1) / OM_Y, nbz = a.n2 >> 5;
    const long long cols = (long long)nby * nbz;
    const long long want = std::max(1LL, 2LL * num_cus() / cols);
    const int seg = std::max(4, (int)((a.n0 + want - 1) / want));
    const long long grid = cols * ((a.n0 + seg - 1) / seg);
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(cnn_conv_out_march, dim3((unsigned)grid), dim3(OM_THREADS), OM_LDS, st, a, seg, nby, nbz);
    return hipGetLastError();
}

// whole volumes (no region list): 4 x 4-row blocks for the input layer, the marching
// kernel for the output layer
template <bool IN>
hipError_t launch_io(const ConvArgs &a, int grid, bool whole, hipStream_t st, const InMaps *mp = nullptr) {
    if (whole && !IN) return launch_out_march(a, st);
    if (whole) {
        const long long t = (long long)((a.n0 + 3) / 4) * ((a.n1 + 3) / 4) * (a.n2 >> 5);
        return launch_in<4, 4>(a, mp, (int)(t < num_cus() ? t : num_cus()), st);
    }
    return IN ? launch_in<FWD_BX, FWD_BY>(a, mp, grid, st) : launch_out<FWD_BX, FWD_BY>(a, grid, st);
}

template <int CIN>
hipError_t launch_wgrad(const WgradArgs &a, int blocks, hipStream_t st) {
    static pvd_device_once once;
    if (hipError_t e = pvd_lds_limit(once, cnn_wgrad<CIN>, wg_lds<CIN>()); e != hipSuccess) return e;
    hipLaunchKernelGGL((cnn_wgrad<CIN>), dim3(blocks), dim3(WG_THREADS), wg_lds<CIN>(), st, a);
    return hipGetLastError();
}

int check_grid(int n0, int n1, int n2) {
    if (n0 < 1 || n1 < 1 || n2 < 32 || (n2 & 31))
        return pvd_set_error(PVD_EINVAL, "CNN grid %dx%dx%d: need n2 a positive multiple of 32", n0, n1, n2);
    return PVD_OK;
}

int wgrad_blocks(int n0, int n1, int n2) {
    const long long total = (long long)((n0 + WG_BX - 1) / WG_BX) * ((n1 + WG_BY - 1) / WG_BY) * (n2 >> 5);
    return (int)(total < WG_MAX_BLOCKS ? total : WG_MAX_BLOCKS);
}

}  // namespace

// =================================================================================
extern "C" {

int pvd_cnn_conv_fwd(const void *x, int cin, const void *w, const float *bias, int epi, const void *resid, void *y,
                     void *act, float *y32, int n0, int n1, int n2, const int *blocks, const int *nblocks,
                     void *stream) {
    if ((blocks == nullptr) != (nblocks == nullptr)) return pvd_set_error(PVD_EINVAL, "blocks and nblocks go together");
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!x || !w) return pvd_set_error(PVD_EINVAL, "null input or weights");
    if (cin != 4 && cin != 16 && cin != 32) return pvd_set_error(PVD_EINVAL, "cin must be 4, 16 or 32 (got %d)", cin);
    if (cin == 4 && (epi != PVD_CNN_EPI_RELU || act))
        return pvd_set_error(PVD_EINVAL, "cin 4 (the input layer) takes the ReLU epilogue without act");
    switch (epi) {
        case PVD_CNN_EPI_RELU: if (!y) return pvd_set_error(PVD_EINVAL, "null output"); break;
        case PVD_CNN_EPI_RESID_RELU:
            if (!y || !resid) return pvd_set_error(PVD_EINVAL, "residual layer needs y and resid");
            break;
        case PVD_CNN_EPI_LINEAR_F32:
        case PVD_CNN_EPI_ACCUM_F32: if (!y32) return pvd_set_error(PVD_EINVAL, "null FP32 output"); break;
        default: return pvd_set_error(PVD_EINVAL, "unknown epilogue %d", epi);
    }
    // BF16 outputs are written as 16-byte chunks of whole 32-voxel tiles
    if ((epi == PVD_CNN_EPI_RELU || epi == PVD_CNN_EPI_RESID_RELU) &&
        ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(act)) & 15))
        return pvd_set_error(PVD_EINVAL, "y and act must be 16-byte aligned");
    ConvArgs a{(const uint16_t *)x, (const uint16_t *)w, bias, (const uint16_t *)resid, (uint16_t *)y,
               (uint16_t *)act, y32, n0, n1, n2, blocks, nblocks, nullptr};
    const long long total = (long long)((n0 + FWD_BX - 1) / FWD_BX) * ((n1 + FWD_BY - 1) / FWD_BY) * (n2 >> 5);
    const int grid = (int)(total < num_cus() ? total : num_cus());
    hipStream_t st = (hipStream_t)stream;
    hipError_t e;
    if (cin == 4) {
        e = launch_io<true>(a, grid, blocks == nullptr, st);
    } else if (cin == 16) {
        switch (epi) {
            case 0: e = launch_fwd<16, 0>(a, grid, st); break;
            case 1: e = launch_fwd<16, 1>(a, grid, st); break;
            case 2: e = launch_fwd<16, 2>(a, grid, st); break;
            default: e = launch_fwd<16, 3>(a, grid, st); break;
        }
    } else {
        switch (epi) {
            case 0: e = launch_fwd<32, 0>(a, grid, st); break;
            case 1:
                e = !blocks && !act && resid == x ? launch_layer(a, st) : launch_fwd<32, 1>(a, grid, st);
                break;
            case 2: e = launch_io<false>(a, grid, blocks == nullptr, st); break;
            default: e = launch_fwd<32, 3>(a, grid, st); break;
        }
    }
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch CNN convolution");
}

int pvd_cnn_input_layer(const float *activity, const float *density, const float *dose_plain, const float *act_max,
                        const float *dose_max, long long pitch, const void *w, const float *bias, void *y, int n0,
                        int n1, int n2, const int *blocks, const int *nblocks, void *stream) {
    if ((blocks == nullptr) != (nblocks == nullptr)) return pvd_set_error(PVD_EINVAL, "blocks and nblocks go together");
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!activity || !density || !dose_plain || !act_max || !dose_max || !w || !y)
        return pvd_set_error(PVD_EINVAL, "null argument");
    if (pitch < n2) return pvd_set_error(PVD_EINVAL, "pitch %lld below the row length %d", pitch, n2);
    if (reinterpret_cast<uintptr_t>(y) & 15) return pvd_set_error(PVD_EINVAL, "y must be 16-byte aligned");
    const ConvArgs a{nullptr, (const uint16_t *)w, bias, nullptr, (uint16_t *)y, nullptr, nullptr, n0, n1, n2, blocks,
                     nblocks, nullptr};
    const InMaps mp{{activity, density, dose_plain}, act_max, dose_max, pitch};
    const long long total = (long long)((n0 + FWD_BX - 1) / FWD_BX) * ((n1 + FWD_BY - 1) / FWD_BY) * (n2 >> 5);
    const hipError_t e = launch_io<true>(a, (int)(total < num_cus() ? total : num_cus()), blocks == nullptr,
                                         (hipStream_t)stream, &mp);
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch CNN input layer");
}

int pvd_cnn_train_layer(const void *x, int cin, const void *w, const float *bias, void *y, unsigned *mask, int n0,
                        int n1, int n2, void *stream) {
    return pvd_cnn_train_layer_blocks(x, cin, w, bias, y, mask, n0, n1, n2, nullptr, nullptr, stream);
}

int pvd_cnn_train_layer_blocks(const void *x, int cin, const void *w, const float *bias, void *y, unsigned *mask,
                               int n0, int n1, int n2, const int *blocks, const int *nblocks, void *stream) {
    if ((blocks == nullptr) != (nblocks == nullptr)) return pvd_set_error(PVD_EINVAL, "blocks and nblocks go together");
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!x || !w || !y || !mask) return pvd_set_error(PVD_EINVAL, "null argument");
    if (cin != 4 && cin != 32) return pvd_set_error(PVD_EINVAL, "cin must be 4 or 32 (got %d)", cin);
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15)
        return pvd_set_error(PVD_EINVAL, "x and y must be 16-byte aligned");
    ConvArgs a{(const uint16_t *)x, (const uint16_t *)w, bias, (const uint16_t *)x, (uint16_t *)y, nullptr, nullptr,
               n0, n1, n2, blocks, nblocks, mask};
    const long long total = (long long)((n0 + FWD_BX - 1) / FWD_BX) * ((n1 + FWD_BY - 1) / FWD_BY) * (n2 >> 5);
    const int grid = (int)(total < num_cus() ? total : num_cus());
    hipStream_t st = (hipStream_t)stream;
    const hipError_t e = cin == 4 ? launch_io<true>(a, grid, !blocks, st)
                         : blocks ? launch_fwd<32, PVD_CNN_EPI_RESID_RELU, true>(a, grid, st) : launch_layer(a, st);
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch CNN training layer");
}

size_t pvd_cnn_grad_parts(int n0, int n1, int n2) {
    if (n0 < 1 || n1 < 1 || n2 < 32) return 0;
    MarchArgs q{};
    march_plan(&q, n0, n1, n2);
    return (size_t)q.nby * q.nbz * q.nseg;
}

int pvd_cnn_layer_grad(const void *dz, const void *w_flipped, const float *dh_in, float *dh_out, const unsigned *mask,
                       void *dz_out, float *dbias_part, int n0, int n1, int n2, void *stream) {
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!dz || !w_flipped || !mask || !dz_out || !dbias_part || (!dh_in && !dh_out))
        return pvd_set_error(PVD_EINVAL, "null argument");
    if (dz == dz_out) return pvd_set_error(PVD_EINVAL, "dz and dz_out must differ");
    if ((reinterpret_cast<uintptr_t>(dz) | reinterpret_cast<uintptr_t>(dz_out) | reinterpret_cast<uintptr_t>(dh_in) |
         reinterpret_cast<uintptr_t>(dh_out)) & 15)
        return pvd_set_error(PVD_EINVAL, "dz, dz_out, dh_in and dh_out must be 16-byte aligned");
    MarchArgs q{};
    q.c = ConvArgs{(const uint16_t *)dz, (const uint16_t *)w_flipped, nullptr, nullptr, (uint16_t *)dz_out, nullptr,
                   nullptr, n0, n1, n2, nullptr, nullptr, const_cast<unsigned *>(mask)};
    q.dh_in = dh_in;
    q.dh_out = dh_out;
    q.part = dbias_part;
    hipStream_t st = (hipStream_t)stream;
    const hipError_t e = !dh_in ? launch_march<MR_GRAD_FIRST>(q, st)
                         : dh_out ? launch_march<MR_GRAD>(q, st) : launch_march<MR_GRAD_LAST>(q, st);
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch CNN layer gradient");
}

int pvd_cnn_flip_weights(const void *w, void *wt, void *stream) {
    if (!w || !wt) return pvd_set_error(PVD_EINVAL, "null argument");
    hipLaunchKernelGGL(cnn_flip, dim3((27 * 32 * 32 + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t *)w, (uint16_t *)wt);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch weight flip");
}

int pvd_cnn_relu_grad(const float *dh, const void *act, void *dz, float *dbias_part, long long n, void *stream) {
    if (!dh || !act || !dz || !dbias_part || n < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    const long long blocks = (n + 1023) / 1024;
    if (blocks > 0x7fffffffLL) return pvd_set_error(PVD_ENOTSUP, "too many voxels");
    hipLaunchKernelGGL(cnn_relu_grad, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, dh,
                       (const uint16_t *)act, (uint16_t *)dz, dbias_part, n);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch ReLU gradient");
}

size_t pvd_cnn_wgrad_work_floats(int n0, int n1, int n2) {
    if (n0 < 1 || n1 < 1 || n2 < 32) return 0;
    return (size_t)wgrad_blocks(n0, n1, n2) * 27 * 32 * 32;
}

int pvd_cnn_wgrad(const void *x, int cin, const void *dz, float *dw, float *work, int n0, int n1, int n2,
                  void *stream) {
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!x || !dz || !dw || !work) return pvd_set_error(PVD_EINVAL, "null argument");
    if (cin != 16 && cin != 32) return pvd_set_error(PVD_EINVAL, "cin must be 16 or 32 (got %d)", cin);
    WgradArgs a{(const uint16_t *)x, (const uint16_t *)dz, work, n0, n1, n2};
    const int blocks = wgrad_blocks(n0, n1, n2);
    hipStream_t st = (hipStream_t)stream;
    hipError_t e = cin == 16 ? launch_wgrad<16>(a, blocks, st) : launch_wgrad<32>(a, blocks, st);
    if (e != hipSuccess) return pvd_hip_error(e, "launch weight gradient");
    const int cols = 27 * 32 * cin;
    hipLaunchKernelGGL(reduce_rows, dim3(std::min((cols - 1) / RED_COLS + 1, RED_GRID)), dim3(RED_COLS * RED_GROUPS), 0, st,
                       (const float *)work, blocks, cols, dw, 0, RED_COLS);
    e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch reduction");
}

int pvd_cnn_loss(const float *r, const float *dp, const float *dt, const float *m, long long n, float inv_count,
                 void *dr, float *loss_part, void *stream) {
    if (!r || !dp || !dt || !m || !dr || !loss_part || n < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    hipLaunchKernelGGL(cnn_loss<true>, dim3(PVD_CNN_LOSS_BLOCKS), dim3(256), 0, (hipStream_t)stream, r, dp, dt, m, n, inv_count,
                       (uint16_t *)dr, loss_part);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch loss");
}

int pvd_cnn_out_loss(const float *r, const float *dp, const float *dt, const float *m, long long n, float inv_count,
                     void *dr, float *loss_part, void *stream) {
    if (!r || !dp || !dt || !m || !dr || !loss_part || n < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    hipLaunchKernelGGL(cnn_loss<false>, dim3(PVD_CNN_LOSS_BLOCKS), dim3(256), 0, (hipStream_t)stream, r, dp, dt, m, n,
                       inv_count, (uint16_t *)dr, loss_part);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch loss");
}

int pvd_cnn_out_wgrad(const void *x, const void *dr, float *dw, float *work, int n0, int n1, int n2, void *stream) {
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!x || !dr || !dw || !work) return pvd_set_error(PVD_EINVAL, "null argument");
    if (reinterpret_cast<uintptr_t>(x) & 15) return pvd_set_error(PVD_EINVAL, "x must be 16-byte aligned");
    static pvd_device_once once;
    if (hipError_t e = pvd_lds_limit(once, cnn_out_wgrad, OW_LDS); e != hipSuccess) return pvd_hip_error(e, "set LDS limit");
    const long long total = (long long)n0 * ((n1 + OW_Y - 1) / OW_Y) * (n2 >> 5);
    if (total > 0x7fffffffLL) return pvd_set_error(PVD_ENOTSUP, "grid too large");
    // (32 partial sums of this layer fit where pvd_cnn_wgrad_work_floats has one workgroup's)
    const long long most = std::min<long long>((long long)OW_BLOCKS_PER_CU * num_cus(), 32LL * wgrad_blocks(n0, n1, n2));
    const int blocks = (int)std::min(total, most);
    hipStream_t st = (hipStream_t)stream;
    const WgradArgs a{(const uint16_t *)x, (const uint16_t *)dr, work, n0, n1, n2};
    hipLaunchKernelGGL(cnn_out_wgrad, dim3(blocks), dim3(WG_THREADS), OW_LDS, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pvd_hip_error(e, "launch output weight gradient");
    hipLaunchKernelGGL(reduce_rows, dim3(27), dim3(RED_COLS * RED_GROUPS), 0, st, (const float *)work, blocks, 27 * 32, dw,
                       0, 32 * 32);
    e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch reduction");
}

size_t pvd_cnn_out_grad_parts(int n0, int n1, int n2) {
    if (n0 < 1 || n1 < 1 || n2 < 32) return 0;
    MarchArgs q{};
    out_grad_plan(&q, n0, n1, n2);
    return (size_t)q.nby * q.nbz * q.nseg;
}

int pvd_cnn_out_grad(const void *dr, const void *w, float *dh_out, const unsigned *mask, void *dz_out, float *dbias_part,
                     int n0, int n1, int n2, void *stream) {
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!dr || !w || !dh_out || !mask || !dz_out || !dbias_part) return pvd_set_error(PVD_EINVAL, "null argument");
    if ((reinterpret_cast<uintptr_t>(dz_out) | reinterpret_cast<uintptr_t>(dh_out)) & 15)
        return pvd_set_error(PVD_EINVAL, "dz_out and dh_out must be 16-byte aligned");
    MarchArgs q{};
    q.c = ConvArgs{(const uint16_t *)dr, (const uint16_t *)w, nullptr, nullptr, (uint16_t *)dz_out, nullptr, nullptr, n0,
                   n1, n2, nullptr, nullptr, const_cast<unsigned *>(mask)};
    q.dh_out = dh_out;
    q.part = dbias_part;
    out_grad_plan(&q, n0, n1, n2);
    const long long grid = ((long long)q.nby * q.nbz * q.nseg + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return pvd_set_error(PVD_ENOTSUP, "grid too large");
    hipLaunchKernelGGL(cnn_out_grad, dim3((unsigned)grid), dim3(FWD_THREADS), OG_LDS, (hipStream_t)stream, q);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch output layer gradient");
}

int pvd_cnn_adam(float *param, const float *grad, float *m, float *v, void *param_bf16, long long n, float lr,
                 float beta1, float beta2, float eps, int step, void *stream) {
    if (!param || !grad || !m || !v || n < 1 || step < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    const float c1 = 1.0f / (1.0f - powf(beta1, (float)step));
    const float c2 = 1.0f / (1.0f - powf(beta2, (float)step));
    long long blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(cnn_adam, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, param, grad, m, v,
                       (uint16_t *)param_bf16, n, lr, beta1, beta2, eps, c1, c2);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch Adam");
}

int pvd_cnn_pack_inputs(const float *activity, const float *density, const float *dose_plain, const float *act_max,
                        const float *dose_max, void *x, long long n, void *stream) {
    if (!activity || !density || !dose_plain || !act_max || !dose_max || !x || n < 1)
        return pvd_set_error(PVD_EINVAL, "bad argument");
    long long blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(cnn_pack, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, activity, density,
                       dose_plain, act_max, dose_max, (uint16_t *)x, n);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch input packing");
}

int pvd_cnn_apply_correction(const float *dp, const float *r, float bound, const float *dose_max, float region_frac,
                             float apply_frac, float *out, unsigned long long *counts, long long n, void *stream) {
    if (!dp || !r || !dose_max || !out || !counts || n < 1 || !(bound >= 0.0f) || !(region_frac >= 0.0f) ||
        !(apply_frac >= 0.0f))
        return pvd_set_error(PVD_EINVAL, "bad argument");
    // 8 or more voxels per thread: the block's reduction and atomics are paid once per
    // 2048 voxels rather than per 256
    long long blocks = (n + 2047) / 2048;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(cnn_apply, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, dp, r, bound, dose_max,
                       region_frac, apply_frac, out, counts, n);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch correction");
}

int pvd_cnn_input_maxima(const float *activity, const float *dose_plain, long long n, float *maxima, void *stream) {
    if (!activity || !dose_plain || !maxima || n < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    long long blocks = (n + 2047) / 2048;
    if (blocks > MAX2_BLOCKS) blocks = MAX2_BLOCKS;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(cnn_max2_part, dim3((unsigned)blocks), dim3(256), 0, st, activity, dose_plain, n, maxima + 2);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pvd_hip_error(e, "launch input maxima");
    hipLaunchKernelGGL(cnn_max2_final, dim3(1), dim3(256), 0, st, (const float *)(maxima + 2), (int)blocks, maxima);
    e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch input maxima");
}

int pvd_cnn_apply_fallback(const float *dp, const unsigned long long *counts, double max_exceed_frac, float *out,
                           long long n, void *stream) {
    if (!dp || !counts || !out || n < 1 || !(max_exceed_frac >= 0.0))
        return pvd_set_error(PVD_EINVAL, "bad argument");
    long long blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;     // blocks that only read the counts, most often
    hipLaunchKernelGGL(cnn_fallback, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, dp, counts,
                       max_exceed_frac, out, n);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch fallback");
}

int pvd_cnn_region_blocks(const float *dp, int n0, int n1, int n2, const float *dose_max, float frac, int *flags,
                          int *blocks, int *nblocks, void *stream) {
    if (int rc = check_grid(n0, n1, n2)) return rc;
    if (!dp || !dose_max || !flags || !blocks || !nblocks || !(frac >= 0.0f))
        return pvd_set_error(PVD_EINVAL, "bad argument");
    const int nbx = (n0 + FWD_BX - 1) / FWD_BX, nby = (n1 + FWD_BY - 1) / FWD_BY, nbz = n2 >> 5;
    const long long total = (long long)nbx * nby * nbz;
    if (total > 0x7fffffffLL) return pvd_set_error(PVD_ENOTSUP, "too many blocks");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(cnn_block_flags, dim3((unsigned)total), dim3(256), 0, st, dp, n0, n1, n2, dose_max, frac, flags,
                       nblocks);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pvd_hip_error(e, "launch region flags");
    const unsigned g = (unsigned)std::min<long long>((total + 255) / 256, 1024);
    hipLaunchKernelGGL(cnn_block_list, dim3(g), dim3(256), 0, st, (const int *)flags, nbx, nby, nbz, blocks, nblocks);
    e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch region list");
}

size_t pvd_cnn_region_block_count(int n0, int n1, int n2) {
    if (n0 < 1 || n1 < 1 || n2 < 32) return 0;
    return (size_t)((n0 + FWD_BX - 1) / FWD_BX) * ((n1 + FWD_BY - 1) / FWD_BY) * (n2 >> 5);
}

int pvd_reduce_rows(const float *part, int rows, int cols, float *out, int accumulate, void *stream) {
    if (!part || !out || rows < 1 || cols < 1) return pvd_set_error(PVD_EINVAL, "bad argument");
    hipLaunchKernelGGL(reduce_rows, dim3(std::min((cols - 1) / RED_COLS + 1, RED_GRID)), dim3(RED_COLS * RED_GROUPS), 0,
                       (hipStream_t)stream, part, rows, cols, out, accumulate, RED_COLS);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch reduction");
}

}  // extern "C"
