// FFT dose-convolution passes of small volumes: the z and y transforms of one x-plane in
// one launch each way.  A plane of a small volume (Ny * Pz/2 complex) fits the LDS of one
// workgroup, so FZ + FY and IY + IZ keep it there: two launches and two round trips of the
// half spectrum through memory less.  A small dose call is bound by the latency of its
// launches, not by bytes or operations: 64^3 35.5 -> 26.3 us (three launches of 9 to 10 us in a
// trace, the five passes 6 to 10 each), 512x64x64 64.3 -> 38.1.  Radix-16 stages are left out:
// with the split or merge they spilled 45-150 VGPRs and cost more than the launches (64^3
// 37.8 then).
//   ZY  load the T weighted maps, z transform of the line pairs, split, y transform, store
//   YZ  load, inverse y transform (roll / fold), merge, inverse z transform, epilogue
// The stages are the Stockham stages of fft_lines (same radices, twiddles and order of the
// sums), over any number of lines rather than a power of two, and the two-for-one pairs
// are the same lines (the z lines of the whole volume in order: with an odd Ny a pair
// straddles two planes, and a workgroup takes both), so the dose has the bits of the
// five-pass form.  The split of the two-for-one spectra is the load of the first y
// stage, the merge the load of the first inverse z stage, and the outermost y stages read
// and write the workspace directly.
#include "pvd_fft_dev.h"

namespace {

enum { kSrcLds = 0, kSrcSplit = 1, kSrcWork = 2, kSrcMerge = 3 };

struct plane_ctx {
    float2 *s;            // the planes: z lines at [k * ldz + pair], y lines at [y * ldy + plane * H + kz]
    float2 *g;            // the first x-plane in the workspace
    int Ny, Py, Pz, H, Hp;
    int nreal;            // real lines of the planes (one plane less at an odd end)
    int ldz, ldy;
    int offy;
    uint32_t gstep;       // bytes from the first plane to the second
};

// Spectrum of the even (first) or odd line of a pair.  Its products stay products: fused
// into the sums of the stage that takes them, those would round differently than after
// the workspace of the five-pass form.
__device__ __forceinline__ float2 split_pair(float2 zk, float2 zm, bool odd) {
#pragma clang fp contract(off)
    return odd ? make_float2(0.5f * (zk.y + zm.y), 0.5f * (zm.x - zk.x))
               : make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
}

// byte offset in the workspace of row y of column l (a missing second plane: the first's)
template <int G>
__device__ __forceinline__ uint32_t plane_offset(const plane_ctx &c, int y, int l) {
    const bool g = G == 2 && l >= c.H;
    return (uint32_t)(y * c.Hp + l - (g ? c.H : 0)) * 8u + (g && c.nreal > c.Ny ? c.gstep : 0u);
}

// output line of the planes, after the inverse y transform: its row of kz columns
template <int G>
__device__ __forceinline__ const float2 *line_row(const plane_ctx &c, int line) {
    const bool g = G == 2 && line >= c.Ny;
    return c.s + wrap_add(line - (g ? c.Ny : 0), c.offy, c.Py) * c.ldy + (g ? c.H : 0);
}

// One Stockham stage of radix R over `lines` lines (see stockham_stage).  `src` says where
// its inputs come from, `out` that its results go to the workspace (forward y only).
// Every input is in registers before the first result is written, so a stage may change
// the layout of the plane.
template <int R, bool INV, int G>
__device__ __forceinline__ void plane_stage(const plane_ctx &c, int src, bool out, int ld, int lines, int n, int Ns,
                                            const float2 *__restrict__ tw) {
    constexpr int IT = (PVD_PLANE_PER + R - 1) / R;
    const int m = n / R;
    const int work = m * lines;
    const int tstride = n / (Ns * R);
    const float inv_ns = 1.0f / (float)Ns, inv_l = 1.0f / (float)lines;
    float2 *s = c.s;
    float2 v[IT][R];
    int dst[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int w = threadIdx.x + it * blockDim.x;
        dst[it] = -1;
        if (w < work) {
            const int j = fast_div(w, lines, inv_l);
            const int l = w - j * lines;
            const int q = fast_div(j, Ns, inv_ns);
            const int k = j - q * Ns;
            if (!INV && src == kSrcSplit) {
                // spectrum of real line y from its pair's: (Z_l + conj Z_-l)/2 or /(2i)
                const int g = G == 2 && l >= c.H, kz = l - (g ? c.H : 0), km = kz ? c.Pz - kz : 0;
                const int y0 = g ? c.Ny : 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int y = j + r * m;
                    const int line = y0 + min(y, c.Ny - 1);
                    const float2 zk = s[kz * c.ldz + (line >> 1)], zm = s[km * c.ldz + (line >> 1)];
                    v[it][r] = y < c.Ny ? split_pair(zk, zm, line & 1) : make_float2(0.f, 0.f);
                }
            } else if (INV && src == kSrcWork) {
                const uint32_t o = plane_offset<G>(c, j, l), step = (uint32_t)(m * c.Hp) * 8u;
#pragma unroll
                for (int r = 0; r < R; ++r) v[it][r] = at((const float2 *)c.g, o + r * step);
            } else if (INV && src == kSrcMerge) {
                // Z_k = A_k + i B_k, and the conjugates' mirror, of output lines 2l and 2l + 1
                const bool h1 = 2 * l + 1 < c.nreal;
                const float2 *pa = line_row<G>(c, 2 * l), *pb = line_row<G>(c, h1 ? 2 * l + 1 : 2 * l);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int kk = j + r * m, h = kk < c.H ? kk : c.Pz - kk;
                    const float2 A = pa[h], B = h1 ? pb[h] : make_float2(0.f, 0.f);
                    v[it][r] = kk < c.H ? make_float2(A.x - B.y, A.y + B.x) : make_float2(A.x + B.y, B.x - A.y);
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) v[it][r] = s[(j + r * m) * ld + l];
            }
            if (k != 0) {
                const int t = k * tstride;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    float2 wv = tw[r * t];
                    if (INV) wv.y = -wv.y;
                    v[it][r] = cmul(v[it][r], wv);
                }
            }
            Dft<R, INV>::run(v[it]);
            if (!INV && out) {
                const uint32_t o = plane_offset<G>(c, q * Ns * R + k, l), step = (uint32_t)(Ns * c.Hp) * 8u;
                if (G == 1 || l < c.H || c.nreal > c.Ny) {
#pragma unroll
                    for (int r = 0; r < R; ++r) at(c.g, o + r * step) = v[it][r];
                }
            } else {
                dst[it] = (q * Ns * R + k) * ld + l;
            }
        }
    }
    if (!INV && out) return;
    lds_barrier();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        if (dst[it] >= 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) s[dst[it] + r * Ns * ld] = v[it][r];
        }
    }
    lds_barrier();
}

template <bool INV, int G>
__device__ __forceinline__ void plane_fft(const plane_ctx &c, const pvd_axis_d &ax, int first, bool out, int ld,
                                          int lines, const float2 *tw) {
    int Ns = 1;
    for (int st = 0; st < ax.nst; ++st) {
        const int R = ax.radix[st];
        const int src = st == 0 ? first : kSrcLds;
        const bool o = out && st == ax.nst - 1;
        switch (R) {
            case 8: plane_stage<8, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            case 4: plane_stage<4, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            case 2: plane_stage<2, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            case 3: plane_stage<3, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            case 5: plane_stage<5, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            case 7: plane_stage<7, INV, G>(c, src, o, ld, lines, ax.n, Ns, tw); break;
            default: break;
        }
        Ns *= R;
    }
}

template <int G>
__device__ __forceinline__ plane_ctx plane_context(const pvd_vol_d &v, float2 *s) {
    plane_ctx c;
    const int x = blockIdx.x * G;
    c.s = s;
    c.g = v.work + (long long)x * v.wplane;
    c.gstep = (uint32_t)v.wplane * 8u;
    c.Ny = v.ax[1].N; c.Py = v.ax[1].n; c.Pz = v.ax[2].n;
    c.H = v.H; c.Hp = v.Hp;
    c.nreal = min(G, v.ax[0].N - x) * c.Ny;
    c.ldz = pvd_plane_ldz(c.Ny, G);
    c.ldy = pvd_plane_ldy(c.H, G);
    c.offy = v.ax[1].off;
    return c;
}

constexpr int kPlB = 4;        // elements per line in flight per thread

// log2 of the threads per line pair of the loads and the epilogue: one round of kPlB elements a
// thread, a wave at most.  (32 for every length left most of them idle on short lines and took
// long ones round after round: 15x115x12, T = 3 44.5 -> 29.0 us, 295x22x527 96.0 -> 90.1, 817
// volumes 2.4 % on average; a volume of a few hundred voxels pays 0.4 us.)
__device__ __forceinline__ int pair_threads(int len) {
    return len <= 16 ? 2 : len <= 32 ? 3 : len <= 64 ? 4 : len <= 128 ? 5 : 6;
}

template <int G>
__global__ __launch_bounds__(1024) void pvd_fft_plane_zy(pvd_vol_d v) {
    extern __shared__ float2 smem[];
    const pvd_axis_d &ay = v.ax[1], &az = v.ax[2];
    float2 *twz = smem, *twy = twz + ((az.n + 7) & ~7), *s = twy + ((ay.n + 7) & ~7);
    const plane_ctx c = plane_context<G>(v, s);
    const int Nz = az.N, npair = (c.nreal + 1) >> 1;
    load_twiddles(twz, az);
    load_twiddles(twy, ay);
    const long long p0 = (long long)blockIdx.x * G * c.Ny * Nz;        // the first plane's first voxel
    const int ltp = pair_threads(c.Pz), tp = 1 << ltp;
    for (int w = threadIdx.x; w < npair << ltp; w += blockDim.x) {
        const int q = w >> ltp, t = w & (tp - 1);
        const bool h1 = 2 * q + 1 < c.nreal;
        const uint32_t o0 = (uint32_t)(2 * q * Nz);
        for (int z0 = t; z0 < c.Pz; z0 += tp * kPlB) {
            float2 a[kPlB];
            for (int tt = 0; tt < v.T; ++tt) {
                const float *m = v.act[tt] + p0;
                const float wt = v.w[tt];
                float xa[kPlB], xb[kPlB];                            // issued together, masked afterwards
#pragma unroll
                for (int u = 0; u < kPlB; ++u) {
                    const int z = z0 + tp * u;
                    xa[u] = at(m, (z < Nz ? o0 + z : 0u) * 4u);
                    xb[u] = at(m, ((z < Nz && h1) ? o0 + Nz + z : 0u) * 4u);
                }
#pragma unroll
                for (int u = 0; u < kPlB; ++u) {
                    a[u].x = tt ? fmaf(wt, xa[u], a[u].x) : wt * xa[u];
                    a[u].y = tt ? fmaf(wt, xb[u], a[u].y) : wt * xb[u];
                }
            }
#pragma unroll
            for (int u = 0; u < kPlB; ++u) {
                const int z = z0 + tp * u;
                if (z < c.Pz) s[z * c.ldz + q] = make_float2(z < Nz ? a[u].x : 0.f, z < Nz && h1 ? a[u].y : 0.f);
            }
        }
    }
    lds_barrier();
    plane_fft<false, G>(c, az, kSrcLds, false, c.ldz, npair, twz);
    plane_fft<false, G>(c, ay, kSrcSplit, true, c.ldy, G * c.H, twy);
}

template <int G>
__global__ __launch_bounds__(1024) void pvd_fft_plane_yz(pvd_vol_d v) {
    extern __shared__ float2 smem[];
    const pvd_axis_d &ay = v.ax[1], &az = v.ax[2];
    float2 *twz = smem, *twy = twz + ((az.n + 7) & ~7), *s = twy + ((ay.n + 7) & ~7);
    const plane_ctx c = plane_context<G>(v, s);
    const int Nz = az.N, npair = (c.nreal + 1) >> 1;
    load_twiddles(twz, az);
    load_twiddles(twy, ay);
    lds_barrier();
    plane_fft<true, G>(c, ay, kSrcWork, false, c.ldy, G * c.H, twy);
    if (ay.foldn) {        // reference-mode wrap of y: output o < foldn also takes index o + Ny
        for (int w = threadIdx.x; w < ay.foldn * G * c.H; w += blockDim.x) {
            const int o = w / (G * c.H), l = w - o * G * c.H;
            float2 *d = s + wrap_add(o, ay.off, c.Py) * c.ldy + l;
            const float2 f = s[((o + c.Ny + ay.off) % c.Py) * c.ldy + l];
            *d = make_float2(d->x + f.x, d->y + f.y);
        }
        lds_barrier();
    }
    plane_fft<true, G>(c, az, kSrcMerge, false, c.ldz, npair, twz);
    const long long p0 = (long long)blockIdx.x * G * c.Ny * Nz;
    const bool has_dens = v.dens != nullptr;
    const float sc = v.scale;
    const int ltp = pair_threads(Nz), tp = 1 << ltp;
    for (int w = threadIdx.x; w < npair << ltp; w += blockDim.x) {
        const int q = w >> ltp, t = w & (tp - 1);
        const bool h1 = 2 * q + 1 < c.nreal;
        const long long o0 = p0 + 2LL * q * Nz;
        for (int z0 = t; z0 < Nz; z0 += tp * kPlB) {
            float2 d[kPlB];
#pragma unroll
            for (int u = 0; u < kPlB; ++u) {
                const int o = z0 + tp * u;
                d[u].x = (has_dens && o < Nz) ? gmem(v.dens)[o0 + o] : 1.f;
                d[u].y = (has_dens && o < Nz && h1) ? gmem(v.dens)[o0 + Nz + o] : 1.f;
            }
#pragma unroll
            for (int u = 0; u < kPlB; ++u) {
                const int o = z0 + tp * u;
                if (o >= Nz) continue;
                float2 val = s[wrap_add(o, az.off, c.Pz) * c.ldz + q];
                if (o < az.foldn) {
                    const float2 f = s[((o + Nz + az.off) % c.Pz) * c.ldz + q];
                    val.x += f.x;
                    val.y += f.y;
                }
                float f0 = sc, f1 = sc;
                if (has_dens) {
                    f0 *= density_factor(d[u].x);
                    f1 *= density_factor(d[u].y);
                }
                gmem(v.out)[o0 + o] = val.x * f0;
                if (h1) gmem(v.out)[o0 + Nz + o] = val.y * f1;
            }
        }
    }
}

}  // namespace

hipError_t pvd_launch_fft_plane(bool inverse, const pvd_vol_d &v, int grid, int block, size_t lds, hipStream_t st) {
    if (v.ax[1].N % 2 == 0) {
        if (inverse) hipLaunchKernelGGL(pvd_fft_plane_yz<1>, dim3(grid), dim3(block), lds, st, v);
        else hipLaunchKernelGGL(pvd_fft_plane_zy<1>, dim3(grid), dim3(block), lds, st, v);
    } else {
        if (inverse) hipLaunchKernelGGL(pvd_fft_plane_yz<2>, dim3(grid), dim3(block), lds, st, v);
        else hipLaunchKernelGGL(pvd_fft_plane_zy<2>, dim3(grid), dim3(block), lds, st, v);
    }
    return hipGetLastError();
}

hipError_t pvd_fft_plane_set_lds(size_t bytes) {
    hipError_t e = hipSuccess;
#define PVD_SETATTR(K) \
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)K, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes)
    PVD_SETATTR(pvd_fft_plane_zy<1>);
    PVD_SETATTR(pvd_fft_plane_zy<2>);
    PVD_SETATTR(pvd_fft_plane_yz<1>);
    PVD_SETATTR(pvd_fft_plane_yz<2>);
#undef PVD_SETATTR
    return e;
}
