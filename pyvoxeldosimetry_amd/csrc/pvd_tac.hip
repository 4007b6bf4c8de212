// Voxelwise time-activity-curve fits: one thread per voxel, FP64
// Levenberg-Marquardt with analytic Jacobians (the reference runs
// scipy.optimize.curve_fit voxel by voxel, time_integration/curve_fitting.py).
// The normal equations are accumulated on the fly (no Jacobian storage).  The kernel is
// compiled per model and per sample count (4, 8 or 16 at most), so that every loop is
// unrolled and nothing is indexed at run time; a thread holds the samples, the system and
// the parameters in registers, except the four- and five-parameter models with 9 to 16
// samples, which spill (388 to 1236 bytes a lane, one wave per SIMD).  Bound by the FP64
// vector instructions (256x256x200 voxels, mono-exponential, 4 samples: 1995 -> 585 us,
// about 1700 instructions a voxel; with one run-time-indexed kernel for all models, each
// trial point evaluated twice and seven divisions a step before; NUKFIT f2 15.7 -> 4.7 ms,
// f3a at 100^3 141 -> 82 us).  The larger models at 48^3, us, run-time-indexed -> now: f4a 6
// samples 3772 -> 2586, 12 samples 5186 -> 3756, 16 samples 6786 -> 4637; f4b 5628 -> 3367
// at 8, 7041 -> 4539 at 16; tri-exponential 5781 -> 3568 at 8, 10528 -> 6813 at 16.
#include "pvd_internal.h"
#include "../../include/pvd_tac.h"

#include <cmath>

namespace {

constexpr double kLn2 = 0.69314718055994530942;

struct TacArgs {
    const float *m[PVD_TAC_MAX_T];
    pvd_tac_params p;
    long long n;
    float *params;
    float *auc;
    unsigned char *status;
};

int n_params_of(int model) {
    switch (model) {
        case PVD_TAC_MONO: case PVD_TAC_NUKFIT_F2: case PVD_TAC_LMFIT_MONO: return 2;
        case PVD_TAC_NUKFIT_F3: case PVD_TAC_NUKFIT_F3A: case PVD_TAC_LMFIT_BI: return 3;
        case PVD_TAC_NUKFIT_F4A: return 4;
        case PVD_TAC_NUKFIT_F4B: case PVD_TAC_NUKFIT_F4C: case PVD_TAC_LMFIT_TRI: return 5;
        default: return -1;
    }
}

// f(t; p) and, when g != nullptr, df/dp (the expressions of curve_fitting.py:136-170)
template <int MODEL>
__device__ __forceinline__ double model_eval(const double *p, double t, double lp, double *g) {
    switch (MODEL) {
        case PVD_TAC_MONO: {
            const double e = exp(-p[1] * t);
            if (g) { g[0] = e; g[1] = -t * p[0] * e; }
            return p[0] * e;
        }
        case PVD_TAC_NUKFIT_F2: {
            const double e = exp(-(p[1] + lp) * t);
            if (g) { g[0] = e; g[1] = -t * p[0] * e; }
            return p[0] * e;
        }
        case PVD_TAC_NUKFIT_F3: {
            const double e1 = exp(-(p[1] + lp) * t), e2 = exp(-(p[2] + lp) * t);
            if (g) { g[0] = e1 - e2; g[1] = -t * p[0] * e1; g[2] = t * p[0] * e2; }
            return p[0] * (e1 - e2);
        }
        case PVD_TAC_NUKFIT_F3A: {
            const double e1 = exp(-(p[2] + lp) * t), ep = exp(-lp * t);
            const double s = p[1] * e1 + (1.0 - p[1]) * ep;
            if (g) { g[0] = s; g[1] = p[0] * (e1 - ep); g[2] = -t * p[0] * p[1] * e1; }
            return p[0] * s;
        }
        case PVD_TAC_NUKFIT_F4A: {
            const double e1 = exp(-(p[1] + lp) * t), e2 = exp(-(p[3] + lp) * t);
            if (g) { g[0] = e1; g[1] = -t * p[0] * e1; g[2] = e2; g[3] = -t * p[2] * e2; }
            return p[0] * e1 + p[2] * e2;
        }
        case PVD_TAC_NUKFIT_F4B: {
            const double e1 = exp(-(p[1] + lp) * t), e2 = exp(-(p[3] + lp) * t), eb = exp(-(p[4] + lp) * t);
            if (g) {
                g[0] = e1 - eb; g[1] = -t * p[0] * e1; g[2] = eb - e2; g[3] = t * p[2] * e2;
                g[4] = t * (p[0] - p[2]) * eb;
            }
            return p[0] * e1 - p[2] * e2 - (p[0] - p[2]) * eb;
        }
        case PVD_TAC_NUKFIT_F4C: {
            const double e1 = exp(-(p[1] + lp) * t), e2 = exp(-(p[3] + lp) * t), eb = exp(-(p[4] + lp) * t);
            if (g) {
                g[0] = e1 - eb; g[1] = -t * p[0] * e1; g[2] = e2 - eb; g[3] = -t * p[2] * e2;
                g[4] = t * (p[0] + p[2]) * eb;
            }
            return p[0] * e1 + p[2] * e2 - (p[0] + p[2]) * eb;
        }
        case PVD_TAC_LMFIT_MONO: {
            const double e = exp(-kLn2 * t / p[1]);
            if (g) { g[0] = e; g[1] = p[0] * e * kLn2 * t / (p[1] * p[1]); }
            return p[0] * e;
        }
        case PVD_TAC_LMFIT_BI: {
            const double e1 = exp(-kLn2 * t / p[1]), e2 = exp(-kLn2 * t / p[2]);
            if (g) {
                g[0] = e1 - e2; g[1] = p[0] * e1 * kLn2 * t / (p[1] * p[1]);
                g[2] = -p[0] * e2 * kLn2 * t / (p[2] * p[2]);
            }
            return p[0] * (e1 - e2);
        }
        default: {   // PVD_TAC_LMFIT_TRI
            const double e1 = exp(-kLn2 * t / p[1]), e2 = exp(-kLn2 * t / p[3]), ep = exp(-kLn2 * t / p[4]);
            if (g) {
                g[0] = e1 - ep; g[1] = p[0] * e1 * kLn2 * t / (p[1] * p[1]); g[2] = ep - e2;
                g[3] = -p[2] * e2 * kLn2 * t / (p[3] * p[3]); g[4] = -(p[0] - p[2]) * ep * kLn2 * t / (p[4] * p[4]);
            }
            return p[0] * e1 - p[2] * e2 - (p[0] - p[2]) * ep;
        }
    }
}

template <int MODEL> constexpr int kNp = 0;
template <> constexpr int kNp<PVD_TAC_MONO> = 2;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F2> = 2;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F3> = 3;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F3A> = 3;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F4A> = 4;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F4B> = 5;
template <> constexpr int kNp<PVD_TAC_NUKFIT_F4C> = 5;
template <> constexpr int kNp<PVD_TAC_LMFIT_MONO> = 2;
template <> constexpr int kNp<PVD_TAC_LMFIT_BI> = 3;
template <> constexpr int kNp<PVD_TAC_LMFIT_TRI> = 5;

// weighted cost sum_i (w_i (y_i - f_i))^2, and A = J^T J (lower triangle), b = J^T e
template <int MODEL, int NT>
__device__ __forceinline__ double accumulate(const TacArgs &a, const double *y, const double *p,
                                             double (*A)[kNp<MODEL>], double *b) {
    constexpr int NP = kNp<MODEL>;
    const pvd_tac_params &q = a.p;
    double cost = 0.0;
#pragma unroll
    for (int r = 0; r < NP; ++r) {
        b[r] = 0.0;
#pragma unroll
        for (int c = 0; c <= r; ++c) A[r][c] = 0.0;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if (i >= q.n_times) continue;          // uniform
        double g[PVD_TAC_MAX_P];
        const double f = model_eval<MODEL>(p, q.t[i], q.lambda_phys, g);
        const double e = q.w[i] * (y[i] - f);
        cost += e * e;
#pragma unroll
        for (int r = 0; r < NP; ++r) {
            const double jr = q.w[i] * g[r];
            b[r] += jr * e;
#pragma unroll
            for (int c = 0; c <= r; ++c) A[r][c] += jr * q.w[i] * g[c];
        }
    }
    return cost;
}

// solve (A + mu diag(d2)) x = b by Cholesky; false if not positive definite.  Two
// parameters take L D L^T (two reciprocals instead of two square roots and seven
// divisions); the models with more are degenerate enough that another rounding of the
// step can end in another minimum, so they keep the textbook form.
template <int NP>
__device__ __forceinline__ bool damped_solve(const double (*A)[NP], const double *b, const double *d2, double mu,
                                             double *x) {
    if constexpr (NP > 2) {
        double L[NP][NP], z[NP];
        bool ok = true;
#pragma unroll
        for (int r = 0; r < NP; ++r) {
#pragma unroll
            for (int c = 0; c <= r; ++c) {
                double s = A[r][c];
                if (r == c) s += mu * d2[r];
#pragma unroll
                for (int k = 0; k < c; ++k) s -= L[r][k] * L[c][k];
                if (r == c) {
                    ok = ok && s > 0.0;
                    L[r][r] = sqrt(s);
                } else {
                    L[r][c] = s / L[c][c];
                }
            }
        }
        if (!ok) return false;
#pragma unroll
        for (int r = 0; r < NP; ++r) {
            double s = b[r];
#pragma unroll
            for (int k = 0; k < r; ++k) s -= L[r][k] * z[k];
            z[r] = s / L[r][r];
        }
#pragma unroll
        for (int r = NP - 1; r >= 0; --r) {
            double s = z[r];
#pragma unroll
            for (int k = r + 1; k < NP; ++k) s -= L[k][r] * x[k];
            x[r] = s / L[r][r];
        }
        return true;
    }
    double L[NP][NP], d[NP], inv[NP], z[NP];
    bool ok = true;
#pragma unroll
    for (int r = 0; r < NP; ++r) {
#pragma unroll
        for (int c = 0; c < r; ++c) {
            double s = A[r][c];
#pragma unroll
            for (int k = 0; k < c; ++k) s -= L[r][k] * d[k] * L[c][k];
            L[r][c] = s * inv[c];
        }
        double s = A[r][r] + mu * d2[r];
#pragma unroll
        for (int k = 0; k < r; ++k) s -= L[r][k] * L[r][k] * d[k];
        ok = ok && s > 0.0;
        d[r] = s;
        inv[r] = 1.0 / s;
    }
    if (!ok) return false;
#pragma unroll
    for (int r = 0; r < NP; ++r) {
        double s = b[r];
#pragma unroll
        for (int k = 0; k < r; ++k) s -= L[r][k] * z[k];
        z[r] = s;
    }
#pragma unroll
    for (int r = NP - 1; r >= 0; --r) {
        double s = z[r] * inv[r];
#pragma unroll
        for (int k = r + 1; k < NP; ++k) s -= L[k][r] * x[k];
        x[r] = s;
    }
    return true;
}

// Levenberg-Marquardt with MINPACK-style scaling: the damping term is
// mu * diag(D^2), D_j the largest Jacobian column norm seen so far, which keeps
// the step scale-invariant and stops the damping from collapsing in directions
// whose curvature vanishes along the path (degenerate valleys of the
// multi-exponential models).  A trial point is evaluated with its Jacobian at once: most
// are accepted, and the exponentials would otherwise be taken twice.
template <int MODEL, int NT>
__device__ __forceinline__ bool lm(const TacArgs &a, const double *y, double *p) {
    constexpr int NP = kNp<MODEL>;
    const double tol = a.p.tol;
    double A[NP][NP], b[NP], d2[NP];
    double cost = accumulate<MODEL, NT>(a, y, p, A, b);
    if (!isfinite(cost)) return false;
#pragma unroll
    for (int k = 0; k < NP; ++k) d2[k] = fmax(A[k][k], 1e-300);
    double mu = 1e-3;
    for (int it = 0; it < a.p.max_iter; ++it) {
        if (cost == 0.0) return true;
#pragma unroll
        for (int k = 0; k < NP; ++k) d2[k] = fmax(d2[k], A[k][k]);
        bool stepped = false;
        for (int attempt = 0; attempt < 60; ++attempt) {
            double d[NP], pn[NP];
            if (damped_solve<NP>(A, b, d2, mu, d)) {
                double An[NP][NP], bn[NP];
#pragma unroll
                for (int k = 0; k < NP; ++k) pn[k] = p[k] + d[k];
                const double cn = accumulate<MODEL, NT>(a, y, pn, An, bn);
                if (isfinite(cn) && cn <= cost) {
                    bool small = true;
#pragma unroll
                    for (int k = 0; k < NP; ++k) small = small && fabs(d[k]) <= tol * (fabs(pn[k]) + tol);
                    const bool flat = (cost - cn) <= tol * cost;
#pragma unroll
                    for (int k = 0; k < NP; ++k) {
                        p[k] = pn[k];
                        b[k] = bn[k];
#pragma unroll
                        for (int c = 0; c <= k; ++c) A[k][c] = An[k][c];
                    }
                    cost = cn;
                    if (small || flat) return true;
                    mu = fmax(mu * 0.3, 1e-15);
                    stepped = true;
                    break;
                }
            }
            mu *= 10.0;
            if (mu > 1e20) return true;      // no descent direction left: at a minimum
        }
        if (!stepped) return true;
    }
    return false;
}

template <int MODEL, int NT>
__global__ __launch_bounds__(256) void tac_fit_kernel(TacArgs a) {
    constexpr int NP = kNp<MODEL>;
    const pvd_tac_params &q = a.p;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < a.n; v += (long long)gridDim.x * 256) {
        double y[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) y[i] = i < q.n_times ? (double)a.m[i][v] : 0.0;
        double p[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) p[k] = q.p0[k];
        if (MODEL == PVD_TAC_MONO && q.p0_from_data) p[0] = y[0];
        if (q.force_zero_at_t0) {
            const double y0 = y[0];
#pragma unroll
            for (int i = 0; i < NT; ++i) y[i] -= y0;
            y[0] = 0.0;
        }
        bool ok = false;
        if constexpr (NP <= NT) {                  // (else n_times <= NT < NP: no form can fit)
            if (NP <= q.n_times) ok = lm<MODEL, NT>(a, y, p);
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) ok = ok && isfinite(p[k]);
        if (!ok) {
#pragma unroll
            for (int k = 0; k < NP; ++k) p[k] = q.fail_params[k];
        }
        double s;
        if (q.auc_mode == PVD_TAC_AUC_MONO_TAIL && NP == 2) {
            s = p[0] / p[1] * (1.0 - exp(-p[1] * q.t_int));
        } else {
            s = 0.0;
            double f0 = model_eval<MODEL>(p, q.t[0], q.lambda_phys, nullptr);
#pragma unroll
            for (int i = 1; i < NT; ++i) {
                if (i >= q.n_times) continue;
                const double f1 = model_eval<MODEL>(p, q.t[i], q.lambda_phys, nullptr);
                s += (q.t[i] - q.t[i - 1]) * (f1 + f0) * 0.5;
                f0 = f1;
            }
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) a.params[k * a.n + v] = (float)p[k];
        if (a.auc) a.auc[v] = (float)s;
        if (a.status) a.status[v] = ok ? 1 : 0;
    }
}

template <int MODEL>
void launch_model(const TacArgs &a, unsigned grid, hipStream_t st) {
    if (a.p.n_times <= 4) hipLaunchKernelGGL((tac_fit_kernel<MODEL, 4>), dim3(grid), dim3(256), 0, st, a);
    else if (a.p.n_times <= 8) hipLaunchKernelGGL((tac_fit_kernel<MODEL, 8>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((tac_fit_kernel<MODEL, PVD_TAC_MAX_T>), dim3(grid), dim3(256), 0, st, a);
}

}  // namespace

extern "C" int pvd_tac_n_params(int model) {
    const int np = n_params_of(model);
    return np > 0 ? np : pvd_set_error(PVD_EINVAL, "unknown TAC model %d", model);
}

extern "C" int pvd_tac_fit(const pvd_tac_params *p, const float *const *maps, long long n, float *params, float *auc,
                           unsigned char *status, void *stream) {
    if (!p || !maps || !params || n < 1) return pvd_set_error(PVD_EINVAL, "null argument or n < 1");
    const int np = n_params_of(p->model);
    if (np < 0) return pvd_set_error(PVD_EINVAL, "unknown TAC model %d", p->model);
    if (p->n_times < 1 || p->n_times > PVD_TAC_MAX_T)
        return pvd_set_error(PVD_EINVAL, "n_times must be 1..%d", PVD_TAC_MAX_T);
    if (p->max_iter < 1 || !(p->tol > 0.0)) return pvd_set_error(PVD_EINVAL, "max_iter >= 1 and tol > 0 required");
    if (p->auc_mode != PVD_TAC_AUC_MONO_TAIL && p->auc_mode != PVD_TAC_AUC_TRAPEZOID)
        return pvd_set_error(PVD_EINVAL, "unknown auc_mode %d", p->auc_mode);
    if (p->auc_mode == PVD_TAC_AUC_MONO_TAIL && np != 2)
        return pvd_set_error(PVD_EINVAL, "the mono-exponential tail integral needs a 2-parameter model");
    TacArgs a{};
    for (int i = 0; i < p->n_times; ++i) {
        if (!maps[i]) return pvd_set_error(PVD_EINVAL, "null map %d", i);
        a.m[i] = maps[i];
    }
    a.p = *p;
    a.n = n;
    a.params = params;
    a.auc = auc;
    a.status = status;
    long long g = (n + 255) / 256;
    if (g > 16384) g = 16384;
    hipStream_t st = (hipStream_t)stream;
    switch (p->model) {
        case PVD_TAC_MONO: launch_model<PVD_TAC_MONO>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F2: launch_model<PVD_TAC_NUKFIT_F2>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F3: launch_model<PVD_TAC_NUKFIT_F3>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F3A: launch_model<PVD_TAC_NUKFIT_F3A>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F4A: launch_model<PVD_TAC_NUKFIT_F4A>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F4B: launch_model<PVD_TAC_NUKFIT_F4B>(a, (unsigned)g, st); break;
        case PVD_TAC_NUKFIT_F4C: launch_model<PVD_TAC_NUKFIT_F4C>(a, (unsigned)g, st); break;
        case PVD_TAC_LMFIT_MONO: launch_model<PVD_TAC_LMFIT_MONO>(a, (unsigned)g, st); break;
        case PVD_TAC_LMFIT_BI: launch_model<PVD_TAC_LMFIT_BI>(a, (unsigned)g, st); break;
        default: launch_model<PVD_TAC_LMFIT_TRI>(a, (unsigned)g, st); break;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PVD_OK : pvd_hip_error(e, "launch TAC fit");
}
