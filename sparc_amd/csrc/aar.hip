// Alternating Anderson-Richardson (AAR) linear solver on the device, with the
// reference's Poisson residual and Jacobi preconditioner built in
// (SPARC AAR src/linearSolver.c:37-159, AndersonExtrapolation
// src/mixing.c:48-139, poisson_residual src/lapVecRoutines.c:69-79,
// Jacobi_preconditioner src/electrostatics.c:1682-1699).
//
// The last m + 1 iterates x_k and preconditioned residuals f_k are kept as they
// are, in two rings; the history differences that Anderson mixing takes are
// formed where they are used.  With the built-in residual and preconditioner a
// Richardson iteration is then one launch (sgpu_launch_aar_step: the stencil
// with f = jac r and x + omega f in its epilogue; x twice, b, f and the new x
// are 5 vectors moved, against 15 for a residual stencil followed by a pass
// that kept r, x_old, f_old and two difference columns).  Anderson steps add
// one pass for F'F and F'f together and one update pass; the m x m
// minimum-norm solve is done on the host in FP64.
#include <algorithm>
#include <cmath>
#include <vector>

#include "sgpu_internal.h"
#include "wave_sum.h"

namespace {

constexpr int kAarMaxM = 8;

// f = jac r (when jac != 0; otherwise f is given) and, when xn is given,
// xn = x + omega f.
__global__ void aar_step(const double *__restrict__ r, double *__restrict__ f, double jac,
                         const double *__restrict__ x, double *__restrict__ xn, double omega, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double fi = jac != 0.0 ? jac * r[i] : f[i];
    if (jac != 0.0) f[i] = fi;
    if (xn) xn[i] = x[i] + omega * fi;
}

struct AarCoeff {
    double g[kAarMaxM];
};

// The ring vectors v_k, v_(k-1), ... by age.
struct AarRing {
    const double *v[kAarMaxM + 1];
};

// Sums over the block's share of F'F (upper triangle) and F'f into partial,
// from the NV accumulators of every thread.
template <int NV>
__device__ __forceinline__ void gram_partial(const double (&acc)[NV], double *__restrict__ partial)
{
    __shared__ double sh[4][NV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double s = acc[k];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (lane == 0) sh[wave][k] = s;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < NV; k += 256)
        partial[(long)blockIdx.x * NV + k] = sh[0][k] + sh[1][k] + sh[2][k] + sh[3][k];
}

// Recorded solves (training pairs) keep one fixed order of operations, so that
// a network trained on them does not depend on the forms chosen for speed: the
// columns of aar_gram / aar_update_cols are the history differences formed by
// aar_columns, in the order d % m of the steps d they come from.
__global__ void aar_columns(AarRing x, AarRing f, int m, int rot, long ld, double *__restrict__ Xh,
                            double *__restrict__ Fh, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int j = 0; j < m; j++) {
        const long at = (long)((rot + m - j) % m) * ld + i;  // age j
        Xh[at] = x.v[j][i] - x.v[j + 1][i];
        Fh[at] = f.v[j][i] - f.v[j + 1][i];
    }
}

// xn = x - Xh G + beta (f - Fh G)
__global__ void aar_update_cols(double *xn, const double *x, const double *__restrict__ f,
                                const double *__restrict__ Xh, const double *__restrict__ Fh, long ldh,
                                int m, AarCoeff G, double beta, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double xw = x[i], fw = f[i];
#pragma unroll
    for (int a = 0; a < kAarMaxM; a++) {
        if (a < m) {
            xw -= Xh[a * ldh + i] * G.g[a];
            fw -= Fh[a * ldh + i] * G.g[a];
        }
    }
    xn[i] = xw + beta * fw;
}

// The same sums as aar_gram for the columns F_j = f_(k-j) - f_(k-j-1), j < m.
// Bound by reading m + 1 vectors; four workgroups per CU (with one, as
// aar_gram has, too few bytes were in flight: 128^3, m = 7, 44 -> 38 us).  The
// block's sums are taken four at a time with lane swaps (rows4_sum): 38 -> 23 us
// there, 19.6 -> 5.3 us at 52^3, where the 35 butterflies of ds_bpermute were
// most of the launch.
template <int M>
__global__ __launch_bounds__(256) void aar_gram_ring(AarRing f, int m, long n,
                                                     double *__restrict__ partial)
{
    constexpr int NV = M * (M + 1) / 2 + M;
    double acc[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = 0.0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        double v[M + 1];
#pragma unroll
        for (int a = 0; a <= M; a++) v[a] = a <= m ? f.v[a][i] : 0.0;
        const double fi = v[0];
#pragma unroll
        for (int a = 0; a < M; a++) v[a] = a < m ? v[a] - v[a + 1] : 0.0;
        int k = 0;
#pragma unroll
        for (int a = 0; a < M; a++)
#pragma unroll
            for (int b = a; b < M; b++) acc[k++] += v[a] * v[b];
#pragma unroll
        for (int a = 0; a < M; a++) acc[k++] += v[a] * fi;
    }
    __shared__ double sh[4][(NV + 3) / 4 * 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k += 4) {
        const double s = rows4_sum(acc[k], k + 1 < NV ? acc[k + 1] : 0.0, k + 2 < NV ? acc[k + 2] : 0.0,
                                   k + 3 < NV ? acc[k + 3] : 0.0);
        if ((lane & 15) == 0) sh[wave][k + (lane >> 4)] = s;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < NV; k += 256)
        partial[(long)blockIdx.x * NV + k] = sh[0][k] + sh[1][k] + sh[2][k] + sh[3][k];
}

// Partial sums of F'F (upper triangle, m(m+1)/2 values) and F'f (m values).
template <int M>
__global__ __launch_bounds__(256) void aar_gram(const double *__restrict__ F, long ldf,
                                                const double *__restrict__ f, int m, long n,
                                                double *__restrict__ partial)
{
    constexpr int NV = M * (M + 1) / 2 + M;
    double acc[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = 0.0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        double v[M];
#pragma unroll
        for (int a = 0; a < M; a++) v[a] = a < m ? F[a * ldf + i] : 0.0;
        const double fi = f[i];
        int k = 0;
#pragma unroll
        for (int a = 0; a < M; a++)
#pragma unroll
            for (int b = a; b < M; b++) acc[k++] += v[a] * v[b];
#pragma unroll
        for (int a = 0; a < M; a++) acc[k++] += v[a] * fi;
    }
    gram_partial<NV>(acc, partial);
}

// One wave per Gram value: lane l sums the partials l, l + 64, ... in order,
// then a fixed butterfly over the wave (deterministic).
__global__ __launch_bounds__(64) void aar_gram_final(const double *__restrict__ partial, int nblk,
                                                     int nv, double *__restrict__ out)
{
    const int k = blockIdx.x, lane = threadIdx.x;
    double s = 0.0;
    for (int b = lane; b < nblk; b += 64) s += partial[(long)b * nv + k];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) out[k] = s;
}

// xn = x_k - X G + beta (f_k - F G) with F_j = f_(k-j) - f_(k-j-1) and
// X_j = x_(k-j) - x_(k-j-1) where bit j of xdiff is set (step k - j - 1 was an
// Anderson one), omega f_(k-j-1) otherwise (a Richardson step moved x by just
// that), which needs no x vectors.  xn may be the oldest x.
template <int M>
__global__ __launch_bounds__(256) void aar_update(double *xn, AarRing x, AarRing f, int m,
                                                  unsigned xdiff, AarCoeff G, double omega, double beta,
                                                  long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double v[M + 1];
#pragma unroll
    for (int a = 0; a <= M; a++) v[a] = a <= m ? f.v[a][i] : 0.0;
    double xw = x.v[0][i], fw = v[0];
#pragma unroll
    for (int a = 0; a < M; a++) {
        if (a < m) {
            const double d = (xdiff >> a & 1) ? x.v[a][i] - x.v[a + 1][i] : omega * v[a + 1];
            xw -= d * G.g[a];
            fw -= (v[a] - v[a + 1]) * G.g[a];
        }
    }
    xn[i] = xw + beta * fw;
}

// Symmetric eigendecomposition by cyclic Jacobi rotations (m <= 8).
void jacobi_eig(int n, double *A, double *w, double *V)
{
    for (int i = 0; i < n; i++)
        for (int j = 0; j < n; j++) V[i + j * n] = i == j;
    for (int sweep = 0; sweep < 64; sweep++) {
        double off = 0.0, tot = 0.0;
        for (int j = 0; j < n; j++)
            for (int i = 0; i < n; i++) {
                tot += A[i + j * n] * A[i + j * n];
                if (i != j) off += A[i + j * n] * A[i + j * n];
            }
        if (off == 0.0 || off <= 1e-30 * tot) break;
        for (int p = 0; p < n - 1; p++)
            for (int q = p + 1; q < n; q++) {
                const double apq = A[p + q * n];
                if (std::fabs(apq) < 1e-300) continue;
                const double th = (A[q + q * n] - A[p + p * n]) / (2.0 * apq);
                const double t = (th >= 0 ? 1.0 : -1.0) / (std::fabs(th) + std::sqrt(th * th + 1.0));
                const double cs = 1.0 / std::sqrt(t * t + 1.0), sn = t * cs;
                for (int k = 0; k < n; k++) {
                    const double akp = A[k + p * n], akq = A[k + q * n];
                    A[k + p * n] = cs * akp - sn * akq;
                    A[k + q * n] = sn * akp + cs * akq;
                }
                for (int k = 0; k < n; k++) {
                    const double apk = A[p + k * n], aqk = A[q + k * n];
                    A[p + k * n] = cs * apk - sn * aqk;
                    A[q + k * n] = sn * apk + cs * aqk;
                }
                for (int k = 0; k < n; k++) {
                    const double vkp = V[k + p * n], vkq = V[k + q * n];
                    V[k + p * n] = cs * vkp - sn * vkq;
                    V[k + q * n] = sn * vkp + cs * vkq;
                }
            }
    }
    for (int i = 0; i < n; i++) w[i] = A[i + i * n];
}

}  // namespace

// Minimum-norm least-squares solution of (F'F) G = F'f, singular values
// below eps * s_max dropped: the result LAPACKE_dgelsd(rcond = -1) returns in
// AndersonExtrapCoeff (src/mixing.c:135).
void anderson_coeff(int m, const double *FtF, const double *Ftf, double *G)
{
    double A[kAarMaxM * kAarMaxM], V[kAarMaxM * kAarMaxM], w[kAarMaxM];
    for (int i = 0; i < m * m; i++) A[i] = FtF[i];
    jacobi_eig(m, A, w, V);
    double smax = 0.0;
    for (int i = 0; i < m; i++) smax = std::max(smax, std::fabs(w[i]));
    const double thr = 2.220446049250313e-16 * smax;
    for (int i = 0; i < m; i++) G[i] = 0.0;
    for (int k = 0; k < m; k++) {
        if (std::fabs(w[k]) <= thr) continue;
        double proj = 0.0;
        for (int i = 0; i < m; i++) proj += V[i + k * m] * Ftf[i];
        proj /= w[k];
        for (int i = 0; i < m; i++) G[i] += V[i + k * m] * proj;
    }
}

// The unpacked sums of a Gram pass (upper triangle of M x M, then F'f) on the
// host: G = pinv(F'F) F'f for the first m columns.
template <int M>
static void gram_solve(const double *sums, int m, double *G)
{
    double FtF[kAarMaxM * kAarMaxM], Ftf[kAarMaxM];
    int k = 0;
    for (int a = 0; a < M; a++)
        for (int bb = a; bb < M; bb++, k++)
            if (a < m && bb < m) FtF[a + bb * m] = FtF[bb + a * m] = sums[k];
    for (int a = 0; a < M; a++, k++)
        if (a < m) Ftf[a] = sums[k];
    anderson_coeff(m, FtF, Ftf, G);
}

// G = pinv(F'F) F'f for device F (n x m, column stride ldf) and f: one pass
// computes F'F and F'f together, the m x m solve runs on the host in FP64.
int sgpu_anderson_coeff_dev(sgpu_context *ctx, const double *F, long ldf, int m, const double *f,
                            long n, double *G)
{
    if (m < 1 || m > kAarMaxM) {
        sgpu_set_error("anderson: history %d outside 1..%d", m, kAarMaxM);
        return SGPU_ERR_ARG;
    }
    const int gram_blocks = 256;
    const int nv = kAarMaxM * (kAarMaxM + 1) / 2 + kAarMaxM;
    double *partial = nullptr;
    SGPU_CHECK(sgpu_reduce_buf(ctx, (size_t)gram_blocks * nv + nv, &partial));
    double *out = partial + (size_t)gram_blocks * nv;
    aar_gram<kAarMaxM><<<gram_blocks, 256, 0, ctx->stream>>>(F, ldf, f, m, n, partial);
    aar_gram_final<<<nv, 64, 0, ctx->stream>>>(partial, gram_blocks, nv, out);
    SGPU_HIP(hipGetLastError());
    SGPU_HIP(hipMemcpyAsync(ctx->host_red, out, nv * sizeof(double), hipMemcpyDeviceToHost,
                            ctx->stream));
    SGPU_HIP(hipStreamSynchronize(ctx->stream));
    gram_solve<kAarMaxM>(ctx->host_red, m, G);
    return SGPU_OK;
}

// G for the ring's differences (aar_gram_ring).
template <int M>
static int ring_coeff(sgpu_context *ctx, const AarRing &f, int m, long n, double *G)
{
    constexpr int nv = M * (M + 1) / 2 + M;
    const int blocks = (int)std::min<long>((n + 255) / 256, 4L * ctx->n_cu);
    double *partial = nullptr;
    SGPU_CHECK(sgpu_reduce_buf(ctx, (size_t)blocks * nv + nv, &partial));
    double *out = partial + (size_t)blocks * nv;
    aar_gram_ring<M><<<blocks, 256, 0, ctx->stream>>>(f, m, n, partial);
    aar_gram_final<<<nv, 64, 0, ctx->stream>>>(partial, blocks, nv, out);
    SGPU_HIP(hipGetLastError());
    SGPU_HIP(hipMemcpyAsync(ctx->host_red, out, nv * sizeof(double), hipMemcpyDeviceToHost,
                            ctx->stream));
    SGPU_HIP(hipStreamSynchronize(ctx->stream));
    gram_solve<M>(ctx->host_red, m, G);
    return SGPU_OK;
}

// AAR on device vectors x (in/out) and b, both of length N = Nd.
int sgpu_aar_device(sgpu_context *ctx, sgpu_res_fn res, sgpu_precond_fn precond, void *user,
                    double c, int N, double *x, const double *b, double omega, double beta, int m,
                    int p, double tol, int max_iter, int *iters, double *relres,
                    const sgpu_aar_recorder *rec)
{
    if (!ctx || !x || !b || N != ctx->nd || m < 1 || m > kAarMaxM || p < 1 || max_iter < 0) {
        sgpu_set_error("AAR: bad arguments (N %d, Nd %ld, m %d, p %d)", N, ctx ? ctx->nd : 0L, m, p);
        return SGPU_ERR_ARG;
    }
    const long n = N;
    const long ld = ctx->ld;
    // r and the rings of x and f (recorded solves: also their differences):
    // cached on the context
    const bool recording = rec && rec->fn;
    const int S = m + 1;
    const size_t elems = (size_t)(1 + 2 * S + (recording ? 2 * m : 0)) * ld;
    if (elems > ctx->aar_elems) {
        SGPU_HIP(hipStreamSynchronize(ctx->stream));
        if (ctx->aar_mem) SGPU_HIP(hipFree(ctx->aar_mem));
        ctx->aar_mem = nullptr;
        ctx->aar_elems = 0;
        SGPU_HIP(hipMalloc((void **)&ctx->aar_mem, elems * sizeof(double)));
        ctx->aar_elems = elems;
    }
    double *r = ctx->aar_mem;
    auto X = [&](int k) { return ctx->aar_mem + (long)(1 + k % S) * ld; };
    auto F = [&](int k) { return ctx->aar_mem + (long)(1 + S + k % S) * ld; };
    const unsigned nb = (unsigned)((n + 255) / 256);
    const double dsum = ctx->d2x[0] + ctx->d2y[0] + ctx->d2z[0] + c;
    const double jac = -1.0 / (std::fabs(dsum) < 1e-14 ? 1.0 : dsum);
    auto anderson = [&](int k) { return k > 0 && (k + 1) % p == 0; };
    // the step in one launch needs no r of its own
    bool fused = !res && !precond && !recording;

    // r_k, and when fused f_k and (Richardson steps) x_(k+1) with it
    auto evaluate = [&](int k) -> int {
        sgpu_tmark t;
        SGPU_CHECK(sgpu_tbegin(ctx, &t));
        if (fused) {
            bool done = false;
            SGPU_CHECK(sgpu_launch_aar_step(ctx, c, X(k), b, F(k), anderson(k) ? nullptr : X(k + 1),
                                            jac, omega, &done));
            if (done) {
                SGPU_CHECK(sgpu_tend(ctx, &t, "aar_residual"));
                return SGPU_OK;
            }
            fused = false;
        }
        if (res) {
            res(user, N, c, X(k), b, r);
        } else {
            // r = b + (Lap + c) x
            SGPU_CHECK(sgpu_launch_stencil(ctx, SGPU_F64, 1, 1.0, 0.0, c, nullptr, X(k), ld, r, ld, b,
                                           ld, 1.0, 1.0, true, true, recording));
            SGPU_CHECK(sgpu_tend(ctx, &t, "aar_residual"));
        }
        if (recording) rec->fn(rec->user, X(k), r);
        return SGPU_OK;
    };
    // |r_k| from what evaluate(k) left
    auto residual_norm = [&](int k, double *norm) -> int {
        const double *v[1] = {fused ? F(k) : r};
        SGPU_CHECK(sgpu_dot_many(ctx, N, 1, v, v, norm));
        *norm = std::sqrt(*norm) / (fused ? std::fabs(jac) : 1.0);
        return SGPU_OK;
    };
    SGPU_HIP(hipMemcpyAsync(X(0), x, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    int it = 0, cur = 0, normed = -1;  // cur: the newest x; normed: the x of rnorm
    double rnorm = 0.0, bnorm = 0.0;
    const double *pb[1] = {b};
    SGPU_CHECK(sgpu_dot_many(ctx, N, 1, pb, pb, &bnorm));
    bnorm = std::sqrt(bnorm);
    SGPU_CHECK(evaluate(0));
    const double atol = tol * bnorm;
    rnorm = atol + 1.0;
    while (rnorm > atol && it < max_iter) {
        const bool and_step = anderson(it);
        if (!fused) {
            if (precond) precond(user, N, c, r, F(it));
            if (!precond || !and_step)
                aar_step<<<nb, 256, 0, ctx->stream>>>(r, F(it), precond ? 0.0 : jac, X(it),
                                                      and_step ? nullptr : X(it + 1), omega, n);
            SGPU_HIP(hipGetLastError());
        }
        if (and_step) {
            const int nh = std::min(it, m);
            AarRing xr, fr;
            AarCoeff G = {{0}};
            unsigned xdiff = 0;
            for (int j = 0; j <= kAarMaxM; j++) {
                xr.v[j] = X(it - std::min(j, nh));
                fr.v[j] = F(it - std::min(j, nh));
                if (j < nh && anderson(it - j - 1)) xdiff |= 1u << j;
            }
            if (recording) {
                double *Xh = ctx->aar_mem + (long)(1 + 2 * S) * ld, *Fh = Xh + (long)m * ld;
                aar_columns<<<nb, 256, 0, ctx->stream>>>(xr, fr, m, (it - 1) % m, ld, Xh, Fh, n);
                SGPU_CHECK(sgpu_anderson_coeff_dev(ctx, Fh, ld, m, F(it), n, G.g));
                aar_update_cols<<<nb, 256, 0, ctx->stream>>>(X(it + 1), X(it), F(it), Xh, Fh, ld, m, G,
                                                             beta, n);
            } else if (m <= 7) {
                SGPU_CHECK(ring_coeff<7>(ctx, fr, nh, n, G.g));
                aar_update<7><<<nb, 256, 0, ctx->stream>>>(X(it + 1), xr, fr, nh, xdiff, G, omega, beta, n);
            } else {
                SGPU_CHECK(ring_coeff<kAarMaxM>(ctx, fr, nh, n, G.g));
                aar_update<kAarMaxM><<<nb, 256, 0, ctx->stream>>>(X(it + 1), xr, fr, nh, xdiff, G, omega,
                                                                  beta, n);
            }
            SGPU_HIP(hipGetLastError());
        }
        cur = it + 1;
        SGPU_CHECK(evaluate(cur));
        if (and_step) {
            SGPU_CHECK(residual_norm(cur, &rnorm));
            normed = cur;
            // diverged (not finite, or 1e6 x the right-hand side's norm, which
            // no converging solve reaches): reported as not converged at once
            // instead of after max_iter iterations
            if (!std::isfinite(rnorm) || (bnorm > 0 && rnorm > 1e6 * bnorm)) break;
        }
        it++;
    }
    double rlast = rnorm;
    if (normed != cur) SGPU_CHECK(residual_norm(cur, &rlast));
    SGPU_HIP(hipMemcpyAsync(x, X(cur), n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    if (relres) *relres = bnorm > 0 ? rlast / bnorm : 0.0;
    if (iters) *iters = it;
    return (!std::isfinite(rnorm) || rnorm > atol) ? SGPU_NOT_CONVERGED : SGPU_OK;
}

extern "C" int sgpu_AAR(sgpu_context *ctx, sgpu_res_fn res, sgpu_precond_fn precond, void *user,
                        double c, int N, double *x_host, const double *b_host, double omega,
                        double beta, int m, int p, double tol, int max_iter, int *iters,
                        double *relres)
{
    if (!ctx || !x_host || !b_host || N != ctx->nd) {
        sgpu_set_error("sgpu_AAR: bad arguments (N %d, Nd %ld)", N, ctx ? ctx->nd : 0L);
        return SGPU_ERR_ARG;
    }
    SGPU_HIP(hipSetDevice(ctx->device));
    const long ld = ctx->ld;
    double *xb = nullptr;
    SGPU_HIP(hipMalloc((void **)&xb, 2 * ld * sizeof(double)));
    double *xd = xb, *bd = xb + ld;
    int st = SGPU_OK;
    if (hipMemcpyAsync(xd, x_host, (size_t)N * sizeof(double), hipMemcpyHostToDevice, ctx->stream) !=
            hipSuccess ||
        hipMemcpyAsync(bd, b_host, (size_t)N * sizeof(double), hipMemcpyHostToDevice, ctx->stream) !=
            hipSuccess) {
        sgpu_set_error("sgpu_AAR: upload failed");
        st = SGPU_ERR_HIP;
    }
    if (st == SGPU_OK)
        st = sgpu_aar_device(ctx, res, precond, user, c, N, xd, bd, omega, beta, m, p, tol, max_iter,
                             iters, relres);
    if (st >= 0 && (hipMemcpyAsync(x_host, xd, (size_t)N * sizeof(double), hipMemcpyDeviceToHost,
                                   ctx->stream) != hipSuccess ||
                    hipStreamSynchronize(ctx->stream) != hipSuccess)) {
        sgpu_set_error("sgpu_AAR: download failed");
        st = SGPU_ERR_HIP;
    }
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(xb);
    return st;
}
