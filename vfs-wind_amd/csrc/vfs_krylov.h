// vfs_krylov.h -- the Gram-Schmidt sweeps over a Krylov basis shared by the
// Poisson FGMRES and the implicit momentum GMRES.  Deterministic: per-block
// partials added in a fixed order by the block that finishes last.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "vfs_reduce.h"

namespace vfs {

// The Gram-Schmidt sweeps over the Krylov basis.  Each is instantiated for a
// maximum basis count NVM (4, 8, 16 or 32; the host picks the smallest that
// holds nv), so that the per-vector accumulators stay in registers without
// spills, and each thread keeps U grid-stride elements in flight.

// dots[v] = <w, V_v> for v < nv and dots[nv] = <w, w>, finished by the last
// block
template <int NVM, int U>
__global__ void __launch_bounds__(RED_THREADS) k_multidot(long long n, int nv, const double *__restrict__ V, long long ld,
                                                          const double *__restrict__ w, double *part, double *out, RedSync rs)
{
    __shared__ double res[NVM + 1];
    double acc[NVM];
#pragma unroll
    for (int v = 0; v < NVM; v++) acc[v] = 0;
    double ww = 0;
    const long long S = (long long)gridDim.x * blockDim.x;
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (; t + (U - 1) * S < n; t += U * S) {
        double wt[U];
#pragma unroll
        for (int u = 0; u < U; u++) wt[u] = w[t + u * S];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) {
                double vt[U];
#pragma unroll
                for (int u = 0; u < U; u++) vt[u] = V[v * ld + t + u * S];
#pragma unroll
                for (int u = 0; u < U; u++) acc[v] += vt[u] * wt[u];
            }
#pragma unroll
        for (int u = 0; u < U; u++) ww += wt[u] * wt[u];
    }
    for (; t < n; t += S) {
        const double wt = w[t];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) acc[v] += V[v * ld + t] * wt;
        ww += wt * wt;
    }
#pragma unroll
    for (int v = 0; v < NVM; v++) {
        if (v < nv) {
            const double r = block_reduce<OpSum>(acc[v]);
            if (threadIdx.x == 0) red_put(part + v * RED_BLOCKS + blockIdx.x, r);
        }
    }
    const double r = block_reduce<OpSum>(ww);
    if (threadIdx.x == 0) red_put(part + nv * RED_BLOCKS + blockIdx.x, r);
    if (red_last(rs, gridDim.x)) red_finish_rows<OpSum>(rs, nv + 1, gridDim.x, part, out, res);
}

// First Gram-Schmidt sweep: w = w - sum_v h[v] V_v, and in the same sweep the
// dot products <V_v, w_new> a second (re-orthogonalisation) pass needs and
// <w_new, w_new>.  The last block finishes them into h2[0 .. nv] and decides on
// that pass: it is made when <w_new, w_new> fell below a quarter of ww0 = h[nv].
// h2[nv + 1] receives the square of the final norm.  After the second pass it
// follows from the dot products (V is orthonormal, so the pass takes sum h2^2
// off it; that sum is a rounding error's square except where w is nothing but
// rounding error), so that w need not be read again for it.  Where w is nothing
// but rounding error the difference has no correct digit; a negative one counts
// as zero, the new vector is then zero and the caller's estimate of the residual
// too: the basis is exhausted, which a measured norm of that rounding says as well.
template <int NVM, int U>
__global__ void __launch_bounds__(RED_THREADS) k_multiaxpy(long long n, int nv, const double *__restrict__ h,
                                                           const double *__restrict__ V, long long ld, double *__restrict__ w,
                                                           double *part, double *h2, RedSync rs)
{
    __shared__ double res[NVM + 1];
    double hv[NVM], acc[NVM];
#pragma unroll
    for (int v = 0; v < NVM; v++) {
        hv[v] = v < nv ? h[v] : 0.0;
        acc[v] = 0;
    }
    double ss = 0;
    const long long S = (long long)gridDim.x * blockDim.x;
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (; t + (U - 1) * S < n; t += U * S) {
        double s[U], vt[NVM][U];
#pragma unroll
        for (int u = 0; u < U; u++) s[u] = w[t + u * S];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv)
#pragma unroll
                for (int u = 0; u < U; u++) vt[v][u] = V[v * ld + t + u * S];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv)
#pragma unroll
                for (int u = 0; u < U; u++) s[u] -= hv[v] * vt[v][u];
#pragma unroll
        for (int u = 0; u < U; u++) {
            w[t + u * S] = s[u];
            ss += s[u] * s[u];
        }
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv)
#pragma unroll
                for (int u = 0; u < U; u++) acc[v] += vt[v][u] * s[u];
    }
    for (; t < n; t += S) {
        double vt[NVM];
        double s = w[t];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) {
                vt[v] = V[v * ld + t];
                s -= hv[v] * vt[v];
            }
        w[t] = s;
        ss += s * s;
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) acc[v] += vt[v] * s;
    }
#pragma unroll
    for (int v = 0; v < NVM; v++) {
        if (v < nv) {
            const double r = block_reduce<OpSum>(acc[v]);
            if (threadIdx.x == 0) red_put(part + v * RED_BLOCKS + blockIdx.x, r);
        }
    }
    ss = block_reduce<OpSum>(ss);
    if (threadIdx.x == 0) red_put(part + nv * RED_BLOCKS + blockIdx.x, ss);
    if (!red_last(rs, gridDim.x)) return;
    RedSync quiet = rs;
    quiet.host = nullptr;
    red_finish_rows<OpSum>(quiet, nv + 1, gridDim.x, part, h2, res);
    if (threadIdx.x == 0) {
        const double ww0 = h[nv];
        double ww = res[nv];
        if (ww < 0.25 * ww0)
            for (int v = 0; v < nv; v++) ww -= res[v] * res[v];
        h2[nv + 1] = ww;
        // the host's copy: h (nv), ww0, h2 (nv), ww1, final ww
        for (int v = 0; v <= nv; v++) {
            red_host(rs.host + v, h[v]);
            red_host(rs.host + nv + 1 + v, res[v]);
        }
        red_host(rs.host + 2 * nv + 2, ww);
    }
    red_publish(rs);
}

// Second sweep and normalisation: y = (w - sum_v h2[v] V_v) / norm where the
// second pass is made, else w / norm (zero for a zero norm); out(t, y) stores
// further copies of it
template <int NVM, class OUT>
__global__ void __launch_bounds__(RED_THREADS) k_orthonormal(long long n, int nv, const double *__restrict__ h,
                                                             const double *__restrict__ h2, const double *__restrict__ V,
                                                             long long ld, const double *w, double *y, OUT out)
{
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double hn = sqrt(h2[nv + 1] > 0 ? h2[nv + 1] : 0), sc = hn > 0 ? 1.0 / hn : 0.0;
    double s = w[t];
    if (h2[nv] < 0.25 * h[nv]) {
        double vt[NVM];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) vt[v] = V[v * ld + t];
#pragma unroll
        for (int v = 0; v < NVM; v++)
            if (v < nv) s -= h2[v] * vt[v];
    }
    const double r = sc * s;
    y[t] = r;
    out(t, r);
}

// y = x / sqrt(ww[0]) (zero for ww[0] <= 0)
template <class OUT>
__global__ void __launch_bounds__(RED_THREADS) k_normalise(long long n, double sign, const double *__restrict__ ww, const double *x,
                                                           double *y, OUT out)
{
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double hn = sqrt(ww[0] > 0 ? ww[0] : 0), sc = hn > 0 ? sign / hn : 0.0;
    const double r = sc * x[t];
    y[t] = r;
    out(t, r);
}

struct NoCopy {
    __device__ void operator()(long long, double) const {}
};

constexpr int KRYLOV_MAXV = 33;                    // basis vectors plus one
constexpr int KRYLOV_R = KRYLOV_MAXV * RED_BLOCKS; // results in the reduction scratch, after the partials
constexpr int KRYLOV_H2 = KRYLOV_R + KRYLOV_MAXV + 1;

// <w, V_v> (v < nv) and <w, w> into scratch[KRYLOV_R ..]; rs tells the host
inline void launch_multidot(hipStream_t st, long long n, int nv, const double *V, const double *w, double *scratch, const RedSync &rs)
{
    const dim3 gb(reduce_blocks(n)), tb(RED_THREADS);
    auto k = nv <= 4 ? k_multidot<4, 4> : nv <= 8 ? k_multidot<8, 4> : nv <= 16 ? k_multidot<16, 2> : k_multidot<KRYLOV_MAXV - 1, 1>;
    hipLaunchKernelGGL(k, gb, tb, 0, st, n, nv, V, n, w, scratch, scratch + KRYLOV_R, rs);
}

// One classical Gram-Schmidt step of w against V_0 .. V_{nv-1} with a second
// pass where the norm drops, and vnext = w / ||w||: three launches, the
// coefficients of each being the device results of the one before.  rs hands
// the host h (nv), ww0, h2 (nv), ww1 and the final <w, w> after the second launch,
// while the third runs.  It was seven launches, a copy and a synchronisation.
template <class OUT>
inline void launch_gram_schmidt(hipStream_t st, long long n, int nv, const double *V, double *w, double *vnext, double *scratch,
                                RedSync rs, const OUT &out)
{
    RedSync quiet = rs;
    quiet.host = nullptr;
    launch_multidot(st, n, nv, V, w, scratch, quiet);
    const dim3 gb(reduce_blocks(n)), tb(RED_THREADS);
    double *h = scratch + KRYLOV_R, *h2 = scratch + KRYLOV_H2;
    auto a = nv <= 4 ? k_multiaxpy<4, 4> : nv <= 8 ? k_multiaxpy<8, 4> : nv <= 16 ? k_multiaxpy<16, 2> : k_multiaxpy<KRYLOV_MAXV - 1, 1>;
    hipLaunchKernelGGL(a, gb, tb, 0, st, n, nv, (const double *)h, V, n, w, scratch, h2, rs);
    auto f = nv <= 4 ? k_orthonormal<4, OUT> : nv <= 8 ? k_orthonormal<8, OUT>
           : nv <= 16 ? k_orthonormal<16, OUT> : k_orthonormal<KRYLOV_MAXV - 1, OUT>;
    hipLaunchKernelGGL(f, dim3((unsigned)((n + RED_THREADS - 1) / RED_THREADS)), tb, 0, st, n, nv, (const double *)h,
                       (const double *)h2, V, n, (const double *)w, vnext, out);
}

// The host's side of a Gram-Schmidt step: the column h of the Hessenberg
// matrix (both passes' coefficients added) and the new vector's norm.
inline double gram_schmidt_column(const double *host, int nv, double *h)
{
    const double ww0 = host[nv], *h2 = host + nv + 1, ww1 = h2[nv], ww = host[2 * nv + 2];
    for (int v = 0; v < nv; v++) h[v] = host[v] + (ww1 < 0.25 * ww0 ? h2[v] : 0.0);
    return std::sqrt(ww > 0 ? ww : 0);
}

}  // namespace vfs
