// implicit.hip -- Crank-Nicolson momentum step, -imp 4 (implicitsolver.c:4203-4446).
//
// Residual (FormFunction_SNES, momentum.c:2237-2336, time_coeff() == 1):
//   R(U) = -(U - U_o)/dt + 0.5 F(U) + 0.5 F(U_o) - dP (+ F_eul)
// with F = Formfunction_2 after the wall-flux zeroing and Contra2Cart of U.
// The reference hands R to PETSc's SNES (trust region, matrix-free finite
// difference Jacobian, GMRES without preconditioner, Eisenstat-Walker
// forcing).  Here the same solve runs on the device: an inexact Newton
// iteration with Eisenstat-Walker forcing and residual-decrease step
// halving, GMRES(m) with classical Gram-Schmidt and one re-orthogonalisation
// pass, and the matrix-free product J v = (R(U + h v) - R(U)) / h with
// PETSc's default differencing parameter.  Every vector (3 doubles per DA
// point) stays in HBM; the host sees only dot products.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "vfs_internal.h"
#include "vfs_reduce.h"
#include "vfs_krylov.h"

#pragma clang fp contract(off)

namespace vfs {

constexpr int IM_TPB = 256;
constexpr int IM_MAXV = KRYLOV_MAXV;  // GMRES basis vectors held by the dot kernel

// wall-flux zeroing of FormFunction_SNES (momentum.c:2258-2282), one thread
// per point of the six boundary planes: every rule acts on its own plane only,
// and no two write one component of a point (a thread per grid point took
// 65 us at 384x192x256)
__host__ __device__ inline long long boundary_points(const Grid &g)
{
    return 2 * ((long long)g.my * g.mz + (long long)g.mx * g.mz + (long long)g.mx * g.my);
}
__global__ void k_snes_bc(Grid g, double *__restrict__ ucont)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long ni = 2LL * g.my * g.mz, nj = 2LL * g.mx * g.mz, nk = 2LL * g.mx * g.my;
    const int mx = g.mx, my = g.my, mz = g.mz;
    int face, i, j, k;
    if (t < ni) {
        face = (int)(t & 1); j = (int)((t >> 1) % my); k = (int)((t >> 1) / my); i = face ? mx - 1 : 0;
    } else if ((t -= ni) < nj) {
        face = 2 + (int)(t & 1); i = (int)((t >> 1) % mx); k = (int)((t >> 1) / mx); j = face & 1 ? my - 1 : 0;
    } else if ((t -= nj) < nk) {
        face = 4 + (int)(t & 1); i = (int)((t >> 1) % mx); j = (int)((t >> 1) / mx); k = face & 1 ? mz - 1 : 0;
    } else {
        return;
    }
    const int *b = g.bc;
#define UC(kk, jj, ii, c) ucont[3 * (((long long)(kk) * my + (jj)) * mx + (ii)) + (c)]
    const bool in_jk = j != 0 && j != my - 1 && k != 0 && k != mz - 1, in_ik = i != 0 && i != mx - 1 && k != 0 && k != mz - 1;
    switch (face) {
    case 0: if (b[0] == 1 || (b[0] == 10 && in_jk)) UC(k, j, i, 0) = 0; break;
    case 1: if (b[1] == 1 || (b[1] == 10 && in_jk)) UC(k, j, i - 1, 0) = 0; break;
    case 2: if (b[2] == 1 || b[2] == 12 || (b[2] == 10 && in_ik)) UC(k, j, i, 1) = 0; break;
    case 3: if (b[3] == 1 || b[3] == 2 || b[3] == 12 || ((b[3] == 10 || b[3] == -10) && in_ik)) UC(k, j - 1, i, 1) = 0; break;
    case 4: if (b[4] == 1) UC(k, j, i, 2) = 0; break;
    default: if (b[5] == 1) UC(k - 1, j, i, 2) = 0; break;
    }
#undef UC
}

// Rhs = 0; Rhs += (-1/dt) U; Rhs += (1/dt) U_o   (PETSc VecAXPY order)
__global__ void k_cn_base(long long n3, double rdt, const double *__restrict__ u, const double *__restrict__ uo,
                          double *__restrict__ rhs)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n3) return;
    double s = 0.0 + (-rdt) * u[t];
    rhs[t] = s + rdt * uo[t];
}

// R = Rhs + 0.5 RHS_o - dP (+ F_eul)
__global__ void k_cn_finish(long long n3, const double *__restrict__ rhs, const double *__restrict__ rhso,
                            const double *__restrict__ dp, const double *__restrict__ feul, double *__restrict__ r)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n3) return;
    double s = rhs[t] + 0.5 * rhso[t];
    s = s + (-1.0) * dp[t];
    if (feul) s = s + feul[t];
    r[t] = s;
}

// post-solve boundary fix of Implicit_MatrixFree (implicitsolver.c:4330-4392)
// for wall (1), slip (10) and outlet (4) faces
__global__ void k_imp_post(Grid g, const double *__restrict__ eta, const double *__restrict__ zet,
                           double *__restrict__ ucont, double *__restrict__ ucat)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= g.n) return;
    const int i = t % g.mx;
    const long long r = t / g.mx;
    const int j = r % g.my, k = r / g.my;
    const int mx = g.mx, my = g.my, mz = g.mz;
    const int *b = g.bc;
    auto wall = [](int c) { return c == 1 || c == -1 || c == -2 || c == 10; };
    double *uc = ucont + 3 * t;
    if (wall(b[0]) && i == 0) uc[0] = 0;
    if (wall(b[1]) && i == mx - 2) uc[0] = 0;
    if (wall(b[2]) && j == 0) uc[1] = 0;
    if ((wall(b[3]) || b[3] == 2) && j == my - 2) uc[1] = 0;
    if (wall(b[4]) && k == 0) uc[2] = 0;
    if (wall(b[5]) && k == mz - 2) uc[2] = 0;
    if ((b[0] == -1 || b[0] == -2) && i == 1) uc[0] = 0;
    if ((b[1] == -1 || b[1] == -2) && i == mx - 3) uc[0] = 0;
    if ((b[2] == -1 || b[2] == -2) && j == 1) uc[1] = 0;
    if ((b[3] == -1 || b[3] == -2) && j == my - 3) uc[1] = 0;
    if ((b[4] == -1 || b[4] == -2) && k == 1) uc[2] = 0;
    if ((b[5] == -1 || b[5] == -2) && k == mz - 3) uc[2] = 0;
    if (b[3] == 4 && j == my - 2) {
        const long long q1 = t + mx;
        for (int c = 0; c < 3; c++) ucat[3 * q1 + c] = ucat[3 * t + c];
        const double *e = eta + 3 * t;
        uc[1] = 0.5 * (ucat[3 * t] + ucat[3 * q1]) * e[0] + 0.5 * (ucat[3 * t + 1] + ucat[3 * q1 + 1]) * e[1] +
                0.5 * (ucat[3 * t + 2] + ucat[3 * q1 + 2]) * e[2];
    }
    if (b[5] == 4 && k == mz - 2) {
        const long long q1 = t + g.plane;
        for (int c = 0; c < 3; c++) ucat[3 * q1 + c] = ucat[3 * t + c];
        const double *z = zet + 3 * t;
        uc[2] = 0.5 * (ucat[3 * t] + ucat[3 * q1]) * z[0] + 0.5 * (ucat[3 * t + 1] + ucat[3 * q1 + 1]) * z[1] +
                0.5 * (ucat[3 * t + 2] + ucat[3 * q1 + 2]) * z[2];
        if (uc[2] < 0) {
            uc[2] = 0;
            for (int c = 0; c < 3; c++) ucat[3 * t + c] = ucat[3 * q1 + c] = 0;
        }
    }
}

// ---- device vector algebra (deterministic reductions; the Gram-Schmidt
// sweeps are vfs_krylov.h's) --------------------------------------------------
// y = a x + b y, coefficients from device memory (a = s[ia], b = s[ib] or 0/1)
__global__ void k_im_axpby(long long n, double a, const double *__restrict__ x, double b, double *__restrict__ y)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    y[t] = a * x[t] + b * y[t];
}

// y = a x
__global__ void k_im_scale(long long n, double a, const double *__restrict__ x, double *__restrict__ y)
{
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t < n) y[t] = a * x[t];
}

// z = x + a y
__global__ void k_im_waxpy(long long n, const double *__restrict__ x, double a, const double *__restrict__ y,
                           double *__restrict__ z)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    z[t] = x[t] + a * y[t];
}

// x = sum_v y[v] V_v (first) or x + sum_v y[v] V_v, the terms added in v
// order with the fused multiply-add of a chain of k_im_axpby updates
struct ImpY {
    double v[IM_MAXV];
};
__global__ void k_im_update(long long n, int nv, ImpY y, const double *__restrict__ V, long long ld,
                            double *__restrict__ x, int first)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    double s = first ? 0.0 : x[t];
    for (int v = 0; v < nv; v++) s = y.v[v] * V[v * ld + t] + s;
    x[t] = s;
}

// z = z2 = x + a y (the line search's trial state and the residual's input)
__global__ void k_im_waxpy2(long long n, const double *__restrict__ x, double a, const double *__restrict__ y,
                            double *__restrict__ z, double *__restrict__ z2)
{
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double v = x[t] + a * y[t];
    z[t] = v;
    z2[t] = v;
}

// sum of |x| (for the differencing parameter)
__global__ void __launch_bounds__(RED_THREADS) k_im_asum_dot(long long n, const double *__restrict__ u,
                                                             const double *__restrict__ v, double *part, double *out, RedSync rs)
{
    __shared__ double res[3];
    double a = 0, d = 0, vv = 0;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
        const double x = v[t];
        a += fabs(x);
        d += u[t] * x;
        vv += x * x;
    }
    a = block_reduce<OpSum>(a);
    d = block_reduce<OpSum>(d);
    vv = block_reduce<OpSum>(vv);
    if (threadIdx.x == 0) {
        red_put(part + blockIdx.x, a);
        red_put(part + RED_BLOCKS + blockIdx.x, d);
        red_put(part + 2 * RED_BLOCKS + blockIdx.x, vv);
    }
    if (red_last(rs, gridDim.x)) red_finish_rows<OpSum>(rs, 3, gridDim.x, part, out, res);
}

}  // namespace vfs

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace vfs {

struct ImpState {
    long long n3 = 0;
    int m = 0;
    double *U = nullptr, *R = nullptr, *W = nullptr, *FW = nullptr, *dx = nullptr, *V = nullptr;
};

// Carve the solver's vectors out of the context's persistent workspace
// (5 + m + 1 vectors of n3 doubles), allocating or
// growing it first when needed.  Every vector is written before it is read.
static int im_workspace(vfs_ctx *c, ImpState &s)
{
    const size_t vb = (size_t)s.n3 * sizeof(double);
    const size_t need = (size_t)(6 + s.m) * vb;
    if (c->imp_ws_bytes < need) {
        VFS_HIP(hipStreamSynchronize(c->stream));
        if (c->imp_ws) hipFree(c->imp_ws);
        c->imp_ws = nullptr;
        c->imp_ws_bytes = 0;
        hipError_t e = hipMalloc((void **)&c->imp_ws, need);
        if (e != hipSuccess) { c->imp_ws = nullptr; return check_hip(e, "hipMalloc (implicit)"); }
        e = hipMemsetAsync(c->imp_ws, 0, need, c->stream);
        if (e != hipSuccess) return check_hip(e, "hipMemsetAsync (implicit)");
        c->imp_ws_bytes = need;
    }
    double *p = c->imp_ws;
    s.U = p; p += s.n3;
    s.R = p; p += s.n3;
    s.W = p; p += s.n3;
    s.FW = p; p += s.n3;
    s.dx = p; p += s.n3;
    s.V = p;
    return VFS_OK;
}

// R(u) into r (FormFunction_SNES); leaves UCONT/UCAT at the BC-zeroed u.
// With rbase, r = da rbase + db R(u) (one k_im_axpby's arithmetic), formed in
// the cell pass on the fused path.
int snes_function(vfs_ctx *c, const double *u, double *r, int use_feul, const double *rbase = nullptr, double da = 0,
                  double db = 0)
{
    const Grid &g = c->g;
    hipStream_t st = c->stream;
    const long long n3 = 3 * g.n;
    if (u != c->f[VFS_UCONT])
        VFS_HIP(hipMemcpyAsync(c->f[VFS_UCONT], u, n3 * sizeof(double), hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_snes_bc, dim3(blocks_for(boundary_points(g), IM_TPB)), dim3(IM_TPB), 0, st, g, c->f[VFS_UCONT]);
    ucat_stale(c);
    VFS_LAUNCH_CHECK("snes bc");
    int rc = c2c(c);
    if (rc) return rc;
    // on the fused path the residual is formed in the cell pass (the same
    // operations in the same order); VFS_FUSED_CN=0 keeps the three passes
    const char *fe = std::getenv("VFS_FUSED_CN");
    if (formfunction2_fused(c) && !(fe && fe[0] == '0')) {
        const CnResidual cn{c->f[VFS_UCONT_O], c->f[VFS_RHS_O], use_feul ? c->f[VFS_FEUL] : nullptr, 1. / c->p.dt, r,
                            rbase, da, db};
        return formfunction2(c, 0.5, nullptr, 0.0, nullptr, &cn);
    }
    hipLaunchKernelGGL(k_cn_base, dim3(blocks_for(n3, IM_TPB)), dim3(IM_TPB), 0, st, n3, 1. / c->p.dt, c->f[VFS_UCONT],
                       c->f[VFS_UCONT_O], c->f[VFS_RHS]);
    rc = formfunction2(c, 0.5, nullptr, 0.0, nullptr);
    if (rc) return rc;
    hipLaunchKernelGGL(k_cn_finish, dim3(blocks_for(n3, IM_TPB)), dim3(IM_TPB), 0, st, n3, c->f[VFS_RHS], c->f[VFS_RHS_O],
                       c->f[VFS_DP], use_feul ? c->f[VFS_FEUL] : (const double *)nullptr, r);
    if (rbase) hipLaunchKernelGGL(k_im_axpby, dim3(blocks_for(n3, IM_TPB)), dim3(IM_TPB), 0, st, n3, da, rbase, db, r);
    VFS_LAUNCH_CHECK("snes residual");
    return VFS_OK;
}

static int im_norm(vfs_ctx *c, long long n, const double *w, double *out)
{
    launch_multidot(c->stream, n, 0, nullptr, w, c->red, red_sync(c));
    VFS_LAUNCH_CHECK("implicit norm");
    const int rc = red_wait(c);
    if (!rc) *out = std::sqrt(c->red_host[0]);
    return rc;
}

// J v = (R(U + h v) - R(U)) / h, PETSc MatMFFD "ds" parameter:
// h = e * (u.v) / |v|^2, or e * umin * sign(u.v) * |v|_1 / |v|^2 when |u.v| < umin |v|_1
static int mffd(vfs_ctx *c, ImpState &s, const double *v, double *jv, int use_feul, int *nfunc)
{
    hipStream_t st = c->stream;
    const long long n = s.n3;
    hipLaunchKernelGGL(k_im_asum_dot, dim3(reduce_blocks(n)), dim3(RED_THREADS), 0, st, n, s.U, v, c->red, c->red + 3 * RED_BLOCKS,
                       red_sync(c));
    VFS_LAUNCH_CHECK("mffd norms");
    int rc = red_wait(c);
    if (rc) return rc;
    const double asum = c->red_host[0], dot = c->red_host[1], vv = c->red_host[2];
    if (vv == 0) {
        VFS_HIP(hipMemsetAsync(jv, 0, n * sizeof(double), st));
        return VFS_OK;
    }
    const double err = 1.490116119384766e-08, umin = 1.e-6;  // sqrt(DBL_EPSILON), PETSc defaults
    double hh = dot;
    if (std::fabs(hh) < umin * asum) hh = (hh >= 0 ? 1.0 : -1.0) * umin * asum;
    hh = err * hh / vv;
    // U + h v goes straight into UCONT, where the residual evaluation reads it
    hipLaunchKernelGGL(k_im_waxpy, dim3(blocks_for(n, IM_TPB)), dim3(IM_TPB), 0, st, n, s.U, hh, v, c->f[VFS_UCONT]);
    // jv = (F(U + h v) - F(U)) / h, the quotient formed with the residual
    rc = snes_function(c, c->f[VFS_UCONT], jv, use_feul, s.R, -1.0 / hh, 1.0 / hh);
    if (rc) return rc;
    (*nfunc)++;
    VFS_LAUNCH_CHECK("mffd");
    return VFS_OK;
}

// GMRES(m) for J dx = -R, dx from zero; bnorm = ||R||; returns iterations
static int gmres(vfs_ctx *c, ImpState &s, double bnorm, double rtol, int maxit, int use_feul, int *its, int *nfunc)
{
    hipStream_t st = c->stream;
    const long long n = s.n3;
    const int m = s.m;
    const unsigned nb = blocks_for(n, IM_TPB);
    int rc = VFS_OK;
    std::vector<double> H((size_t)(m + 1) * m), cs(m), sn(m), gv(m + 1), y(m);
    // r0 = -R (dx = 0); dx is first written by the first restart's update
    *its = 0;
    if (bnorm == 0) {
        VFS_HIP(hipMemsetAsync(s.dx, 0, n * sizeof(double), st));
        return VFS_OK;
    }
    double beta = bnorm;
    bool first = true, restart0 = true;
    while (*its < maxit) {
        double *V0 = s.V;
        if (first) {
            hipLaunchKernelGGL(k_im_scale, dim3(nb), dim3(IM_TPB), 0, st, n, -1.0 / beta, (const double *)s.R, V0);
        } else {
            // r = -R - J dx
            rc = mffd(c, s, s.dx, s.FW, use_feul, nfunc);
            if (rc) return rc;
            hipLaunchKernelGGL(k_im_axpby, dim3(nb), dim3(IM_TPB), 0, st, n, -1.0, s.R, -1.0, s.FW);
            rc = im_norm(c, n, s.FW, &beta);
            if (rc) return rc;
            if (beta <= rtol * bnorm) break;
            hipLaunchKernelGGL(k_im_scale, dim3(nb), dim3(IM_TPB), 0, st, n, 1.0 / beta, (const double *)s.FW, V0);
        }
        first = false;
        std::fill(gv.begin(), gv.end(), 0.0);
        gv[0] = beta;
        int jj;
        for (jj = 0; jj < m && *its < maxit; jj++, (*its)++) {
            double *vj = s.V + (size_t)jj * n, *w = s.V + (size_t)(jj + 1) * n;
            rc = mffd(c, s, vj, w, use_feul, nfunc);
            if (rc) return rc;
            // classical Gram-Schmidt with a second pass where the norm drops; w is
            // normalised in place
            double h[IM_MAXV];
            launch_gram_schmidt(st, n, jj + 1, s.V, w, w, c->red, red_sync(c), NoCopy{});
            VFS_LAUNCH_CHECK("implicit gram-schmidt");
            rc = red_wait(c);
            if (rc) return rc;
            const double hn = gram_schmidt_column(c->red_host, jj + 1, h);
            for (int v = 0; v <= jj; v++) H[(size_t)v * m + jj] = h[v];
            H[(size_t)(jj + 1) * m + jj] = hn;
            for (int i = 0; i < jj; i++) {
                const double tmp = cs[i] * H[(size_t)i * m + jj] + sn[i] * H[(size_t)(i + 1) * m + jj];
                H[(size_t)(i + 1) * m + jj] = -sn[i] * H[(size_t)i * m + jj] + cs[i] * H[(size_t)(i + 1) * m + jj];
                H[(size_t)i * m + jj] = tmp;
            }
            const double a = H[(size_t)jj * m + jj], bb = H[(size_t)(jj + 1) * m + jj];
            const double den = std::sqrt(a * a + bb * bb);
            cs[jj] = den > 0 ? a / den : 1.0;
            sn[jj] = den > 0 ? bb / den : 0.0;
            H[(size_t)jj * m + jj] = den;
            H[(size_t)(jj + 1) * m + jj] = 0;
            gv[jj + 1] = -sn[jj] * gv[jj];
            gv[jj] = cs[jj] * gv[jj];
            if (std::fabs(gv[jj + 1]) <= rtol * bnorm || hn == 0) { jj++; (*its)++; break; }
        }
        for (int i = jj - 1; i >= 0; i--) {
            double sacc = gv[i];
            for (int q = i + 1; q < jj; q++) sacc -= H[(size_t)i * m + q] * y[q];
            y[i] = H[(size_t)i * m + i] != 0 ? sacc / H[(size_t)i * m + i] : 0.0;
        }
        // dx += sum_q y_q V_q in one sweep (dx = 0 before the first restart)
        ImpY yk;
        for (int q = 0; q < jj; q++) yk.v[q] = y[q];
        hipLaunchKernelGGL(k_im_update, dim3(nb), dim3(IM_TPB), 0, st, n, jj, yk, s.V, n, s.dx, restart0 ? 1 : 0);
        restart0 = false;
        VFS_LAUNCH_CHECK("gmres update");
        if (std::fabs(gv[jj]) <= rtol * bnorm) break;
    }
    if (restart0) VFS_HIP(hipMemsetAsync(s.dx, 0, n * sizeof(double), st));  // no update was made
    return VFS_OK;
}

}  // namespace vfs

using namespace vfs;

extern "C" {

int vfs_formfunction_snes(vfs_ctx *c, const double *u_dev, double *r_dev, int use_feul)
{
    if (!c || !u_dev || !r_dev) return set_error(VFS_EINVAL, "vfs_formfunction_snes: null argument");
    return snes_function(c, u_dev, r_dev, use_feul);
}

int vfs_store_old_state(vfs_ctx *c)
{
    if (!c) return set_error(VFS_EINVAL, "null context");
    const size_t n3 = 3 * (size_t)c->g.n;
    // Ucont_o = Ucont; RHS_o = Formfunction_2(Ucont) (solvers.c:627-628)
    VFS_HIP(hipMemcpyAsync(c->f[VFS_UCONT_O], c->f[VFS_UCONT], n3 * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    VFS_HIP(hipMemsetAsync(c->f[VFS_RHS], 0, n3 * sizeof(double), c->stream));
    int rc = formfunction2(c, 1.0, nullptr, 0.0, nullptr);
    if (rc) return rc;
    VFS_HIP(hipMemcpyAsync(c->f[VFS_RHS_O], c->f[VFS_RHS], n3 * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    return VFS_OK;
}

int vfs_implicit_matrixfree(vfs_ctx *c, const vfs_newton_opts *o, vfs_newton_stats *stats)
{
    using clk = std::chrono::steady_clock;
    auto t0 = clk::now();
    if (!c || !o) return set_error(VFS_EINVAL, "vfs_implicit_matrixfree: null argument");
    const int m = o->restart > 0 ? (o->restart < IM_MAXV - 1 ? o->restart : IM_MAXV - 2) : 30;
    ImpState s;
    s.n3 = 3 * c->g.n;
    s.m = m;
    const size_t vb = (size_t)s.n3 * sizeof(double);
    int rc = im_workspace(c, s);
    if (rc) return rc;
    hipStream_t st = c->stream;
    const long long n = s.n3;
    const unsigned nb = blocks_for(n, IM_TPB);
    auto fail = [&](int code) { return code; };
    // InflowFlux, then FormBCS with outflow_scale = 0 (implicitsolver.c:4293-4297)
    rc = inflow_flux(c, nullptr);
    if (!rc) rc = form_bcs(c, 0);
    if (rc) return fail(rc);
    VFS_HIP(hipMemcpyAsync(s.U, c->f[VFS_UCONT], vb, hipMemcpyDeviceToDevice, st));
    int nfunc = 0, newton = 0, lin_total = 0;
    rc = snes_function(c, s.U, s.R, o->use_feul);
    if (rc) return fail(rc);
    nfunc++;
    double fnorm;
    rc = im_norm(c, n, s.R, &fnorm);
    if (rc) return fail(rc);
    const double fnorm0 = fnorm;
    const double rtol = o->rtol > 0 ? o->rtol : 1e-4;
    const int maxit = o->max_newton > 0 ? o->max_newton : 50;
    const int maxlin = o->max_linear > 0 ? o->max_linear : 1000;
    // Eisenstat-Walker, version 3 parameters (implicitsolver.c:4251-4252, PETSc defaults)
    const double ew_rtol0 = 0.3, ew_max = 0.9, ew_gamma = 1.0, ew_alpha = 0.5 * (1.0 + std::sqrt(5.0)), ew_thresh = 0.1;
    double eta = ew_rtol0, fnorm_last = fnorm;
    bool converged = fnorm <= rtol * fnorm0 || fnorm == 0;
    while (!converged && newton < maxit) {
        if (newton > 0) {
            double e = ew_gamma * std::pow(fnorm / fnorm_last, ew_alpha);
            const double sg = ew_gamma * std::pow(eta, ew_alpha);
            if (sg > ew_thresh) e = std::fmax(e, sg);
            eta = std::fmin(e, ew_max);
        }
        int its = 0;
        rc = gmres(c, s, fnorm, eta, maxlin, o->use_feul, &its, &nfunc);
        if (rc) return fail(rc);
        lin_total += its;
        // step with halving while the residual does not decrease
        double lam = 1.0, fnew = 0;
        bool accepted = false;
        for (int half = 0; half < 8; half++) {
            hipLaunchKernelGGL(k_im_waxpy2, dim3(nb), dim3(IM_TPB), 0, st, n, s.U, lam, s.dx, s.W, c->f[VFS_UCONT]);
            rc = snes_function(c, c->f[VFS_UCONT], s.FW, o->use_feul);
            if (rc) return fail(rc);
            nfunc++;
            rc = im_norm(c, n, s.FW, &fnew);
            if (rc) return fail(rc);
            if (fnew < fnorm) { accepted = true; break; }
            lam *= 0.5;
        }
        newton++;
        if (!accepted) break;
        std::swap(s.U, s.W);
        std::swap(s.R, s.FW);
        fnorm_last = fnorm;
        fnorm = fnew;
        converged = fnorm <= rtol * fnorm0;
    }
    // U -> Ucont with Ucat as the last residual evaluation at U left it, the
    // post-solve boundary fix and FormBCS(outflow_scale = 1)
    VFS_HIP(hipMemcpyAsync(c->f[VFS_UCONT], s.U, vb, hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_snes_bc, dim3(blocks_for(boundary_points(c->g), IM_TPB)), dim3(IM_TPB), 0, st, c->g, c->f[VFS_UCONT]);
    ucat_stale(c);
    rc = c2c(c);
    if (rc) return fail(rc);
    hipLaunchKernelGGL(k_imp_post, dim3(blocks_for(c->g.n, IM_TPB)), dim3(IM_TPB), 0, st, c->g, c->f[VFS_ETA], c->f[VFS_ZET],
                       c->f[VFS_UCONT], c->f[VFS_UCAT]);
    ucat_stale(c);
    VFS_LAUNCH_CHECK("implicit post");
    rc = form_bcs(c, 1);
    if (rc) return fail(rc);
    VFS_HIP(hipStreamSynchronize(st));
    if (stats) {
        stats->newton_iterations = newton;
        stats->linear_iterations = lin_total;
        stats->function_evals = nfunc;
        stats->fnorm0 = fnorm0;
        stats->fnorm = fnorm;
        stats->ms = std::chrono::duration<double, std::milli>(clk::now() - t0).count();
    }
    if (!converged) return set_error(VFS_ENOCONV, "implicit momentum: Newton did not reach the tolerance");
    return VFS_OK;
}

}  // extern "C"
