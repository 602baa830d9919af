// vfs_reduce.h -- deterministic FP64 reductions for CDNA4 (64-wide waves).
//
// Each block reduces a grid-stride range with a fixed tree (wave shuffles,
// then LDS across the block's waves); the per-block partials are reduced by a
// single block in a second launch.  The order never depends on timing, so a
// result is bitwise reproducible run to run.
#pragma once

#include <hip/hip_runtime.h>

namespace vfs {

constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS = 1024;  // partials per reduction (fits ctx->red)

// blocks of a reduction over n elements: no more than have one each thread
inline unsigned reduce_blocks(long long n)
{
    const long long b = (n + RED_THREADS - 1) / RED_THREADS;
    return (unsigned)(b < 1 ? 1 : b < RED_BLOCKS ? b : RED_BLOCKS);
}

struct OpSum {
    __device__ static double init() { return 0.0; }
    __device__ static double op(double a, double b) { return a + b; }
};
struct OpMax {
    __device__ static double init() { return -1.0e308; }
    __device__ static double op(double a, double b) { return a > b ? a : b; }
};
struct OpMin {
    __device__ static double init() { return 1.0e308; }
    __device__ static double op(double a, double b) { return a < b ? a : b; }
};

// ---- reductions finished inside the kernel that makes the partials ----------
// Each block's thread 0 writes its partials past its own L2 (agent-scope
// stores: the XCDs' L2s are not coherent within a kernel) and counts itself;
// the block that counts last adds all partials, in block order, and can hand the
// results to the host at once through pinned memory.  Against a second launch,
// a copy and a stream synchronisation this takes 10 to 20 us off every scalar
// the host waits for.  The counters are zero between kernels.
constexpr int RED_CTRS = 33, RED_CTR_STRIDE = 32;  // 32 groups and the root, a cache line each
struct RedSync {
    unsigned *ctr;            // RED_CTRS * RED_CTR_STRIDE words, zero
    double *host;             // results for the host (pinned), or null
    unsigned long long *flag; // set to seq when they are there
    unsigned long long seq;
};
__device__ inline void red_put(double *p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline double red_get(const double *p)
{
    return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every store this wavefront has issued has reached its scope
__device__ inline void red_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Whether this block is the last of nb to get here (the same answer in all of
// its threads); thread 0 has red_put the block's partials.  Blocks count in 32
// groups first, so that no counter takes more than nb / 32 updates.
__device__ inline bool red_last(const RedSync &rs, unsigned nb)
{
    __shared__ unsigned last;
    if (threadIdx.x == 0) {
        red_drain();
        const unsigned grp = blockIdx.x & 31u, in = (nb - grp + 31u) / 32u, ngrp = nb < 32u ? nb : 32u;
        unsigned *c = rs.ctr + grp * RED_CTR_STRIDE, *root = rs.ctr + 32 * RED_CTR_STRIDE;
        last = 0;
        if (__hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == in - 1) {
            __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            red_drain();
            if (__hip_atomic_fetch_add(root, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ngrp - 1) {
                __hip_atomic_store(root, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = 1;
            }
        }
    }
    __syncthreads();
    return last != 0;
}
// results of the last block to the host: every thread of the block calls it;
// thread 0's earlier red_host stores are ordered before the flag
__device__ inline void red_host(double *p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
__device__ inline void red_publish(const RedSync &rs)
{
    red_drain();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(rs.flag, rs.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <class Op>
__device__ inline double wave_reduce(double v)
{
    for (int off = 32; off > 0; off >>= 1) v = Op::op(v, __shfl_down(v, off, 64));
    return v;
}

// Reduces v over the block; the result is valid in thread 0.
template <class Op>
__device__ inline double block_reduce(double v)
{
    __shared__ double part[RED_THREADS / 64];
    v = wave_reduce<Op>(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) part[w] = v;
    __syncthreads();
    double r = Op::init();
    if (threadIdx.x == 0)
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) r = Op::op(r, part[q]);
    __syncthreads();
    return r;
}

// The last block's sums of the nv partial rows part[v * RED_BLOCKS + 0 .. nb):
// a wavefront per row, 64 lanes wide, fixed order; results in out (device), in
// res (LDS) and, when the host waits, in rs.host.
template <class Op>
__device__ inline void red_finish_rows(const RedSync &rs, int nv, unsigned nb, const double *part, double *out, double *res)
{
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    for (int v = threadIdx.x >> 6; v < nv; v += nw) {
        double s = Op::init();
        for (unsigned q0 = lane; q0 < nb; q0 += 256) {
            double p[4];
#pragma unroll
            for (int e = 0; e < 4; e++) p[e] = q0 + 64 * e < nb ? red_get(part + v * RED_BLOCKS + q0 + 64 * e) : Op::init();
#pragma unroll
            for (int e = 0; e < 4; e++) s = Op::op(s, p[e]);
        }
        s = wave_reduce<Op>(s);
        if (lane == 0) {
            out[v] = s;
            res[v] = s;
            if (rs.host) red_host(rs.host + v, s);
        }
    }
    if (rs.host) red_publish(rs);
    else __syncthreads();
}

// Second stage: reduce `n` partials (n <= RED_BLOCKS * k) into out[0].
template <class Op>
__global__ void __launch_bounds__(RED_THREADS) finish_reduce(const double *__restrict__ part, int n,
                                                             double *__restrict__ out)
{
    double v = Op::init();
    for (int q = threadIdx.x; q < n; q += blockDim.x) v = Op::op(v, part[q]);
    v = block_reduce<Op>(v);
    if (threadIdx.x == 0) out[0] = v;
}

// The same, adding the result to out[0] (partial results of several passes
// summed in launch order).
template <class Op>
__global__ void __launch_bounds__(RED_THREADS) finish_reduce_add(const double *__restrict__ part, int n,
                                                                 double *__restrict__ out)
{
    double v = Op::init();
    for (int q = threadIdx.x; q < n; q += blockDim.x) v = Op::op(v, part[q]);
    v = block_reduce<Op>(v);
    if (threadIdx.x == 0) out[0] = Op::op(out[0], v);
}

}  // namespace vfs
