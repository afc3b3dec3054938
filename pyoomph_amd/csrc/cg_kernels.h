// Vector work of preconditioned conjugate gradients in four launches per iteration, per
// sub-problem, on the chunks of gmres_kernels.h (256, 512 or 1024 rows of one sub-problem):
//   cg_dots  partials of (p, q), q = A p
//   cg_step  alpha = rz / (p, q);  x += alpha p, r -= alpha q [, x0 = W r]
//   cg_dots  partials of (r, r) and (r, z), z = M^-1 r
//   cg_dir   convergence test on (r, r), beta = rz_new / rz;  p = z + beta p
// cg_step and cg_dir sum the partials of their sub-problem in every block (lane-strided over
// its chunks, then an xor tree) and derive the scalars there; the sub-problem's first block
// stores them. That replaces two reductions and two scalar launches, 1.4-3 us each, of an
// iteration. rz alternates between two arrays, since a first block may store the new value
// while other blocks still read the old one. Sub-problems of more than kGsFusedChunks chunks
// get their sums from a launch of cg_sums (same order, same bits).
// Bound: HBM (cg_step 5-6 vectors, cg_dir 3, the dots 2 each); launches for small systems.
#pragma once
#include "gmres_kernels.h"

namespace pyhip {

constexpr int kCgThreads = 256;
constexpr int kGsFusedChunks = 640;   // the blocks of a longer sub-problem would read over 5 KB each

// sum over the block's 256 threads: wave trees, then the waves in order; in thread 0
__device__ __forceinline__ double cg_block_sum(double v, double *sh) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}

// (a, b) and, with c given, (c, d), per chunk: part[chunk], part[count + chunk]
template <typename T>
__global__ __launch_bounds__(kCgThreads) void cg_dots_kernel(const T *__restrict__ a, const T *__restrict__ b,
                                                             const T *__restrict__ c, const T *__restrict__ d,
                                                             GsChunks C, const int32_t *__restrict__ active,
                                                             double *__restrict__ part) {
    __shared__ double sh[2][4];
    if (active && !active[C.sub[blockIdx.x]]) return;   // the whole block
    const int64_t r0 = C.begin[blockIdx.x], r1 = C.end[blockIdx.x];
    double s = 0.0, t = 0.0;
#pragma unroll 4
    for (int64_t i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
        s += double(a[i]) * double(b[i]);
        if (c) t += double(c[i]) * double(d[i]);
    }
    s = cg_block_sum(s, sh[0]);
    if (c) t = cg_block_sum(t, sh[1]);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s;
        if (c) part[C.count + blockIdx.x] = t;
    }
}

// sums[v][s] of the partials' row v (nv rows) for every sub-problem, one wave each
__global__ __launch_bounds__(64) void cg_sums_kernel(int nsub, GsChunks C, const int32_t *__restrict__ active,
                                                        const double *__restrict__ part, double *__restrict__ sums) {
    const int v = blockIdx.x / nsub, s = blockIdx.x % nsub;
    if (active && !active[s]) return;
    double a = 0.0;
    for (int32_t c = C.ptr[s] + (int32_t)threadIdx.x; c < C.ptr[s + 1]; c += 64) a += part[v * C.count + c];
    a = wave_sum(a);
    if (threadIdx.x == 0) sums[v * nsub + s] = a;
}

// the sum of partial row v of sub-problem s, in every thread (sh: one double per row)
__device__ __forceinline__ void cg_total(int v, int nsub, int s, const GsChunks &C, const double *__restrict__ part,
                                         const double *__restrict__ sums, double *sh) {
    if ((int)(threadIdx.x >> 6) != v) return;   // wave v sums row v
    double a = 0.0;
    if (sums) {
        a = sums[v * nsub + s];
    } else {
        for (int32_t c = C.ptr[s] + (int32_t)(threadIdx.x & 63); c < C.ptr[s + 1]; c += 64) a += part[v * C.count + c];
        a = wave_sum(a);
    }
    if ((threadIdx.x & 63) == 0) *sh = a;
}

// flags and counters of a sub-problem: fail[s] on a non-positive curvature (breakdown),
// nspmv[s] the iterations whose spmv visited it
template <typename T>
__global__ __launch_bounds__(kCgThreads) void cg_step_kernel(int nsub, const T *__restrict__ p, const T *__restrict__ q,
                                                             T *__restrict__ x, T *__restrict__ r,
                                                             const double *__restrict__ rz, GsChunks C,
                                                             const double *__restrict__ part,
                                                             const double *__restrict__ sums, int32_t *active,
                                                             int32_t *__restrict__ fail, int32_t *__restrict__ nspmv,
                                                             const T *__restrict__ w0, T *__restrict__ x0) {
    __shared__ double sh;
    __shared__ int run;
    const int s = C.sub[blockIdx.x];
    if (threadIdx.x == 0) run = active[s];   // one read: the block takes one way
    cg_total(0, nsub, s, C, part, sums, &sh);
    __syncthreads();
    if (!run) return;
    const double pq = sh;
    const bool bad = !(pq > 0.0) || !isfinite(pq);
    if (threadIdx.x == 0 && (int32_t)blockIdx.x == C.ptr[s]) {
        nspmv[s] += 1;
        if (bad) {
            active[s] = 0;
            fail[s] = 1;
        }
    }
    if (bad) return;   // every block of the sub-problem finds the same
    const double a = rz[s] / pq;
    const int64_t r1 = C.end[blockIdx.x];
#pragma unroll 4
    for (int64_t i = C.begin[blockIdx.x] + threadIdx.x; i < r1; i += kCgThreads) {
        x[i] = T(double(x[i]) + a * double(p[i]));
        const T rn = T(double(r[i]) - a * double(q[i]));
        r[i] = rn;
        // the multigrid V-cycle's first smoothing x0 = W r of the new residual
        if (x0) x0[i] = w0[i] * rn;
    }
}

// rzold / rznew: the two arrays of (r, z); nprec[s]: the preconditioner applies that visited s
template <typename T>
__global__ __launch_bounds__(kCgThreads) void cg_dir_kernel(int nsub, const T *__restrict__ z, T *__restrict__ p,
                                                            const double *__restrict__ rzold,
                                                            double *__restrict__ rznew, GsChunks C,
                                                            const double *__restrict__ part,
                                                            const double *__restrict__ sums,
                                                            const double *__restrict__ bnorm, double rtol,
                                                            int32_t *active, int32_t *__restrict__ nprec) {
    __shared__ double sh[2];
    __shared__ int run;
    const int s = C.sub[blockIdx.x];
    if (threadIdx.x == 0) run = active[s];
    cg_total(0, nsub, s, C, part, sums, &sh[0]);
    cg_total(1, nsub, s, C, part, sums, &sh[1]);
    __syncthreads();
    if (!run) return;
    const double rr = sh[0], rzn = sh[1];
    const bool done = !(sqrt(rr) > rtol * bnorm[s]) || !isfinite(rr);
    if (threadIdx.x == 0 && (int32_t)blockIdx.x == C.ptr[s]) {
        nprec[s] += 1;
        rznew[s] = rzn;
        if (done) active[s] = 0;
    }
    if (done) return;
    const double beta = rzn / rzold[s];
    const int64_t r1 = C.end[blockIdx.x];
#pragma unroll 4
    for (int64_t i = C.begin[blockIdx.x] + threadIdx.x; i < r1; i += kCgThreads)
        p[i] = T(double(z[i]) + beta * double(p[i]));
}

}  // namespace pyhip
