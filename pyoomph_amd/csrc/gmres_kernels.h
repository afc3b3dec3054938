// Orthogonalisation of one GMRES iteration in four launches (classical Gram-Schmidt twice,
// norm, Givens rotation), per sub-problem:
//   1 gs_dot     partials of d1_j = (V_j, w)
//   2 gs_update  w -= sum_j d1_j V_j, then partials of d2_j = (V_j, w)
//   3 gs_update  w -= sum_j d2_j V_j, then partials of (w, w)
//   4 gs_finish  V_{k+1} = w / |w| and, in a sub-problem's first block, its Givens step
// One block of 1024 threads owns a chunk of 256, 512 or 1024 rows of one sub-problem (by the
// sub-problem's rows, so that small systems still spread over many CUs and a sub-problem's
// sums are the same alone and in any batch). The partials of a reduction are summed by every
// block that needs the result (lane-strided over the sub-problem's chunks, then an xor tree)
// instead of by a launch of its own, up to kGsFusedPartials values a block; beyond, a launch of
// gs_reduce adds them in the same order. Launches with nothing but such sums, counters and
// single-thread loops took 25 us of an iteration.
// Bound: reading V three times per iteration (once per pass and a second time in pass 2, from
// L2 where the resident blocks' chunks of V fit it: 64 blocks an XCD, so up to some 30 vectors of
// 256 rows), in 16-byte loads; launch latency for small systems.
#pragma once
#include "common.h"

namespace pyhip {

constexpr int kGsThreads = 1024, kGsWaves = kGsThreads / 64;
constexpr int kGsMaxRows = 1024;
// Most partials (chunks x vectors) of a sub-problem that every block adds up for itself. 300
// iterations of GMRES(100) / GMRES(30), summed by the blocks and by launches: 16129 rows (64
// chunks) 10.9 / 9.2 and 11.6 / 10.9 ms; 64516 (127) 13.7 / 9.5 and 13.3 / 10.3; 129600 (254)
// 20.2 / 11.1 and 18.7 / 11.7; 622521 (608) 79.9 / 32.9 and 70.2 / 30.8.
constexpr int kGsFusedPartials = 8192;

inline int gs_chunk_rows(int64_t rows) { return rows <= 32768 ? 256 : rows <= 131072 ? 512 : 1024; }

// two rows of a vector; rows start anywhere, so only the element's alignment is assumed
template <typename T> struct GsPair {
    typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};

struct GsChunks {
    const int64_t *begin, *end;   // rows of each chunk
    const int32_t *sub;           // its sub-problem
    const int32_t *ptr;           // [nsub + 1] chunks of each sub-problem
    int64_t count;
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// sums over the chunks of sub-problem s of part[j][chunk] for the vectors j of this wave
// (j = wave, wave + kGsWaves, ...), into h[j] (LDS) and, in the sub-problem's first block,
// out[j][s]. With `reduced` h[j] is out[j][s] (summed by a launch of its own).
__device__ __forceinline__ void gs_coefficients(int nvec, int nsub, int s, const GsChunks &C,
                                                const double *__restrict__ part, double *__restrict__ out,
                                                bool reduced, double *h) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t c0 = C.ptr[s], c1 = C.ptr[s + 1];
    if (reduced) {
        for (int j = threadIdx.x; j < nvec; j += kGsThreads) h[j] = out[(int64_t)j * nsub + s];
        return;
    }
    const bool first = (int32_t)blockIdx.x == c0;
    for (int j = wave; j < nvec; j += kGsWaves) {
        double a = 0.0;
        for (int32_t c = c0 + lane; c < c1; c += 64) a += part[(int64_t)j * C.count + c];
        a = wave_sum(a);
        if (lane == 0) {
            h[j] = a;
            if (first) out[(int64_t)j * nsub + s] = a;
        }
    }
}

// part[j][chunk] = sum over the chunk's rows of V_j w, w in LDS (zero past the rows); wave q
// takes the vectors q, q + kGsWaves, ...; lanes take pairs of rows
template <typename T>
__device__ __forceinline__ void gs_dots(int nvec, const T *__restrict__ V, int64_t ldv, int64_t r0, int rows,
                                        const T *w, double *__restrict__ part, int64_t count) {
    using P = typename GsPair<T>::type;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int j = wave; j < nvec; j += kGsWaves) {
        const T *v = V + (int64_t)j * ldv + r0;
        double a = 0.0, b = 0.0;
#pragma unroll 4
        for (int i = 2 * lane; i + 1 < rows; i += 128) {
            const P x = *(const P *)(v + i);
            a += double(x.x) * double(w[i]);
            b += double(x.y) * double(w[i + 1]);
        }
        if ((rows & 1) && lane == 0) a += double(v[rows - 1]) * double(w[rows - 1]);
        a = wave_sum(a + b);
        if (lane == 0) part[(int64_t)j * count + blockIdx.x] = a;
    }
}

template <typename T>
__global__ __launch_bounds__(kGsThreads) void gs_dot_kernel(int nvec, const T *__restrict__ V, int64_t ldv,
                                                            const T *__restrict__ w, GsChunks C,
                                                            const int32_t *__restrict__ active,
                                                            double *__restrict__ part) {
    __shared__ T wl[kGsMaxRows];
    const int s = C.sub[blockIdx.x];
    if (!active[s]) return;
    const int64_t r0 = C.begin[blockIdx.x];
    const int rows = (int)(C.end[blockIdx.x] - r0);
    if ((int)threadIdx.x < rows) wl[threadIdx.x] = w[r0 + threadIdx.x];
    __syncthreads();
    gs_dots<T>(nvec, V, ldv, r0, rows, wl, part, C.count);
}

// w -= sum_j h_j V_j, h summed from part_in; then, NORM: part_out[chunk] = (w, w), else
// part_out[j][chunk] = (V_j, w). The rows of a chunk are taken in pairs by kGsThreads / pairs
// groups of threads, group g adding the vectors g, g + groups, ...; the groups' sums are added
// in group order.
template <typename T, bool NORM>
__global__ __launch_bounds__(kGsThreads) void gs_update_kernel(int nvec, int nsub, const T *__restrict__ V, int64_t ldv,
                                                               T *__restrict__ w, GsChunks C,
                                                               const int32_t *__restrict__ active,
                                                               const double *__restrict__ part_in,
                                                               double *__restrict__ coef, int reduced,
                                                               double *__restrict__ part_out) {
    using P = typename GsPair<T>::type;
    extern __shared__ __align__(16) unsigned char gs_lds[];
    double *red = (double *)gs_lds;                          // [groups][rows of a chunk]: 2 * kGsThreads
    T *wl = (T *)(red + 2 * kGsThreads);                     // [rows]
    double *h = (double *)(wl + kGsMaxRows);                 // [nvec]
    const int s = C.sub[blockIdx.x];
    if (!active[s]) return;   // the whole block
    const int64_t r0 = C.begin[blockIdx.x];
    const int rows = (int)(C.end[blockIdx.x] - r0);
    gs_coefficients(nvec, nsub, s, C, part_in, coef, reduced != 0, h);
    __syncthreads();
    // pairs of rows, rounded up to a power of two so that the groups are whole waves
    int np = 64;
    while (2 * np < rows) np *= 2;
    const int groups = kGsThreads / np, g = threadIdx.x / np, i = 2 * (threadIdx.x & (np - 1));
    double a = 0.0, b = 0.0;
    if (i + 1 < rows) {
        const T *v = V + r0 + i;
#pragma unroll 8
        for (int j = g; j < nvec; j += groups) {
            const P x = *(const P *)(v + (int64_t)j * ldv);
            a += h[j] * double(x.x);
            b += h[j] * double(x.y);
        }
    } else if (i < rows) {
        const T *v = V + r0 + i;
        for (int j = g; j < nvec; j += groups) a += h[j] * double(v[(int64_t)j * ldv]);
    }
    red[g * 2 * np + i] = a;
    red[g * 2 * np + i + 1] = b;
    __syncthreads();
    double ww = 0.0;
    if ((int)threadIdx.x < rows) {
        double acc = 0.0;
        for (int q = 0; q < groups; q++) acc += red[q * 2 * np + threadIdx.x];
        const T x = T(double(w[r0 + threadIdx.x]) - acc);
        w[r0 + threadIdx.x] = x;
        wl[threadIdx.x] = x;
        ww = double(x) * double(x);
    }
    if constexpr (NORM) {
        // waves, then the waves' sums in order
        ww = wave_sum(ww);
        if ((threadIdx.x & 63) == 0) h[threadIdx.x >> 6] = ww;   // h is read no more
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = 0.0;
            for (int q = 0; q < kGsWaves; q++) t += h[q];
            part_out[blockIdx.x] = t;
        }
    } else {
        __syncthreads();
        gs_dots<T>(nvec, V, ldv, r0, rows, wl, part_out, C.count);
    }
}
inline size_t gs_update_lds(int nvec, size_t esize) {
    return 2 * kGsThreads * sizeof(double) + kGsMaxRows * esize +
           (size_t)(nvec > kGsWaves ? nvec : kGsWaves) * sizeof(double);
}

// out[j][s] = sum over the chunks of s of part[j][chunk] (above kGsFusedPartials), one wave
// per (j, s)
__global__ __launch_bounds__(64) void gs_reduce_kernel(int nsub, GsChunks C, const int32_t *__restrict__ active,
                                                       const double *__restrict__ part, double *__restrict__ out) {
    const int j = blockIdx.x / nsub, s = blockIdx.x % nsub;
    if (!active[s]) return;
    double a = 0.0;
    for (int32_t c = C.ptr[s] + (int32_t)threadIdx.x; c < C.ptr[s + 1]; c += 64) a += part[(int64_t)j * C.count + c];
    a = wave_sum(a);
    if (threadIdx.x == 0) out[(int64_t)j * nsub + s] = a;
}

// V_{k+1} = w / |w| with |w|^2 summed from part; the first block of a sub-problem then takes
// its Givens step: column k of the Hessenberg is h_i = d1_i + d2_i (i <= k) and |w|, rotated by
// the earlier rotations; g and the flags as the rotation leaves them. m: stride of the
// Hessenberg / Givens arrays, mr <= m: the restart length (the cycle ends after column mr - 1).
// Other blocks may see active[s] already cleared: the vector they then skip is read by nobody.
template <typename T>
__global__ __launch_bounds__(kGsThreads) void gs_finish_kernel(
    int nsub, int m, int mr, int k, const T *__restrict__ w, T *__restrict__ vnext, GsChunks C,
    const double *__restrict__ part, const double *__restrict__ d1, const double *__restrict__ d2,
    double *__restrict__ H, double *__restrict__ cs, double *__restrict__ sn, double *__restrict__ g,
    const double *__restrict__ bnorm, double tol, int32_t *active, int32_t *__restrict__ kcols) {
    extern __shared__ __align__(16) unsigned char gs_lds[];
    double *hl = (double *)gs_lds, *cl = hl + m + 1, *sl = cl + m + 1;   // [k + 1] each
    __shared__ double n2;
    const int s = C.sub[blockIdx.x];
    __shared__ int run;
    if (threadIdx.x == 0) run = active[s];   // one read: every thread of the block takes the same way
    __syncthreads();
    if (!run) return;
    const int32_t c0 = C.ptr[s], c1 = C.ptr[s + 1];
    const bool first = (int32_t)blockIdx.x == c0;
    if (threadIdx.x < 64) {
        double a = 0.0;
        for (int32_t c = c0 + (int32_t)threadIdx.x; c < c1; c += 64) a += part[c];
        a = wave_sum(a);
        if (threadIdx.x == 0) n2 = a;
    }
    if (first)
        for (int i = threadIdx.x; i <= k; i += kGsThreads) {
            hl[i] = d1[(int64_t)i * nsub + s] + d2[(int64_t)i * nsub + s];
            if (i < k) {
                cl[i] = cs[(int64_t)s * m + i];
                sl[i] = sn[(int64_t)s * m + i];
            }
        }
    __syncthreads();
    const double nr = sqrt(n2);
    const int64_t r0 = C.begin[blockIdx.x], row = r0 + threadIdx.x;
    if (row < C.end[blockIdx.x]) vnext[row] = nr > 0.0 ? T(double(w[row]) / nr) : T(0);
    if (!first) return;
    if (threadIdx.x == 0) {
        double hi = hl[0];
#pragma unroll 4
        for (int i = 0; i < k; i++) {
            const double hn = hl[i + 1], c = cl[i], v = sl[i];
            hl[i] = c * hi + v * hn;
            hi = -v * hi + c * hn;
        }
        const double den = hypot(hi, nr);
        double c = 1.0, v = 0.0;
        if (den > 0.0) {
            c = hi / den;
            v = nr / den;
        }
        cs[(int64_t)s * m + k] = c;
        sn[(int64_t)s * m + k] = v;
        hl[k] = den;
        double *gs = g + (int64_t)s * (m + 1);
        const double gk = gs[k], gn = -v * gk;
        gs[k + 1] = gn;
        gs[k] = c * gk;
        kcols[s] = k + 1;
        if (!(fabs(gn) > tol * bnorm[s]) || nr == 0.0 || den == 0.0 || !isfinite(gn) || k + 1 == mr) active[s] = 0;
    }
    __syncthreads();
    double *Hs = H + (int64_t)s * (m + 1) * m;
    for (int i = threadIdx.x; i <= k; i += kGsThreads) Hs[(int64_t)i * m + k] = hl[i];
}

// y = R^-1 g, R the rotated Hessenberg, column by column in one wave per sub-problem; y and,
// up to kGsBackCols columns, R's packed upper triangle in LDS (else read from memory).
constexpr int kGsBackCols = 180;
inline size_t gs_backsolve_lds(int m, int mr) {
    const int c = mr < kGsBackCols ? mr : kGsBackCols;
    return ((size_t)m + (size_t)c * (c + 1) / 2) * sizeof(double);
}
__global__ __launch_bounds__(64) void gs_backsolve_kernel(int m, const double *__restrict__ H,
                                                          const double *__restrict__ g,
                                                          const int32_t *__restrict__ kcols, int lds_cols,
                                                          double *__restrict__ y) {
    extern __shared__ __align__(16) unsigned char gs_lds[];
    double *yl = (double *)gs_lds, *R = yl + m;         // column j of R at j (j + 1) / 2
    const int s = blockIdx.x, lane = threadIdx.x;
    const double *Hs = H + (int64_t)s * (m + 1) * m;
    const int k = kcols[s];
    const bool in_lds = k <= lds_cols;
    for (int i = lane; i < m; i += 64) yl[i] = i < k ? g[(int64_t)s * (m + 1) + i] : 0.0;
    if (in_lds)
        for (int i = 0; i < k; i++)
            for (int j = i + lane; j < k; j += 64) R[j * (j + 1) / 2 + i] = Hs[(int64_t)i * m + j];
    __syncthreads();
    for (int j = k - 1; j >= 0; j--) {
        const double d = in_lds ? R[j * (j + 1) / 2 + j] : Hs[(int64_t)j * m + j];
        const double v = d != 0.0 ? yl[j] / d : 0.0;
        __syncthreads();
        if (lane == 0) yl[j] = v;
        for (int i = lane; i < j; i += 64) yl[i] -= (in_lds ? R[j * (j + 1) / 2 + i] : Hs[(int64_t)i * m + j]) * v;
        __syncthreads();
    }
    for (int i = lane; i < m; i += 64) y[(int64_t)s * m + i] = yl[i];
}

}  // namespace pyhip
