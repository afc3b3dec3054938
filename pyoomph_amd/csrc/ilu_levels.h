// ILU(0) triangular solves level by level (layout: ilu_plan.h), for the sub-problems whose
// solves do not run in one workgroup (ilu_sliced.h). Latency bound: a level of some thousand
// rows is a few dependent loads long. A thread finds its entries from the segment numbers in
// the kernel arguments, so the chain is column / factor entry -> vector entry -> sum, where
// row lists, row pointers and pivot positions took two more dependent loads; vectors stay in
// the problem's numbering, so no permutation launches are needed; the first lower level (rows
// without lower entries) is copied by the second level's launch, and a row without upper
// entries is finished by its lower level, so the first upper level has no launch either.
// Sums: a row's entries in 8 stripes combined in a fixed tree (as the spmv's rows), whatever
// the lanes: the result does not depend on the other sub-problems of a level.
#pragma once
#include "ilu_plan.h"
#include "spmv.h"

namespace pyhip {

template <typename T, int LANES>
__device__ __forceinline__ T ilu_row_sum(const IluLevel &L, int32_t row, int u, const int32_t *__restrict__ col,
                                         const T *__restrict__ val, const T *__restrict__ x) {
    constexpr int NS = 8 / LANES;
    int g = 0;
#pragma unroll
    for (int k = 1; k < kIluSegments; k++)
        if (k < L.nseg && row >= L.seg_row[k]) g = k;
    const int64_t S = (int64_t)(L.seg_row[g + 1] - L.seg_row[g]) * LANES;
    const int64_t at = L.off[g] + (int64_t)(row - L.seg_row[g]) * LANES + u;
    const int steps = L.steps[g];
    T s[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) s[j] = T(0);
    constexpr int U = LANES / 2;   // steps in flight
    for (int t = 0; t < steps; t += U) {
        int32_t c[U][NS];
        T v[U][NS], xx[U][NS];
#pragma unroll
        for (int q = 0; q < U; q++)
#pragma unroll
            for (int j = 0; j < NS; j++)
                if (t + q < steps) {
                    const int64_t k = at + ((int64_t)(t + q) * NS + j) * S;
                    c[q][j] = col[k];
                    v[q][j] = val[k];
                }
#pragma unroll
        for (int q = 0; q < U; q++)
#pragma unroll
            for (int j = 0; j < NS; j++)
                if (t + q < steps) xx[q][j] = x[c[q][j]];
#pragma unroll
        for (int q = 0; q < U; q++)
#pragma unroll
            for (int j = 0; j < NS; j++)
                if (t + q < steps) s[j] = fmadd(v[q][j], xx[q][j], s[j]);
    }
    T a;
    if constexpr (LANES == 8) a = s[0];
    else if constexpr (LANES == 4) a = s[0] + s[1];
    else a = (s[0] + s[2]) + (s[1] + s[3]);
    if constexpr (LANES >= 8) a = a + __shfl_xor(a, 4, LANES);
    if constexpr (LANES >= 4) a = a + __shfl_xor(a, 2, LANES);
    a = a + __shfl_xor(a, 1, LANES);
    return a;
}

// One level. Lower: y = v - sum of l x over the row's lower entries (x = v on the second level,
// whose columns all lie in the first; then y), and z = y / pivot for rows without upper
// entries. Upper: z = (y - sum of u z) / pivot. first: rows [0, nfirst) of the list, the
// first lower level, copied by the blocks after the level's own.
template <typename T, int LANES, bool LOWER>
__global__ __launch_bounds__(256) void ilu_level_kernel(IluLevel L, int32_t nfirst, const int32_t *__restrict__ rows,
                                                        const int32_t *__restrict__ col, const T *__restrict__ val,
                                                        const T *__restrict__ rdiag, const T *__restrict__ v,
                                                        const T *x, T *y, T *z) {
    const int64_t own = ((int64_t)L.rows * LANES + 255) / 256;
    if (LOWER && (int64_t)blockIdx.x >= own) {
        const int64_t i = ((int64_t)blockIdx.x - own) * 256 + threadIdx.x;
        if (i >= nfirst) return;
        const int32_t r = rows[i], row = r & ~kIluLast;
        const T a = v[row];
        y[row] = a;
        if (r < 0) z[row] = a * rdiag[i];
        return;
    }
    const int64_t slot = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int32_t i = (int32_t)(slot / LANES);
    const int u = (int)(slot % LANES);
    if (i >= L.rows) return;   // whole lane groups
    const int32_t r = rows[L.row0 + i], row = r & ~kIluLast;
    const T d = rdiag[L.row0 + i];
    const T rhs = LOWER ? v[row] : y[row];
    const T a = rhs - ilu_row_sum<T, LANES>(L, i, u, col, val, x);
    if (u != 0) return;
    if constexpr (LOWER) {
        y[row] = a;
        if (r < 0) z[row] = a * d;
    } else {
        z[row] = a * d;
    }
}

// Level of place q in a side's row list (nlev levels, consecutive rows)
__device__ __forceinline__ const IluLevel &ilu_level_of(const IluLevel *lev, int nlev, int32_t q) {
    int lo = 0, hi = nlev;   // lev[lo].row0 <= q < lev[hi].row0
    while (hi - lo > 1) {
        const int m = (lo + hi) >> 1;
        if (lev[m].row0 <= q) lo = m;
        else hi = m;
    }
    return lev[lo];
}

// The rows and columns of a side, once per plan; a thread per (row, stripe)
__global__ __launch_bounds__(256) void ilu_level_index_kernel(int64_t stripes, const IluLevel *__restrict__ lev, int nlev,
                                                              const int32_t *__restrict__ order,
                                                              const int32_t *__restrict__ prs,
                                                              const int32_t *__restrict__ pcol,
                                                              const int32_t *__restrict__ pdiag,
                                                              const int32_t *__restrict__ perm, bool lower,
                                                              int32_t *__restrict__ row, int32_t *__restrict__ col) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= stripes) return;
    const int32_t q = (int32_t)(t / 8), r = order[q];
    const IluLevel &L = ilu_level_of(lev, nlev, q);
    const int32_t k0 = lower ? prs[r] : pdiag[r] + 1, n = (lower ? pdiag[r] : prs[r + 1]) - k0;
    if (t % 8 == 0) row[q] = ilu_level_row(r, prs, pdiag, perm, lower);
    ilu_level_stripe(L, q - L.row0, (int)(t % 8),
                     [&](int64_t at, int k) { col[at] = ilu_level_col(r, k0, n, k, pcol, perm); });
}

// The factor of a side (0 at padding) and each row's reciprocal pivot
template <typename T>
__global__ __launch_bounds__(256) void ilu_level_fill_kernel(int64_t stripes, const IluLevel *__restrict__ lev, int nlev,
                                                             const int32_t *__restrict__ order,
                                                             const int32_t *__restrict__ prs,
                                                             const int32_t *__restrict__ pdiag, bool lower,
                                                             const T *__restrict__ lu, T *__restrict__ val,
                                                             T *__restrict__ rdiag) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= stripes) return;
    const int32_t q = (int32_t)(t / 8), r = order[q];
    const IluLevel &L = ilu_level_of(lev, nlev, q);
    const int32_t k0 = lower ? prs[r] : pdiag[r] + 1, n = (lower ? pdiag[r] : prs[r + 1]) - k0;
    if (t % 8 == 0) rdiag[q] = T(1) / lu[pdiag[r]];
    ilu_level_stripe(L, q - L.row0, (int)(t % 8),
                     [&](int64_t at, int k) { val[at] = k < n ? lu[k0 + k] : T(0); });
}

}  // namespace pyhip
