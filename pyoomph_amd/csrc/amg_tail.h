// The coarse levels of the V-cycle in one workgroup per sub-problem (included by amg.hip).
//
// On levels of some hundred rows every launch of the cycle (two down, two up, one or two dense
// solves per level) takes its 3 to 5 us whatever it computes: twelve of the thirty launches of a
// GMRES iteration with a 46 000 row velocity block, some 45 of its 158 us. One workgroup takes
// a sub-problem through all of them with the vectors in LDS (24 us there; 64 sub-problems in
// FP32: 12 launches of 54 us, now 21). Bound: the wave instructions of one CU's row sums (512
// threads 29, 256 44 us); row starts in LDS and more entries in flight per lane gained
// nothing. Rows are summed in the canonical order (spmv.h) by eight lanes each and every other
// operation is the launches' own, so the results are the same bits and the first level can be
// chosen for speed (amg_tail_level).
#pragma once

constexpr int kTailThreads = 1024, kTailLevels = 8;
constexpr int kTailRows = 2, kTailAhead = 2;   // rows and entries per row a lane keeps in flight
template <typename T>
struct AmgTailLevel {
    const int32_t *rs, *col, *trs, *trow, *prs, *pcol, *cont;
    const T *vals, *w, *ptv, *pv;
    const int64_t *sub_off;
};
template <typename T>
struct AmgTail {
    AmgTailLevel<T> lv[kTailLevels + 1];   // the last one: the coarsest level (only sub_off used)
    int nl;                                // levels with a coarser one
};

// f(i, sum of val[k] x[col[k] - c0] over row i's entries) for rows i = 0 .. n - 1 of the
// rows from r0 on, x in LDS
template <typename T, typename F>
__device__ __forceinline__ void tail_rows(int n, int64_t r0, const int32_t *__restrict__ rs,
                                          const int32_t *__restrict__ col, const T *__restrict__ val, int64_t c0,
                                          const T *x, F f) {
    constexpr int NG = kTailThreads / 8, NR = kTailRows, NU = kTailAhead;
    const int lane = threadIdx.x % 8, g = threadIdx.x / 8;
    for (int ib = g; ib < n; ib += NG * NR) {
        int32_t k0[NR], k1[NR], len = 0;
        T acc[NR];
#pragma unroll
        for (int p = 0; p < NR; p++) {
            const int i = ib + p * NG;
            k0[p] = i < n ? rs[r0 + i] : 0;
            k1[p] = i < n ? rs[r0 + i + 1] : 0;
            acc[p] = T(0);
        }
#pragma unroll
        for (int p = 0; p < NR; p++) len = max(len, k1[p] - k0[p]);
        for (int32_t base = lane; base < len; base += 8 * NU) {
            int32_t cc[NR][NU];
            T vv[NR][NU];
#pragma unroll
            for (int p = 0; p < NR; p++)
#pragma unroll
                for (int u = 0; u < NU; u++) {
                    const int32_t k = k0[p] + base + 8 * u;
                    const bool in = k < k1[p];
                    cc[p][u] = in ? (int32_t)(col[k] - c0) : -1;
                    vv[p][u] = in ? val[k] : T(0);
                }
#pragma unroll
            for (int p = 0; p < NR; p++)
#pragma unroll
                for (int u = 0; u < NU; u++)
                    if (cc[p][u] >= 0) acc[p] = fmadd(vv[p][u], x[cc[p][u]], acc[p]);
        }
#pragma unroll
        for (int p = 0; p < NR; p++) {
            T v = acc[p];
            v = v + __shfl_xor(v, 4, 8);
            v = v + __shfl_xor(v, 2, 8);
            v = v + __shfl_xor(v, 1, 8);
            const int i = ib + p * NG;
            if (i < n && lane == 0) f(i, v);
        }
    }
}

// x0 = the cycle's result on level lv[0] for the right-hand side b0
template <typename T>
__global__ __launch_bounds__(kTailThreads) void amg_tail_kernel(AmgTail<T> A, const T *__restrict__ cinv,
                                                                const T *b0, T *x0,
                                                                const int32_t *__restrict__ act) {
    extern __shared__ __align__(16) unsigned char tail_mem[];
    const int s = blockIdx.x, t = threadIdx.x;
    if (act && !act[s]) return;   // the whole workgroup
    const int64_t f0 = A.lv[0].sub_off[s];
    const int n0 = (int)(A.lv[0].sub_off[s + 1] - f0);
    if (n0 == 0) return;
    T *r = (T *)tail_mem, *b = r + n0;   // a level's b and x follow each other, the next level's after them
    int l = 0, n = n0;
    int64_t f = f0;
    for (int i = t; i < n; i += kTailThreads) {
        b[i] = b0[f + i];
        b[n + i] = A.lv[0].w ? A.lv[0].w[f + i] * b[i] : T(0);   // (a coarsest level has no weights)
    }
    __syncthreads();
    // down: to the level where the sub-problem ends
    while (l < A.nl && A.lv[l].cont[s]) {
        const AmgTailLevel<T> &L = A.lv[l], &C = A.lv[l + 1];
        tail_rows<T>(n, f, L.rs, L.col, L.vals, f, b + n, [&](int i, T v) { r[i] = b[i] - v; });
        __syncthreads();
        const int64_t fc = C.sub_off[s];
        const int nc = (int)(C.sub_off[s + 1] - fc);
        T *bc = b + 2 * n;
        tail_rows<T>(nc, fc, L.trs, L.trow, L.ptv, f, r, [&](int i, T v) {
            bc[i] = v;
            if (C.w) bc[nc + i] = C.w[fc + i] * v;
        });
        __syncthreads();
        l++;
        b = bc;
        n = nc;
        f = fc;
    }
    // its dense solve (amg_chol_solve_kernel's sums), into x
    const T *X = cinv + (int64_t)s * kBottomMaxRows * kBottomMaxRows;
    if (t < n) {
        T acc = T(0);
#pragma unroll 8
        for (int j = 0; j < n; j++) acc = fmadd(X[j * kBottomMaxRows + t], b[j], acc);
        b[n + t] = acc;
    }
    __syncthreads();
    const T *xc = b + n;   // the coarser level's result
    while (l > 0) {
        const int64_t fc = f;
        l--;
        const AmgTailLevel<T> &L = A.lv[l];
        f = L.sub_off[s];
        n = (int)(L.sub_off[s + 1] - f);
        b -= 2 * n;
        T *x = b + n;
        tail_rows<T>(n, f, L.prs, L.pcol, L.pv, fc, xc, [&](int i, T v) { x[i] = x[i] + v; });
        __syncthreads();
        tail_rows<T>(n, f, L.rs, L.col, L.vals, f, x, [&](int i, T v) { r[i] = x[i] + L.w[f + i] * (b[i] - v); });
        __syncthreads();
        xc = r;
    }
    for (int i = t; i < n0; i += kTailThreads) x0[f0 + i] = xc[i];
}
