// ILU(0) triangular solves of one sub-problem in one workgroup (layout: ilu_plan.h).
//
// The level-scheduled solves need a launch per level (7 + 7 on a P2 mesh in multicolour
// order, 23 + 23 for Taylor-Hood, up to 64 + 64 in natural order), each 3-4 us however few
// rows it has, and two launches to permute. Here a workgroup of 16 waves keeps the
// sub-problem's vector in LDS (FP64: up to kIluSlicedRows rows of the CU's 160 KB), runs
// every level of both solves with a workgroup barrier in between, and reads the factor as
// slices of 64 lanes with 16-byte loads, 11 bytes an entry (one CU streams 145 GB/s in
// 16-byte loads, 73 GB/s in 8-byte ones).
// Bound: the one CU's load bandwidth on large sub-problems, the barrier and LDS latency of
// the levels on small ones.
// Sums: a row's entries go to its lanes round robin, each lane keeps two running sums,
// combined in a fixed order and then across the lanes by an xor tree: a sub-problem's result
// depends on its own plan only.
#pragma once
#include "ilu_plan.h"
#include "spmv.h"

namespace pyhip {

constexpr int kIluSlicedThreads = 64 * kIluSliceWaves;
// rows whose FP64 vector (and the zero behind it) fits the CU's LDS
constexpr int kIluSlicedRows = 20000;
template <typename T>
constexpr size_t ilu_sliced_lds(int rows) {
    return (size_t)(rows + 1) * sizeof(T);
}

template <typename T>
struct IluSlicedDev {
    const int32_t *nlev, *chunk0;
    const uint16_t *idx;
    const T *val;    // factor entries in chunk order
    const T *rdiag;  // [chunks * 64] upper side: the reciprocal pivot of each lane's row
};

// A workgroup barrier that orders LDS accesses only: the loads of a wave's next tasks stay in
// flight across it (a full __syncthreads waits for them).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename T> struct IluPair { typedef T type __attribute__((ext_vector_type(2))); };
typedef uint32_t ilu_u32x4 __attribute__((ext_vector_type(4)));

// One chunk in registers
template <typename T>
struct IluChunkRegs {
    ilu_u32x4 ix;                       // 16-bit columns, two per word; word 3: row, mark
    typename IluPair<T>::type v[kIluChunk / 2];
    T d;
};

// One triangular solve in place on x (LDS, complete before the call and, after the last
// level's barrier, after it); every thread of the workgroup calls it. A wave walks its
// stream of chunks kIluDepth ahead: the loads do not depend on x, so they are in flight
// across the levels' barriers. Every fetch issues the same loads (past the stream's end,
// those of its last chunk again), so that the waits count exactly.
template <typename T, bool LOWER>
__device__ __forceinline__ void ilu_sliced_solve(const IluSlicedDev<T> &F, int t, T *x) {
    using P = typename IluPair<T>::type;
    const uint32_t lane = threadIdx.x & 63;
    const int wave = t * kIluSliceWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int32_t c0 = __builtin_amdgcn_readfirstlane(F.chunk0[wave]);
    const int32_t c1 = __builtin_amdgcn_readfirstlane(F.chunk0[wave + 1]);
    const int nlev = __builtin_amdgcn_readfirstlane(F.nlev[t]);
    int lev = 0;   // barriers passed: the levels below lev are complete
    if (c0 < c1) {
        IluChunkRegs<T> A[kIluDepth];
        auto fetch = [&](int k, int32_t ch) {
            ch = min(ch, c1 - 1);
            A[k].ix = ((const ilu_u32x4 *)F.idx + (int64_t)ch * kIluSliceLanes)[lane];
            const P *v = (const P *)F.val + (int64_t)ch * (kIluChunkVal / 2);
#pragma unroll
            for (int j = 0; j < kIluChunk / 2; j++) A[k].v[j] = (v + j * kIluSliceLanes)[lane];
            if constexpr (!LOWER) A[k].d = (F.rdiag + (int64_t)ch * kIluSliceLanes)[lane];
        };
#pragma unroll
        for (int k = 0; k < kIluDepth; k++) fetch(k, c0 + k);
        T s0 = T(0), s1 = T(0);
        for (int32_t ch = c0; ch < c1; ch += kIluDepth) {
#pragma unroll
            for (int k = 0; k < kIluDepth; k++) {
                const uint32_t mark = (uint32_t)__builtin_amdgcn_readfirstlane(A[k].ix[3]) >> 16;
                for (const int l = mark & 0xfff; lev < l; lev++) lds_barrier();
                const uint32_t row = A[k].ix[3] & 0xffff;
                const int lanes = 1 << ((mark >> 12) & 7);
                const bool own = row != kIluNoRow && (lane & (lanes - 1)) == 0;
                const T rhs = own ? x[row] : T(0);
#pragma unroll
                for (int j = 0; j < kIluChunk / 2; j++) {
                    const uint32_t c = A[k].ix[j];
                    s0 = fmadd(A[k].v[j].x, x[c & 0xffff], s0);
                    s1 = fmadd(A[k].v[j].y, x[c >> 16], s1);
                }
                if (!(mark >> 15)) {
                    T acc = s0 + s1;
                    for (int off = lanes >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
                    if (own) x[row] = LOWER ? rhs - acc : (rhs - acc) * A[k].d;
                    s0 = s1 = T(0);
                }
                fetch(k, ch + k + kIluDepth);
            }
        }
    }
    for (; lev < nlev; lev++) lds_barrier();   // every wave passes nlev barriers
}

// z = (L U)^-1 v for the handled sub-problems, one workgroup each; dynamic LDS of
// (max rows + 1) values. Sub-problems with act[sub] == 0 (act given) keep their z.
template <typename T>
__global__ __launch_bounds__(kIluSlicedThreads) void ilu_sliced_apply_kernel(
    const int32_t *__restrict__ subs, const int32_t *__restrict__ row0, const int32_t *__restrict__ rows,
    const int32_t *__restrict__ perm, IluSlicedDev<T> lo, IluSlicedDev<T> up, const T *__restrict__ v,
    T *__restrict__ z, const int32_t *__restrict__ act) {
    extern __shared__ __align__(16) unsigned char ilu_lds[];
    T *x = (T *)ilu_lds;
    const int t = blockIdx.x;
    if (act && !act[subs[t]]) return;   // the whole workgroup leaves together
    const int n = rows[t];
    const int32_t *pm = perm + row0[t];
    constexpr int U = 8;   // rows of a thread loaded together
    for (int b = threadIdx.x; b < n; b += U * kIluSlicedThreads) {
        int32_t q[U];
        T w[U];
#pragma unroll
        for (int u = 0; u < U; u++) q[u] = b + u * kIluSlicedThreads < n ? pm[b + u * kIluSlicedThreads] : -1;
#pragma unroll
        for (int u = 0; u < U; u++) w[u] = q[u] >= 0 ? v[q[u]] : T(0);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (q[u] >= 0) x[b + u * kIluSlicedThreads] = w[u];
    }
    if (threadIdx.x == 0) x[n] = T(0);
    __syncthreads();
    ilu_sliced_solve<T, true>(lo, t, x);
    ilu_sliced_solve<T, false>(up, t, x);
    for (int b = threadIdx.x; b < n; b += U * kIluSlicedThreads) {
        int32_t q[U];
#pragma unroll
        for (int u = 0; u < U; u++) q[u] = b + u * kIluSlicedThreads < n ? pm[b + u * kIluSlicedThreads] : -1;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (q[u] >= 0) z[q[u]] = x[b + u * kIluSlicedThreads];
    }
}

// The chunks' columns, rows and marks, once per plan; a thread per (chunk, lane)
__global__ __launch_bounds__(256) void ilu_sliced_index_kernel(int64_t lanes, const IluChunk *__restrict__ chunk,
                                                               const int32_t *__restrict__ order,
                                                               const int32_t *__restrict__ prs,
                                                               const int32_t *__restrict__ pcol,
                                                               const int32_t *__restrict__ pdiag,
                                                               const int32_t *__restrict__ row0,
                                                               const int32_t *__restrict__ rows, bool lower,
                                                               ilu_u32x4 *__restrict__ idx) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= lanes) return;
    const IluChunk C = chunk[k / kIluSliceLanes];
    const IluLane L = ilu_chunk_lane(C, (int)(k % kIluSliceLanes), order, prs, pdiag, lower);
    const int32_t r0 = row0[C.slot], dummy = rows[C.slot];
    uint32_t c[kIluChunk];
#pragma unroll
    for (int j = 0; j < kIluChunk; j++) c[j] = (uint32_t)(L.e(j) < L.len ? pcol[L.k0 + L.e(j)] - r0 : dummy);
    const uint32_t row = L.row >= 0 ? (uint32_t)(L.row - r0) : (uint32_t)kIluNoRow;
    idx[k] = ilu_u32x4{c[0] | c[1] << 16, c[2] | c[3] << 16, c[4] | c[5] << 16, row | (uint32_t)C.mark << 16};
}

// The factor in chunk order (0 at padding) and, with rdiag, each lane's reciprocal pivot
template <typename T>
__global__ __launch_bounds__(256) void ilu_sliced_fill_kernel(int64_t lanes, const IluChunk *__restrict__ chunk,
                                                              const int32_t *__restrict__ order,
                                                              const int32_t *__restrict__ prs,
                                                              const int32_t *__restrict__ pdiag, bool lower,
                                                              const T *__restrict__ lu, T *__restrict__ val,
                                                              T *__restrict__ rdiag) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= lanes) return;
    const int64_t c = k / kIluSliceLanes;
    const int lane = (int)(k % kIluSliceLanes);
    const IluLane L = ilu_chunk_lane(chunk[c], lane, order, prs, pdiag, lower);
    using P = typename IluPair<T>::type;
    P *v = (P *)val + c * (kIluChunkVal / 2) + lane;
#pragma unroll
    for (int j = 0; j < kIluChunk; j += 2) {
        P q;
        q.x = L.e(j) < L.len ? lu[L.k0 + L.e(j)] : T(0);
        q.y = L.e(j + 1) < L.len ? lu[L.k0 + L.e(j + 1)] : T(0);
        v[j / 2 * kIluSliceLanes] = q;
    }
    if (rdiag) rdiag[k] = L.row >= 0 ? T(1) / lu[pdiag[L.row]] : T(0);
}

}  // namespace pyhip
