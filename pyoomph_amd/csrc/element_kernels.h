// Batched element residual / Jacobian / parameter-derivative kernels.
//
// Included by elements_f64.hip (built with -ffp-contract=off: the FP64 kernels execute
// exactly the written operation order, the same order as the CPU restatement of the
// generated element code) and elements_f32.hip (FP32, contraction allowed).
//
// What each thread computes follows the code pyoomph generates per element
// (src/codegen.cpp:3912-4109, 2015-2257; accumulation macros src/jitbridge_nohang.h:
// 23-50): integration-point loop, geometry as BulkElementBase::fill_shape_info_at_s
// (src/elements.cpp:3593-3700, 3800-3840, 3960-3990) with weight*det
// (src/elements.cpp:4564-4575), field interpolation, then the test-function row and its
// shape-function columns, skipping pinned equations (local_eqn < 0).
//
// Residuals and Jacobians of triangles, bricks and Taylor-Hood elements have kernels of their
// own further down (a thread, nine lanes, a thread per node); quadrilaterals, parameter
// derivatives, mass matrices and Hessian products take the general ones.
//
// Mapping of the general ones (one workgroup = a block of elements, 64-wide waves):
//   thread = (element, slot row i) in phase B and (element, integration point) in
//   phase A; EPB = 256 / max(NS, points per chunk) elements per workgroup.
//   Per element the nodal coordinates, slot values, equations and auxiliary field are
//   staged once in LDS (coalesced slot-major gathers). Per integration point, one thread
//   computes the geometry (tangents, metric inverse, w*det, dx_shape of every node) and
//   the interpolated fields once into LDS; then every thread runs its residual entry and
//   Jacobian row over the points, reading them as LDS broadcasts.
//   Reference-element tables (weights, psi, dpsi/ds) are read with uniform indices, so
//   they come through the scalar cache.
// Output: element vectors Er[e][i] and matrices Ej[e][i][j] in slot numbering; the
// deterministic gather (scatter.hip) sums them into the residual and the CSR values.
#pragma once
#include <type_traits>

#include "common.h"
#include "element_common.h"

namespace pyhip {

// Taylor-Hood Q2/Q1 slot layout = oomph local dof order (node-major, value-minor):
// node 0: ux uy p | 1: ux uy | 2: ux uy p | 3,4,5: ux uy | 6: ux uy p | 7: ux uy | 8: ux uy p
__device__ __constant__ const int8_t kTHSlotNode[22] = {0, 0, 0, 1, 1, 2, 2, 2, 3, 3, 4,
                                                        4, 5, 5, 6, 6, 6, 7, 7, 8, 8, 8};
__device__ __constant__ const int8_t kTHSlotKind[22] = {0, 1, 2, 0, 1, 0, 1, 2, 0, 1, 0,
                                                        1, 0, 1, 0, 1, 2, 0, 1, 0, 1, 2};
__device__ __constant__ const int8_t kTHSlotP[22] = {-1, -1, 0,  -1, -1, -1, -1, 1,  -1, -1, -1,
                                                     -1, -1, -1, -1, -1, 2,  -1, -1, -1, -1, 3};
// velocity-x slot of each node (velocity-y is the next slot)
__device__ __constant__ const int8_t kTHNodeSlot[9] = {0, 3, 5, 8, 10, 12, 14, 17, 19};

// Scalar weak forms (Poisson / Bratu / reaction-diffusion): slot = node.
// Phase A (per chunk of integration points): thread t of an element computes points
// q = t, t + NS, ... of the chunk: geometry, dx_shape of all nodes, u, grad u and the
// source term and its derivative. Phase B: thread = test row i, accumulates its residual
// and Jacobian row over the chunk's points in increasing point order.

constexpr int kTriThreads = 128;   // elements per workgroup of tri_element_kernel

// Triangles take a thread per element from this many elements on (-1: never). Below, a thread
// per row fills the chip better. FP64, row and element: P2 matrices 10.4 and 12.2 us on 512
// elements, 12.2 and 14.0 on 8192, 21.6 both ways on 32768, 36.8 and 24.3 on 80000; P2
// residuals 6.4 and 9.6 on 3200, 10.1 and 10.6 on 32768, 20.1 and 17.1 on 80000; P1 residuals 4.1
// and 4.4 on 18432, 8.1 and 7.5 on 80000; P1 matrices never slower; Poisson with its
// exponentials per point: matrices 31.6 and 32.8 on 52000, 41.9 and 32.8 on 81000, residuals
// 20.2 and 25.5, 28.1 and 27.9. Both kernels give the same FP64 bits. In FP32 contraction is the
// compiler's choice, so one kernel serves every size and a sub-problem has the same bits alone and
// in a batch: an element per thread (8.8 us both ways on 512 elements, 23.3 and 19.3 on 80000),
// for Poisson a row per thread (9.4 and 12.2 us, 27.1 and 26.7).
template <typename T, int KIND, int FORM>
constexpr int tri_min_elements(bool jac) {
    if (sizeof(T) == 4) return FORM == PYHIP_FORM_POISSON ? -1 : 0;
    if (FORM == PYHIP_FORM_POISSON) return jac ? 65536 : 81920;
    return jac ? (KIND == ELEM_TRI_P1 ? 0 : 32768) : 65536;
}

// Bricks that hex_element_kernel takes, n of a launch; the others a thread per row, in FP64 the
// same bits. A wave's points are a chain of its own, so that few bricks take longer: FP64 matrices, row
// and wave: 56 and 90 us for 1 brick, 94 and 93 for 8, 120 and 101 for 512; FP64 residuals 22 and
// 17 us for 1 (its points in one round, as those of 2), 22 and 25 for 8, 25 and 30 for 512 to 2197,
// 46 and 30 for 2744: the row kernel's workgroups hold 9 bricks, 2304 on the 256 CUs at once.
// In FP32 one kernel serves every size (a sub-problem has the same bits alone and in a batch).
template <typename T>
constexpr bool hex_takes(int n, bool jac) {
    return sizeof(T) == 4 || (jac ? n >= 8 : n <= 2 || n > 2304);
}

// TR: the form has a time derivative (a.transient); HV: the matrix output is the
// Hessian-vector product sum_k dJ_ij/du_k y_k = int d2src (sum_k y_k psi_k) psi_j psi_i
// (d2src: Bratu -lambda e^u, reaction-diffusion 6u, Poisson 0), symmetric in i, j and k,
// so the transposed product (a.htr) is the same matrix. Separate instantiations keep the
// steady kernels' LDS and registers.
template <typename T, int KIND, int FORM, bool TR, bool HV>
__global__ __launch_bounds__(256) void scalar_element_kernel(ElemArgs<T> a) {
    using Tr = ElemTraits<KIND>;
    constexpr int NN = Tr::NN, DIM = Tr::DIM, NQ = Tr::NQ, NS = NN;
    constexpr int EPB = scalar_epb<KIND>();
    constexpr int QC = ScalarChunk<KIND>::QC;
    // per point: src, dsrc, grad u[, du/dt][, d2src, y]
    constexpr int NQV = 2 + DIM + (TR ? 1 : 0) + (HV ? 2 : 0);
    constexpr int QT = 2 + DIM, QH = 2 + DIM + (TR ? 1 : 0);
    __shared__ T sX[EPB][NN][DIM];
    __shared__ T sU[EPB][NN];
    __shared__ T sH[TR ? EPB : 1][NN];   // history combination tw1 u(t-1) + tw2 u(t-2) per node
    __shared__ T sY[HV ? EPB : 1][NN];   // Hessian-vector product direction per node
    __shared__ T sF[FORM == PYHIP_FORM_REACTION_DIFFUSION ? EPB : 1][NN];
    __shared__ int sEq[EPB][NS];
    __shared__ T sW[EPB][QC];
    __shared__ T sDx[EPB][QC][NN][DIM];
    __shared__ T sQ[EPB][QC][NQV];

    const int le = threadIdx.x / NS;        // element within block
    const int row = threadIdx.x % NS;       // slot row of this thread
    const int e = a.e0 + (int)blockIdx.x * EPB + le;
    const bool active = (le < EPB) && (e < a.e1);

    if (active) {
        const int node = a.conn[(int64_t)row * a.nel + e];
        const int eq = a.seqn[(int64_t)row * a.nel + e];
#pragma unroll
        for (int d = 0; d < DIM; d++) sX[le][row][d] = T(a.coords[(int64_t)node * 3 + d]);
        sU[le][row] = T(eq >= 0 ? a.dofs[eq] : a.pinned[(int64_t)node * a.nvalue]);
        if constexpr (FORM == PYHIP_FORM_REACTION_DIFFUSION) sF[le][row] = T(a.aux[node]);
        if constexpr (TR) {
            const double pin = a.pinned[(int64_t)node * a.nvalue];
            const double u1 = eq >= 0 ? a.hist1[eq] : pin, u2 = eq >= 0 ? a.hist2[eq] : pin;
            sH[le][row] = T(a.tw1 * u1 + a.tw2 * u2);
        }
        if constexpr (HV) sY[le][row] = T(eq >= 0 ? a.hvec[eq] : 0.0);
        sEq[le][row] = eq;
    }
    __syncthreads();

    // phase-A thread: point qa of the current chunk of element la
    const int la = threadIdx.x / QC, qa = threadIdx.x % QC;
    const int ea = a.e0 + (int)blockIdx.x * EPB + la;
    const bool active_a = (la < EPB) && (ea < a.e1);
    T par0 = T(0);
    const double *par = nullptr;
    if (active_a) {
        par = a.params + (int64_t)a.sub[ea] * a.pstride;
        par0 = T(par[0]);
    }
    const bool myrow = active && sEq[le][row] >= 0;
    T Racc = T(0);
    T Jacc[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) Jacc[j] = T(0);

    for (int q0 = 0; q0 < NQ; q0 += QC) {
        // ---- phase A: per-point quantities (element la, point q0 + qa)
        if (active_a && q0 + qa < NQ) {
            {
                const int le = la, qq = qa;
                const int q = q0 + qq;
                const T *D = a.tab->dpsi + q * NN * DIM;
                const T *P = a.tab->psi + q * NN;
                const T W = point_geometry<T, NN, DIM>(sX[le], D, a.tab->w[q], sDx[le][qq]);
                sW[le][qq] = W;
                T u = T(0);
#pragma unroll
                for (int l = 0; l < NN; l++) u = u + sU[le][l] * P[l];
#pragma unroll
                for (int i = 0; i < DIM; i++) {
                    T sacc = T(0);
#pragma unroll
                    for (int l = 0; l < NN; l++) sacc = sacc + sU[le][l] * sDx[le][qq][l][i];
                    sQ[le][qq][2 + i] = sacc;
                }
                T src = T(0), dsrc = T(0);
                if constexpr (FORM == PYHIP_FORM_POISSON) {
                    T x = T(0), y = T(0);
#pragma unroll
                    for (int l = 0; l < NN; l++) x = x + sX[le][l][0] * P[l];
#pragma unroll
                    for (int l = 0; l < NN; l++) y = y + sX[le][l][1] * P[l];
                    T f = T(0);
                    const int ng = (int)par[0];  // Gaussians follow as (cx, cy, w, a)
                    for (int k = 1; k < 1 + 4 * ng; k += 4) {
                        T ddx = x - T(par[k + 0]), ddy = y - T(par[k + 1]);
                        T r2 = ddx * ddx + ddy * ddy;
                        T wk = T(par[k + 2]);
                        f = f + T(par[k + 3]) * texp(-r2 / (wk * wk));
                    }
                    src = -f;
                } else if constexpr (FORM == PYHIP_FORM_BRATU) {
                    T ev = texp(u);
                    if (a.deriv) {
                        src = -ev;
                        dsrc = -ev;
                    } else {
                        src = -par0 * ev;
                        dsrc = -par0 * ev;
                    }
                } else {
                    T f = T(0);
#pragma unroll
                    for (int l = 0; l < NN; l++) f = f + sF[le][l] * P[l];
                    src = u * u * u - f;
                    dsrc = T(3) * (u * u);
                }
                sQ[le][qq][0] = src;
                sQ[le][qq][1] = dsrc;
                if constexpr (TR) {
                    T hq = T(0);
#pragma unroll
                    for (int l = 0; l < NN; l++) hq = hq + sH[le][l] * P[l];
                    sQ[le][qq][QT] = T(a.tw0) * u + hq;
                }
                if constexpr (HV) {
                    T yq = T(0);
#pragma unroll
                    for (int l = 0; l < NN; l++) yq = yq + sY[le][l] * P[l];
                    T d2 = T(0);
                    if constexpr (FORM == PYHIP_FORM_BRATU) d2 = -par0 * texp(u);
                    else if constexpr (FORM == PYHIP_FORM_REACTION_DIFFUSION) d2 = T(6) * u;
                    sQ[le][qq][QH] = d2;
                    sQ[le][qq][QH + 1] = yq;
                }
            }
        }
        __syncthreads();
        // ---- phase B: this thread's residual entry and Jacobian row
        if (myrow) {
            for (int qq = 0; qq < QC && q0 + qq < NQ; qq++) {
                const int q = q0 + qq;
                const T *P = a.tab->psi + q * NN;
                const T W = sW[le][qq];
                const T *dxi = sDx[le][qq][row];
                const T src = sQ[le][qq][0], dsrc = sQ[le][qq][1];
                const bool tr = TR && !a.deriv;
                if (a.deriv)
                    Racc = Racc + W * (src * P[row]);
                else if (tr)
                    Racc = Racc + W * ((dotv<T, DIM>(&sQ[le][qq][2], dxi) + src * P[row]) +
                                       sQ[le][qq][QT] * P[row]);
                else
                    Racc = Racc + W * (dotv<T, DIM>(&sQ[le][qq][2], dxi) + src * P[row]);
                if (a.flag == 2 && !TR) continue;   // no time derivative: mass matrix 0
                if (a.flag) {
                    const T tw0 = T(a.tw0);
#pragma unroll
                    for (int j = 0; j < NS; j++) {
                        if (sEq[le][j] < 0) continue;
                        const T *dxj = sDx[le][qq][j];
                        T v;
                        if constexpr (HV) {
                            v = W * (((sQ[le][qq][QH] * sQ[le][qq][QH + 1]) * P[j]) * P[row]);
                        } else if (a.flag == 2) {
                            v = W * (P[j] * P[row]);
                        } else if (a.deriv) {
                            v = W * ((dsrc * P[j]) * P[row]);
                        } else {
                            T inner;
                            if constexpr (FORM == PYHIP_FORM_POISSON)
                                inner = dotv<T, DIM>(dxj, dxi);
                            else
                                inner = dotv<T, DIM>(dxj, dxi) + (dsrc * P[j]) * P[row];
                            v = tr ? W * (inner + (tw0 * P[j]) * P[row]) : W * inner;
                        }
                        Jacc[j] = Jacc[j] + v;
                    }
                }
            }
        }
        if (q0 + QC < NQ) __syncthreads();
    }
    if (myrow) {
        a.Er[(int64_t)e * NS + row] = Racc;
        if (a.flag) {
            T *dst = a.Ej + ((int64_t)e * NS + row) * NS;
#pragma unroll
            for (int j = 0; j < NS; j++) dst[j] = Jacc[j];
        }
    }
}

// Scalar forms on triangles, one thread per element: residual (JAC false) or residual and
// Jacobian, steady or with the time derivative (TR). The element matrix (9 or 36 values), the
// coordinates and one point's geometry fit a thread's registers, so no value is read twice
// from LDS: with a thread per (element, row) every matrix entry of every point took its
// gradients, shape values and equation number from LDS, and the kernel waited 68 % of its
// time (sweep of 192 problems: P2 part 585 us, now 264, P1 part 63, now 39). Same operations in the same order per
// output. The matrices leave through LDS (odd stride per element: no bank conflicts), as
// coalesced stores over the block's elements; entries of pinned rows and columns are
// written too (nothing reads them). Bound: FP64 ALU without contraction, then the stores.
template <typename T, int KIND, int FORM, bool TR, bool JAC>
__global__ __launch_bounds__(kTriThreads) void tri_element_kernel(ElemArgs<T> a) {
    using Tt = ElemTraits<KIND>;
    constexpr int NN = Tt::NN, DIM = 2, NQ = Tt::NQ, NJ = NN * NN, ST = (JAC ? NJ : NQ) | 1;
    constexpr bool GAUSS = FORM == PYHIP_FORM_POISSON;
    __shared__ T out[JAC || GAUSS ? kTriThreads * ST : 1];   // the matrices; before, the sources
    const int eb = a.e0 + (int)blockIdx.x * kTriThreads, e = eb + (int)threadIdx.x;
    const int el = e < a.e1 ? e : a.e1 - 1;   // the threads past the end repeat the last element
    T X[NN][DIM], U[NN], F[FORM == PYHIP_FORM_REACTION_DIFFUSION ? NN : 1], H[TR ? NN : 1];
#pragma unroll
    for (int l = 0; l < NN; l++) {
        const int node = a.conn[(int64_t)l * a.nel + el], eq = a.seqn[(int64_t)l * a.nel + el];
#pragma unroll
        for (int d = 0; d < DIM; d++) X[l][d] = T(a.coords[(int64_t)node * 3 + d]);
        const double pin = a.pinned[(int64_t)node * a.nvalue];
        U[l] = T(eq >= 0 ? a.dofs[eq] : pin);
        if constexpr (FORM == PYHIP_FORM_REACTION_DIFFUSION) F[l] = T(a.aux[node]);
        if constexpr (TR) {
            const double u1 = eq >= 0 ? a.hist1[eq] : pin, u2 = eq >= 0 ? a.hist2[eq] : pin;
            H[l] = T(a.tw1 * u1 + a.tw2 * u2);
        }
    }
    const double *par = a.params + (int64_t)a.sub[el] * a.pstride;
    const T par0 = T(par[0]), tw0 = T(a.tw0);
    T R[NN], J[JAC ? NJ : 1];
#pragma unroll
    for (int i = 0; i < NN; i++) R[i] = T(0);
#pragma unroll
    for (int k = 0; k < (JAC ? NJ : 1); k++) J[k] = T(0);
    if constexpr (GAUSS) {
        // the sources of all points together, a Gaussian read once and NQ exponentials of it
        // independent of each other (point by point: 36 us for 81000 elements, now 33)
        T x[NQ], y[NQ], f[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const T *P = a.tab->psi + q * NN;
            x[q] = y[q] = f[q] = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) x[q] = x[q] + X[l][0] * P[l];
#pragma unroll
            for (int l = 0; l < NN; l++) y[q] = y[q] + X[l][1] * P[l];
        }
        const int ng = (int)par[0];  // Gaussians follow as (cx, cy, w, a)
#pragma unroll 1
        for (int k = 1; k < 1 + 4 * ng; k += 4) {
            const T cx = T(par[k + 0]), cy = T(par[k + 1]), wk = T(par[k + 2]), ak = T(par[k + 3]);
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                T ddx = x[q] - cx, ddy = y[q] - cy;
                T r2 = ddx * ddx + ddy * ddy;
                f[q] = f[q] + ak * texp(-r2 / (wk * wk));
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; q++) out[threadIdx.x * ST + q] = f[q];
    }
#pragma unroll 1
    for (int q = 0; q < NQ; q++) {
        const T *P = a.tab->psi + q * NN;
        T dx[NN][DIM];
        const T W = point_geometry<T, NN, DIM>(X, a.tab->dpsi + q * NN * DIM, a.tab->w[q], dx);
        T u = T(0);
#pragma unroll
        for (int l = 0; l < NN; l++) u = u + U[l] * P[l];
        T gu[DIM];
#pragma unroll
        for (int i = 0; i < DIM; i++) {
            T sacc = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) sacc = sacc + U[l] * dx[l][i];
            gu[i] = sacc;
        }
        T src = T(0), dsrc = T(0);
        if constexpr (FORM == PYHIP_FORM_POISSON) {
            src = -out[threadIdx.x * ST + q];
        } else if constexpr (FORM == PYHIP_FORM_BRATU) {
            T ev = texp(u);
            src = -par0 * ev;
            dsrc = -par0 * ev;
        } else {
            T f = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) f = f + F[l] * P[l];
            src = u * u * u - f;
            dsrc = T(3) * (u * u);
        }
        T ut = T(0);
        if constexpr (TR) {
            T hq = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) hq = hq + H[l] * P[l];
            ut = tw0 * u + hq;
        }
#pragma unroll
        for (int i = 0; i < NN; i++) {
            if constexpr (TR) R[i] = R[i] + W * ((dotv<T, DIM>(gu, dx[i]) + src * P[i]) + ut * P[i]);
            else R[i] = R[i] + W * (dotv<T, DIM>(gu, dx[i]) + src * P[i]);
            if constexpr (JAC) {
#pragma unroll
                for (int j = 0; j < NN; j++) {
                    T inner;
                    if constexpr (FORM == PYHIP_FORM_POISSON) inner = dotv<T, DIM>(dx[j], dx[i]);
                    else inner = dotv<T, DIM>(dx[j], dx[i]) + (dsrc * P[j]) * P[i];
                    const T v = TR ? W * (inner + (tw0 * P[j]) * P[i]) : W * inner;
                    J[i * NN + j] = J[i * NN + j] + v;
                }
            }
        }
    }
    if (e < a.e1) {
#pragma unroll
        for (int i = 0; i < NN; i++) a.Er[(int64_t)e * NN + i] = R[i];
    }
    if constexpr (JAC) {
#pragma unroll
        for (int k = 0; k < NJ; k++) out[threadIdx.x * ST + k] = J[k];
        __syncthreads();
        const int n = min(kTriThreads, a.e1 - eb) * NJ;
        T *dst = a.Ej + (int64_t)eb * NJ;
#pragma unroll 4
        for (int k = threadIdx.x; k < n; k += kTriThreads) dst[k] = out[(k / NJ) * ST + k % NJ];
    }
}

// Scalar forms on Q2 bricks: residual (JAC false) or residual and Jacobian, steady or with the
// time derivative (TR). A wave owns seven elements and needs no workgroup barrier after the
// reference tables are in LDS.
// Phase A: a thread per (element, point), three rounds of 63: tangents, metric, interpolated
// fields and source in its registers; only the dual vectors, the weight and the fields stay
// (15 or 16 values per point in LDS), not the 81 gradients.
// Phase B: nine lanes per element walk the points; each forms the gradients of three nodes
// from the dual vectors (15 operations a node) and shares them through LDS, adds its three
// residual rows and its 9 x 9 block of the matrix (rows 9 (t / 3) .., columns 9 (t % 3) ..),
// which stays in registers: 18 nodes' gradients read per point serve 81 entries. A thread per
// row read the gradients, shape value and equation number of every entry from LDS (four reads
// for nine operations). FP64 takes 256 registers and so one wave per SIMD; 18 lanes with 9 x 5
// blocks and twice the waves gave the same for the matrix and more for the residual. Same
// operations in the same order per output. Bound: FP64 ALU without contraction (9 operations
// per entry and point) with the LDS reads beside it. Before and now: 13824 elements FP32 with
// the matrix 320 and 85 us; 32000 FP64 858 and 585 us, residual only 234 (shared records of an
// even number of doubles, whose lanes meet on few banks) and 151 us.
constexpr int kHexPerWave = 7, kHexWaves = 4, kHexPerBlock = kHexPerWave * kHexWaves;
template <typename T, int FORM, bool TR>
struct HexWave {   // one wave's LDS
    // odd in FP64: an even number of doubles puts the lanes of a column on few banks
    static constexpr int kRec = 15 + (TR ? 2 : 0), kG = sizeof(T) == 8 ? 5 : 4;
    T rec[kHexPerWave][27][kRec];   // dual vectors [3][3], weight, src, dsrc, grad u, du/dt
    union {
        struct {
            T X[kHexPerWave][27][3], U[kHexPerWave][27];
            T F[FORM == PYHIP_FORM_REACTION_DIFFUSION ? kHexPerWave : 1][27], H[TR ? kHexPerWave : 1][27];
        } in;
        T g[kHexPerWave][27][kG];    // gradient of each node, and (source derivative) * shape
    } u;
};
template <typename T, int FORM, bool TR>
constexpr size_t hex_lds() {
    return 27 * 27 * 4 * sizeof(T) + kHexWaves * sizeof(HexWave<T, FORM, TR>);
}
template <typename T, int FORM, bool TR, bool JAC>
__global__ __launch_bounds__(64 * kHexWaves) void hex_element_kernel(ElemArgs<T> a) {
    constexpr int NN = 27, DIM = 3, NQ = 27, B = 9;
    extern __shared__ __align__(16) unsigned char hex_mem[];
    T *tD = (T *)hex_mem, *tP = tD + NQ * NN * DIM;
    using Wave = HexWave<T, FORM, TR>;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    Wave &M = ((Wave *)(tP + NQ * NN))[wave];
    for (int k = threadIdx.x; k < NQ * NN * DIM; k += 64 * kHexWaves) tD[k] = a.tab->dpsi[k];
    for (int k = threadIdx.x; k < NQ * NN; k += 64 * kHexWaves) tP[k] = a.tab->psi[k];
    const int ew = a.e0 + (int)blockIdx.x * kHexPerBlock + wave * kHexPerWave;   // the wave's first element
    const int ne = min(kHexPerWave, a.e1 - ew);                                     // (<= 0: none)
    for (int k = lane; k < ne * NN; k += 64) {
        const int le = k / NN, l = k % NN, e = ew + le;
        const int node = a.conn[(int64_t)l * a.nel + e], eq = a.seqn[(int64_t)l * a.nel + e];
#pragma unroll
        for (int d = 0; d < DIM; d++) M.u.in.X[le][l][d] = T(a.coords[(int64_t)node * 3 + d]);
        const double pin = a.pinned[(int64_t)node * a.nvalue];
        M.u.in.U[le][l] = T(eq >= 0 ? a.dofs[eq] : pin);
        if constexpr (FORM == PYHIP_FORM_REACTION_DIFFUSION) M.u.in.F[le][l] = T(a.aux[node]);
        if constexpr (TR) {
            const double u1 = eq >= 0 ? a.hist1[eq] : pin, u2 = eq >= 0 ? a.hist2[eq] : pin;
            M.u.in.H[le][l] = T(a.tw1 * u1 + a.tw2 * u2);
        }
    }
    __syncthreads();
    auto sync = []() {   // the wave's LDS writes before its later reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const T tw0 = T(a.tw0);
    // ---- phase A
#pragma unroll 1
    for (int k = lane; k < ne * NQ; k += 63) {
        if (lane == 63) break;
        const int le = k / NQ, q = k % NQ;
        const T *D = tD + q * NN * DIM, *P = tP + q * NN;
        const T(*X)[DIM] = M.u.in.X[le];
        T t[DIM][DIM], g[DIM][DIM];
#pragma unroll
        for (int i = 0; i < DIM; i++)
#pragma unroll
            for (int j = 0; j < DIM; j++) t[i][j] = T(0);
#pragma unroll 3
        for (int l = 0; l < NN; l++)
#pragma unroll
            for (int i = 0; i < DIM; i++)
#pragma unroll
                for (int j = 0; j < DIM; j++) t[j][i] = t[j][i] + X[l][i] * D[l * DIM + j];
        T *r = M.rec[le][q];
        const T W = metric<T, DIM>(t, a.tab->w[q], g);
        T u = T(0), f = T(0), hq = T(0), gu[DIM] = {T(0), T(0), T(0)}, x = T(0), y = T(0);
#pragma unroll 3
        for (int l = 0; l < NN; l++) {
            const T ul = M.u.in.U[le][l];
            u = u + ul * P[l];
#pragma unroll
            for (int i = 0; i < DIM; i++) {
                T s = T(0);
#pragma unroll
                for (int b = 0; b < DIM; b++) s = s + g[b][i] * D[l * DIM + b];
                gu[i] = gu[i] + ul * s;
            }
            if constexpr (FORM == PYHIP_FORM_REACTION_DIFFUSION) f = f + M.u.in.F[le][l] * P[l];
            if constexpr (FORM == PYHIP_FORM_POISSON) {
                x = x + X[l][0] * P[l];
                y = y + X[l][1] * P[l];
            }
            if constexpr (TR) hq = hq + M.u.in.H[le][l] * P[l];
        }
        const double *par = a.params + (int64_t)a.sub[ew + le] * a.pstride;
        T src = T(0), dsrc = T(0);
        if constexpr (FORM == PYHIP_FORM_POISSON) {
            const int ng = (int)par[0];  // Gaussians follow as (cx, cy, w, a)
            for (int c = 1; c < 1 + 4 * ng; c += 4) {
                T ddx = x - T(par[c + 0]), ddy = y - T(par[c + 1]);
                T r2 = ddx * ddx + ddy * ddy;
                T wk = T(par[c + 2]);
                f = f + T(par[c + 3]) * texp(-r2 / (wk * wk));
            }
            src = -f;
        } else if constexpr (FORM == PYHIP_FORM_BRATU) {
            const T par0 = T(par[0]), ev = texp(u);
            src = -par0 * ev;
            dsrc = -par0 * ev;
        } else {
            src = u * u * u - f;
            dsrc = T(3) * (u * u);
        }
#pragma unroll
        for (int b = 0; b < DIM; b++)
#pragma unroll
            for (int i = 0; i < DIM; i++) r[b * DIM + i] = g[b][i];
        r[9] = W;
        r[10] = src;
        r[11] = dsrc;
#pragma unroll
        for (int i = 0; i < DIM; i++) r[12 + i] = gu[i];
        if constexpr (TR) r[15] = tw0 * u + hq;
    }
    sync();
    // ---- phase B
    const int le = lane / B, t = lane % B, e = ew + le;
    const bool active = le < ne && lane < B * kHexPerWave;
    const int r0 = (t / 3) * B, c0 = (t % 3) * B;
    T J[JAC ? B : 1][B], R[3];   // lane t's residual rows: t, t + 9, t + 18
#pragma unroll
    for (int i = 0; i < (JAC ? B : 1); i++)
#pragma unroll
        for (int j = 0; j < B; j++) J[i][j] = T(0);
#pragma unroll
    for (int i = 0; i < 3; i++) R[i] = T(0);
#pragma unroll 1
    for (int q = 0; q < NQ; q++) {
        const T *D = tD + q * NN * DIM, *P = tP + q * NN;
        const T *r = M.rec[active ? le : 0][q];
        const T W = r[9];
        if (active) {
            T g[DIM][DIM];
#pragma unroll
            for (int b = 0; b < DIM; b++)
#pragma unroll
                for (int i = 0; i < DIM; i++) g[b][i] = r[b * DIM + i];
            const T src = r[10], dsrc = r[11], gu[DIM] = {r[12], r[13], r[14]};
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const int l = t + k * B;
                T dx[DIM];
#pragma unroll
                for (int i = 0; i < DIM; i++) {
                    T s = T(0);
#pragma unroll
                    for (int b = 0; b < DIM; b++) s = s + g[b][i] * D[l * DIM + b];
                    dx[i] = s;
                }
                const T p = P[l];
                if constexpr (TR) R[k] = R[k] + W * ((dotv<T, DIM>(gu, dx) + src * p) + r[15] * p);
                else R[k] = R[k] + W * (dotv<T, DIM>(gu, dx) + src * p);
                if constexpr (JAC) {
#pragma unroll
                    for (int i = 0; i < DIM; i++) M.u.g[le][l][i] = dx[i];
                    M.u.g[le][l][3] = dsrc * p;
                }
            }
        }
        if constexpr (JAC) {
            sync();
            if (active) {
                // columns in two groups held in registers, the rows read for each
                auto block = [&](auto first, auto count) {
                    constexpr int J0 = decltype(first)::value, NJ = decltype(count)::value;
                    T gj[NJ][4], tp[TR ? NJ : 1];
#pragma unroll
                    for (int j = 0; j < NJ; j++) {
#pragma unroll
                        for (int k = 0; k < 4; k++) gj[j][k] = M.u.g[le][c0 + J0 + j][k];
                        if constexpr (TR) tp[j] = tw0 * P[c0 + J0 + j];
                    }
#pragma unroll
                    for (int i = 0; i < B; i++) {
                        const T *gi = M.u.g[le][r0 + i];
                        const T dxi[DIM] = {gi[0], gi[1], gi[2]};
                        const T pi = P[r0 + i];
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            T inner;
                            if constexpr (FORM == PYHIP_FORM_POISSON) inner = dotv<T, DIM>(gj[j], dxi);
                            else inner = dotv<T, DIM>(gj[j], dxi) + gj[j][3] * pi;
                            T v;
                            if constexpr (TR) v = W * (inner + tp[j] * pi);
                            else v = W * inner;
                            J[i][J0 + j] = J[i][J0 + j] + v;
                        }
                    }
                };
                block(std::integral_constant<int, 0>{}, std::integral_constant<int, 5>{});
                block(std::integral_constant<int, 5>{}, std::integral_constant<int, 4>{});
            }
            sync();   // the next point overwrites the gradients
        }
    }
    if (!active) return;
#pragma unroll
    for (int k = 0; k < 3; k++) a.Er[(int64_t)e * NN + t + k * B] = R[k];
    if constexpr (JAC)
#pragma unroll
        for (int i = 0; i < B; i++) {
            T *dst = a.Ej + ((int64_t)e * NN + r0 + i) * NN + c0;
#pragma unroll
            for (int j = 0; j < B; j++) dst[j] = J[i][j];
        }
}

// Taylor-Hood Navier-Stokes: residual (JAC false) or residual and Jacobian, steady or with the
// time derivative (TR). Phase A as th_element_kernel: a thread per (element, integration
// point). Phase B: a thread per (element, node) holds the node's two velocity rows (44 values)
// in registers and walks the points and the nine column nodes; the four pressure rows follow.
// A thread per slot row put the three kinds of rows side by side in a wave, which then ran
// every kind's code for every entry, with an equation-number read and branch for each
// (16384 elements: 181 us, now 44). Same operations in the same order per output; the entries of
// pinned rows and columns are written too (nothing reads them). Bound: FP64 ALU without
// contraction.
constexpr int kThPer = 14, kThThreads = 128;   // elements and threads per workgroup (9 threads per element)
template <typename T, bool TR, bool JAC>
__global__ __launch_bounds__(kThThreads) void th_node_kernel(ElemArgs<T> a) {
    constexpr int NN = 9, DIM = 2, NQ = 9, NS = 22, QV = TR ? 9 : 7;
    constexpr int kSlot[9] = {0, 3, 5, 8, 10, 12, 14, 17, 19};   // velocity-x slot of each node
    constexpr int kPress[4] = {2, 7, 16, 21};
    struct El {
        T X[NN][DIM], V[NS], H[TR ? NS : 1], W[NQ], g[NQ][NN][DIM], Q[NQ][QV];
    };
    __shared__ El els[kThPer];
    __shared__ T sP[NQ][NN];
    const int le = threadIdx.x / NN, t = threadIdx.x % NN;
    const int e = a.e0 + (int)blockIdx.x * kThPer + le;
    const bool active = le < kThPer && e < a.e1;
    El &E = els[le < kThPer ? le : 0];
    for (int k = threadIdx.x; k < NQ * NN; k += kThThreads) sP[k / NN][k % NN] = a.tab->psi[k];
    T mu = T(0), rho = T(0);
    if (active) {
        const double *par = a.params + (int64_t)a.sub[e] * a.pstride;
        mu = T(par[0]);
        rho = T(par[1]);
        const int node = a.conn[(int64_t)t * a.nel + e];
        E.X[t][0] = T(a.coords[(int64_t)node * 3 + 0]);
        E.X[t][1] = T(a.coords[(int64_t)node * 3 + 1]);
        // corners (nodes 0, 2, 6, 8) carry the pressure after their velocities
        const int s0 = kTHNodeSlot[t], nk = (t & 1) == 0 && t != 4 ? 3 : 2;
        for (int k = 0; k < nk; k++) {
            const int eq = a.seqn[(int64_t)(s0 + k) * a.nel + e];
            const double pin = a.pinned[(int64_t)node * a.nvalue + k];
            E.V[s0 + k] = T(eq >= 0 ? a.dofs[eq] : pin);
            if constexpr (TR) {
                const double u1 = eq >= 0 ? a.hist1[eq] : pin, u2 = eq >= 0 ? a.hist2[eq] : pin;
                E.H[s0 + k] = T(a.tw1 * u1 + a.tw2 * u2);
            }
        }
    }
    __syncthreads();
    if (active) {
        const int q = t;
        const T *D = a.tab->dpsi + q * NN * DIM;
        const T *P = sP[q];
        const T *C = a.tab->psi1 + q * 4;
        E.W[q] = point_geometry<T, NN, DIM>(E.X, D, a.tab->w[q], E.g[q]);
        T u0 = T(0), u1 = T(0), p = T(0);
#pragma unroll
        for (int l = 0; l < NN; l++) u0 = u0 + E.V[kSlot[l]] * P[l];
#pragma unroll
        for (int l = 0; l < NN; l++) u1 = u1 + E.V[kSlot[l] + 1] * P[l];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            T s0 = T(0), s1 = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) s0 = s0 + E.V[kSlot[l]] * E.g[q][l][b];
#pragma unroll
            for (int l = 0; l < NN; l++) s1 = s1 + E.V[kSlot[l] + 1] * E.g[q][l][b];
            E.Q[q][2 + b] = s0;       // du[0][b]
            E.Q[q][4 + b] = s1;       // du[1][b]
        }
#pragma unroll
        for (int k = 0; k < 4; k++) p = p + E.V[kPress[k]] * C[k];
        E.Q[q][0] = u0;
        E.Q[q][1] = u1;
        E.Q[q][6] = p;
        if constexpr (TR) {
            T h0 = T(0), h1 = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) h0 = h0 + E.H[kSlot[l]] * P[l];
#pragma unroll
            for (int l = 0; l < NN; l++) h1 = h1 + E.H[kSlot[l] + 1] * P[l];
            E.Q[q][7] = T(a.tw0) * u0 + h0;
            E.Q[q][8] = T(a.tw0) * u1 + h1;
        }
    }
    __syncthreads();
    if (active) {
        T R0 = T(0), R1 = T(0), J0[JAC ? NS : 1], J1[JAC ? NS : 1];
#pragma unroll
        for (int j = 0; j < (JAC ? NS : 1); j++) J0[j] = J1[j] = T(0);
#pragma unroll 1
        for (int q = 0; q < NQ; q++) {
            const T *P = a.tab->psi + q * NN, *C = a.tab->psi1 + q * 4;
            const T W = E.W[q], pl = sP[q][t];
            const T u0 = E.Q[q][0], u1 = E.Q[q][1], p = E.Q[q][6];
            const T d00 = E.Q[q][2], d01 = E.Q[q][3], d10 = E.Q[q][4], d11 = E.Q[q][5];
            const T l0 = E.g[q][t][0], l1 = E.g[q][t][1];
            const T s00 = mu * (d00 + d00) - p, s01 = mu * (d01 + d10), s10 = mu * (d10 + d01), s11 = mu * (d11 + d11) - p;
            const T c0 = rho * (u0 * d00 + u1 * d01), c1 = rho * (u0 * d10 + u1 * d11);
            if constexpr (TR) {
                R0 = R0 + W * (((s00 * l0 + s01 * l1) + c0 * pl) + (rho * E.Q[q][7]) * pl);
                R1 = R1 + W * (((s10 * l0 + s11 * l1) + c1 * pl) + (rho * E.Q[q][8]) * pl);
            } else {
                R0 = R0 + W * ((s00 * l0 + s01 * l1) + c0 * pl);
                R1 = R1 + W * ((s10 * l0 + s11 * l1) + c1 * pl);
            }
            if constexpr (JAC) {
#pragma unroll
                for (int n = 0; n < NN; n++) {
                    const T x0 = E.g[q][n][0], x1 = E.g[q][n][1], ps = P[n];
                    const T lap = x0 * l0 + x1 * l1, adv = u0 * x0 + u1 * x1;
                    const T a00 = mu * (lap + x0 * l0) + (rho * (ps * d00 + adv)) * pl;
                    const T a01 = mu * (x0 * l1) + (rho * (ps * d01)) * pl;
                    const T a10 = mu * (x1 * l0) + (rho * (ps * d10)) * pl;
                    const T a11 = mu * (lap + x1 * l1) + (rho * (ps * d11 + adv)) * pl;
                    const int c = kSlot[n];
                    if constexpr (TR) {
                        const T m = ((rho * T(a.tw0)) * ps) * pl;
                        J0[c] = J0[c] + W * (a00 + m);
                        J1[c + 1] = J1[c + 1] + W * (a11 + m);
                    } else {
                        J0[c] = J0[c] + W * a00;
                        J1[c + 1] = J1[c + 1] + W * a11;
                    }
                    J0[c + 1] = J0[c + 1] + W * a01;
                    J1[c] = J1[c] + W * a10;
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    J0[kPress[k]] = J0[kPress[k]] + W * (-(C[k] * l0));
                    J1[kPress[k]] = J1[kPress[k]] + W * (-(C[k] * l1));
                }
            }
        }
        const int64_t row = (int64_t)e * NS + kTHNodeSlot[t];
        a.Er[row] = R0;
        a.Er[row + 1] = R1;
        if constexpr (JAC) {
            T *dst = a.Ej + row * NS;
#pragma unroll
            for (int j = 0; j < NS; j++) dst[j] = J0[j];
#pragma unroll
            for (int j = 0; j < NS; j++) dst[NS + j] = J1[j];
        }
    }
    // pressure rows: a thread per (element, corner)
    const int lp = threadIdx.x / 4, k = threadIdx.x % 4, ep = a.e0 + (int)blockIdx.x * kThPer + lp;
    if (lp >= kThPer || ep >= a.e1) return;
    const El &F = els[lp];
    T R = T(0), J[JAC ? NN : 1][DIM];
#pragma unroll
    for (int n = 0; n < (JAC ? NN : 1); n++) J[n][0] = J[n][1] = T(0);
#pragma unroll 1
    for (int q = 0; q < NQ; q++) {
        const T W = F.W[q], c = a.tab->psi1[q * 4 + k];
        R = R + W * ((F.Q[q][2] + F.Q[q][5]) * c);
        if constexpr (JAC)
#pragma unroll
            for (int n = 0; n < NN; n++) {
                J[n][0] = J[n][0] + W * (F.g[q][n][0] * c);
                J[n][1] = J[n][1] + W * (F.g[q][n][1] * c);
            }
    }
    const int64_t row = (int64_t)ep * NS + (k == 0 ? kPress[0] : k == 1 ? kPress[1] : k == 2 ? kPress[2] : kPress[3]);
    a.Er[row] = R;
    if constexpr (JAC) {
        T *dst = a.Ej + row * NS;
#pragma unroll
        for (int n = 0; n < NN; n++) {
            dst[kSlot[n]] = J[n][0];
            dst[kSlot[n] + 1] = J[n][1];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) dst[kPress[j]] = T(0);
    }
}

// Mass matrices (flag 2) and Hessian-vector products (HV) of the Taylor-Hood Q2/Q1 Navier-Stokes
// form, each beside the residual (22 slots, 9 geometric nodes). Phase A: thread t < 9 of an element
// computes integration point t (geometry, dx_shape, u, grad u, p); phase B: thread = slot row.
// TR: time derivative of the velocities (a.transient): du/dt = tw0 u + sum_l H psi_l with
// H = tw1 u(t-1) + tw2 u(t-2) per slot; momentum rows gain (rho du/dt) psi_i, and the mass
// matrix is rho psi_j psi_i on the diagonal velocity blocks (none without TR).
template <typename T, bool TR, bool HV = false>
__global__ __launch_bounds__(256) void th_element_kernel(ElemArgs<T> a) {
    constexpr int NN = 9, DIM = 2, NQ = 9, NS = 22;
    constexpr int EPB = 256 / NS;  // 11 elements, 242 threads
    // per point: u0, u1, du00, du01, du10, du11, p[, du0/dt, du1/dt][, y0, y1, dy00, dy01, dy10, dy11]
    constexpr int QY = TR ? 9 : 7;
    __shared__ T sX[EPB][NN][DIM];
    __shared__ T sV[EPB][NS];
    __shared__ int sEq[EPB][NS];
    __shared__ T sW[EPB][NQ];
    __shared__ T sDx[EPB][NQ][NN][DIM];
    __shared__ T sQ[EPB][NQ][QY + (HV ? 6 : 0)];
    __shared__ T sH[TR ? EPB : 1][NS];
    __shared__ T sY[HV ? EPB : 1][NS];   // Hessian-vector product direction per slot

    const int le = threadIdx.x / NS;
    const int slot = threadIdx.x % NS;
    const int e = a.e0 + (int)blockIdx.x * EPB + le;
    const bool active = (le < EPB) && (e < a.e1);
    if (active) {
        const int ln = kTHSlotNode[slot];
        const int kind = kTHSlotKind[slot];
        const int node = a.conn[(int64_t)ln * a.nel + e];
        const int eq = a.seqn[(int64_t)slot * a.nel + e];
        if (slot < NN) {
            const int gn = a.conn[(int64_t)slot * a.nel + e];
            sX[le][slot][0] = T(a.coords[(int64_t)gn * 3 + 0]);
            sX[le][slot][1] = T(a.coords[(int64_t)gn * 3 + 1]);
        }
        sV[le][slot] = T(eq >= 0 ? a.dofs[eq] : a.pinned[(int64_t)node * a.nvalue + kind]);
        if constexpr (TR) {
            const double pin = a.pinned[(int64_t)node * a.nvalue + kind];
            const double u1 = eq >= 0 ? a.hist1[eq] : pin, u2 = eq >= 0 ? a.hist2[eq] : pin;
            sH[le][slot] = T(a.tw1 * u1 + a.tw2 * u2);
        }
        if constexpr (HV) sY[le][slot] = T(eq >= 0 ? a.hvec[eq] : 0.0);
        sEq[le][slot] = eq;
    }
    __syncthreads();
    T mu = T(0), rho = T(0);
    if (active) {
        const double *par = a.params + (int64_t)a.sub[e] * a.pstride;
        mu = T(par[0]);
        rho = T(par[1]);
    }
    if (active && slot < NQ) {
        const int q = slot;
        const T *D = a.tab->dpsi + q * NN * DIM;
        const T *P = a.tab->psi + q * NN;
        const T *C = a.tab->psi1 + q * 4;
        sW[le][q] = point_geometry<T, NN, DIM>(sX[le], D, a.tab->w[q], sDx[le][q]);
        T u0 = T(0), u1 = T(0), p = T(0);
#pragma unroll
        for (int l = 0; l < NN; l++) u0 = u0 + sV[le][kTHNodeSlot[l]] * P[l];
#pragma unroll
        for (int l = 0; l < NN; l++) u1 = u1 + sV[le][1 + kTHNodeSlot[l]] * P[l];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            T s0 = T(0), s1 = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) s0 = s0 + sV[le][kTHNodeSlot[l]] * sDx[le][q][l][b];
#pragma unroll
            for (int l = 0; l < NN; l++) s1 = s1 + sV[le][kTHNodeSlot[l] + 1] * sDx[le][q][l][b];
            sQ[le][q][2 + b] = s0;       // du[0][b]
            sQ[le][q][4 + b] = s1;       // du[1][b]
        }
        // pressure slots 2, 7, 16, 21 hold corner nodes 0, 2, 6, 8
        p = p + sV[le][2] * C[0];
        p = p + sV[le][7] * C[1];
        p = p + sV[le][16] * C[2];
        p = p + sV[le][21] * C[3];
        sQ[le][q][0] = u0;
        sQ[le][q][1] = u1;
        sQ[le][q][6] = p;
        if constexpr (TR) {
            T h0 = T(0), h1 = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) h0 = h0 + sH[le][kTHNodeSlot[l]] * P[l];
#pragma unroll
            for (int l = 0; l < NN; l++) h1 = h1 + sH[le][kTHNodeSlot[l] + 1] * P[l];
            sQ[le][q][7] = T(a.tw0) * u0 + h0;
            sQ[le][q][8] = T(a.tw0) * u1 + h1;
        }
        if constexpr (HV) {
            T y0 = T(0), y1 = T(0);
#pragma unroll
            for (int l = 0; l < NN; l++) y0 = y0 + sY[le][kTHNodeSlot[l]] * P[l];
#pragma unroll
            for (int l = 0; l < NN; l++) y1 = y1 + sY[le][1 + kTHNodeSlot[l]] * P[l];
#pragma unroll
            for (int b = 0; b < 2; b++) {
                T s0 = T(0), s1 = T(0);
#pragma unroll
                for (int l = 0; l < NN; l++) s0 = s0 + sY[le][kTHNodeSlot[l]] * sDx[le][q][l][b];
#pragma unroll
                for (int l = 0; l < NN; l++) s1 = s1 + sY[le][kTHNodeSlot[l] + 1] * sDx[le][q][l][b];
                sQ[le][q][QY + 2 + b] = s0;   // dy[0][b]
                sQ[le][q][QY + 4 + b] = s1;   // dy[1][b]
            }
            sQ[le][q][QY] = y0;
            sQ[le][q][QY + 1] = y1;
        }
    }
    __syncthreads();
    const bool myrow = active && sEq[le][slot] >= 0;
    if (!myrow) return;
    const int kt = kTHSlotKind[slot], lt = kTHSlotNode[slot];
    T Racc = T(0);
    T Jacc[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) Jacc[j] = T(0);
    for (int q = 0; q < NQ; q++) {
        const T *P = a.tab->psi + q * NN;
        const T *C = a.tab->psi1 + q * 4;
        const T W = sW[le][q];
        const T u0 = sQ[le][q][0], u1 = sQ[le][q][1], p = sQ[le][q][6];
        T du[2][2];
        du[0][0] = sQ[le][q][2];
        du[0][1] = sQ[le][q][3];
        du[1][0] = sQ[le][q][4];
        du[1][1] = sQ[le][q][5];
        T sig[2][2];
#pragma unroll
        for (int aa = 0; aa < 2; aa++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                T s = mu * (du[aa][b] + du[b][aa]);
                if (aa == b) s = s - p;
                sig[aa][b] = s;
            }
        const T *dxl = sDx[le][q][lt];
        if (kt < 2) {
            const T conv = rho * (u0 * du[kt][0] + u1 * du[kt][1]);
            if constexpr (TR)
                Racc = Racc + W * (((sig[kt][0] * dxl[0] + sig[kt][1] * dxl[1]) + conv * P[lt]) +
                                   (rho * sQ[le][q][7 + kt]) * P[lt]);
            else
                Racc = Racc + W * ((sig[kt][0] * dxl[0] + sig[kt][1] * dxl[1]) + conv * P[lt]);
        } else {
            const int pidx = kTHSlotP[slot];
            Racc = Racc + W * ((du[0][0] + du[1][1]) * C[pidx]);
        }
        if (a.flag == 2 && !TR) continue;   // no time derivative: mass matrix 0
        if (a.flag) {
#pragma unroll
            for (int ss = 0; ss < NS; ss++) {
                if (sEq[le][ss] < 0) continue;
                const int ks = kTHSlotKind[ss], ls = kTHSlotNode[ss];
                T v;
                if constexpr (HV) {
                    if (kt < 2 && ks < 2) {
                        const T *dxs = sDx[le][q][ls];
                        if (a.htr) {
                            // Hessian of y . R (row kt,lt; column ks,ls): only the convection
                            // term is not linear, rho (psi_lt d_kt psi_ls y_ks + psi_ls d_ks psi_lt y_kt)
                            const T cvt = P[lt] * dxs[kt] * sQ[le][q][QY + ks] + P[ls] * dxl[ks] * sQ[le][q][QY + kt];
                            v = W * (rho * cvt);
                        } else {
                            // d/du of the convection block in the direction y: the block with u -> y
                            T cvy = P[ls] * sQ[le][q][QY + 2 + 2 * kt + ks];
                            if (kt == ks) cvy = cvy + (sQ[le][q][QY] * dxs[0] + sQ[le][q][QY + 1] * dxs[1]);
                            v = W * ((rho * cvy) * P[lt]);
                        }
                    } else {
                        continue;
                    }
                } else {
                    if (kt < 2 && kt == ks) v = W * ((rho * P[ls]) * P[lt]);
                    else continue;
                }
                Jacc[ss] = Jacc[ss] + v;
            }
        }
    }
    a.Er[(int64_t)e * NS + slot] = Racc;
    if (a.flag) {
        T *dst = a.Ej + ((int64_t)e * NS + slot) * NS;
#pragma unroll
        for (int j = 0; j < NS; j++) dst[j] = Jacc[j];
    }
}

}  // namespace pyhip
