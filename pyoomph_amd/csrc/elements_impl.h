// Launch dispatch for the element kernels of one precision (included once per TU).
#pragma once
#include "element_kernels.h"

namespace pyhip {

template <typename T, int KIND, int FORM>
static int launch_scalar(const ElemArgs<T> &a, hipStream_t s) {
    constexpr int EPB = scalar_epb<KIND>();
    const int blocks = (a.e1 - a.e0 + EPB - 1) / EPB;
    if (blocks == 0) return PYHIP_OK;
    if constexpr (KIND == ELEM_TRI_P1 || KIND == ELEM_TRI_P2) {
        // residuals and Jacobians of many elements: a thread per element; few, parameter
        // derivatives, mass matrices and Hessian products: a thread per row
        if constexpr (tri_min_elements<T, KIND, FORM>(true) >= 0) {
            if (!a.hvec && !a.deriv && a.flag < 2 && a.e1 - a.e0 >= tri_min_elements<T, KIND, FORM>(a.flag)) {
                const dim3 g((a.e1 - a.e0 + kTriThreads - 1) / kTriThreads), t(kTriThreads);
                if (a.transient) {
                    if (a.flag) hipLaunchKernelGGL((tri_element_kernel<T, KIND, FORM, true, true>), g, t, 0, s, a);
                    else hipLaunchKernelGGL((tri_element_kernel<T, KIND, FORM, true, false>), g, t, 0, s, a);
                } else {
                    if (a.flag) hipLaunchKernelGGL((tri_element_kernel<T, KIND, FORM, false, true>), g, t, 0, s, a);
                    else hipLaunchKernelGGL((tri_element_kernel<T, KIND, FORM, false, false>), g, t, 0, s, a);
                }
                PYHIP_CHECK_HIP(hipGetLastError());
                return PYHIP_OK;
            }
        }
    }
    if constexpr (KIND == ELEM_HEX_Q2) {
        if (!a.hvec && !a.deriv && a.flag < 2 && hex_takes<T>(a.e1 - a.e0, a.flag)) {
            const dim3 g((a.e1 - a.e0 + kHexPerBlock - 1) / kHexPerBlock), t(64 * kHexWaves);
            // most of a CU's LDS
            auto run = [&](auto *kernel, size_t lds) -> int {
                PYHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                hipLaunchKernelGGL(kernel, g, t, lds, s, a);
                PYHIP_CHECK_HIP(hipGetLastError());
                return PYHIP_OK;
            };
            if (a.transient) {
                constexpr size_t lds = hex_lds<T, FORM, true>();
                return a.flag ? run(&hex_element_kernel<T, FORM, true, true>, lds)
                              : run(&hex_element_kernel<T, FORM, true, false>, lds);
            }
            constexpr size_t lds = hex_lds<T, FORM, false>();
            return a.flag ? run(&hex_element_kernel<T, FORM, false, true>, lds)
                          : run(&hex_element_kernel<T, FORM, false, false>, lds);
        }
    }
    if (a.hvec)
        hipLaunchKernelGGL((scalar_element_kernel<T, KIND, FORM, false, true>), dim3(blocks), dim3(256), 0, s, a);
    else if (a.transient)
        hipLaunchKernelGGL((scalar_element_kernel<T, KIND, FORM, true, false>), dim3(blocks), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((scalar_element_kernel<T, KIND, FORM, false, false>), dim3(blocks), dim3(256), 0, s, a);
    PYHIP_CHECK_HIP(hipGetLastError());
    return PYHIP_OK;
}

template <typename T, int KIND>
static int launch_kind(int form, const ElemArgs<T> &a, hipStream_t s) {
    switch (form) {
    case PYHIP_FORM_POISSON: return launch_scalar<T, KIND, PYHIP_FORM_POISSON>(a, s);
    case PYHIP_FORM_BRATU: return launch_scalar<T, KIND, PYHIP_FORM_BRATU>(a, s);
    case PYHIP_FORM_REACTION_DIFFUSION:
        return launch_scalar<T, KIND, PYHIP_FORM_REACTION_DIFFUSION>(a, s);
    }
    set_error("weak form not available on this element family");
    return PYHIP_ERR_INVALID;
}

template <typename T>
static int launch_elements_impl(int kind, int form, const ElemArgs<T> &a, hipStream_t s) {
    if (form == PYHIP_FORM_NAVIER_STOKES_TH) {
        if (kind != ELEM_QUAD_Q2) {
            set_error("Taylor-Hood Navier-Stokes needs Q2 quadrilaterals");
            return PYHIP_ERR_INVALID;
        }
        constexpr int EPB = 256 / 22;
        const int blocks = (a.e1 - a.e0 + EPB - 1) / EPB;
        if (blocks == 0) return PYHIP_OK;
        if (!a.hvec && a.flag < 2) {
            // mass matrices and Hessian products: a thread per slot row
            const dim3 g((a.e1 - a.e0 + kThPer - 1) / kThPer), t(kThThreads);
            if (a.transient) {
                if (a.flag) hipLaunchKernelGGL((th_node_kernel<T, true, true>), g, t, 0, s, a);
                else hipLaunchKernelGGL((th_node_kernel<T, true, false>), g, t, 0, s, a);
            } else {
                if (a.flag) hipLaunchKernelGGL((th_node_kernel<T, false, true>), g, t, 0, s, a);
                else hipLaunchKernelGGL((th_node_kernel<T, false, false>), g, t, 0, s, a);
            }
            PYHIP_CHECK_HIP(hipGetLastError());
            return PYHIP_OK;
        }
        if (a.hvec) {
            // the product of the steady Jacobian (the time term is linear)
            hipLaunchKernelGGL((th_element_kernel<T, false, true>), dim3(blocks), dim3(256), 0, s, a);
        } else if (a.transient)
            hipLaunchKernelGGL((th_element_kernel<T, true>), dim3(blocks), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((th_element_kernel<T, false>), dim3(blocks), dim3(256), 0, s, a);
        PYHIP_CHECK_HIP(hipGetLastError());
        return PYHIP_OK;
    }
    switch (kind) {
    case ELEM_TRI_P1: return launch_kind<T, ELEM_TRI_P1>(form, a, s);
    case ELEM_TRI_P2: return launch_kind<T, ELEM_TRI_P2>(form, a, s);
    case ELEM_QUAD_Q2: return launch_kind<T, ELEM_QUAD_Q2>(form, a, s);
    case ELEM_HEX_Q2: return launch_kind<T, ELEM_HEX_Q2>(form, a, s);
    }
    set_error("unknown element family");
    return PYHIP_ERR_INVALID;
}

}  // namespace pyhip
