// dz = delta .* act'(y, pre) for VEC consecutive elements, and the matching store: shared by the streaming
// pullback kernels of bias_activation and by the passes that write dz in a second layout as well.
#pragma once

#include "common.h"

namespace luxhip {

// How the pre-activation of an element comes from what `pre` points to
struct Stored {                                  // it is the pre-activation
    __device__ __forceinline__ float operator()(float p, int) const { return p; }
};
template <typename T, int N>
struct PlusBias {                                // it is the operator's input: the bias of element k, rounded to what a stored pre-activation holds
    float b[N];
    __device__ __forceinline__ float operator()(float x, int k) const {
        const float p = x + b[N == 1 ? 0 : k];
        if constexpr (sizeof(T) == 2) return bf16_to_f32(f32_to_bf16(p));
        else return p;
    }
};
// RAGGED: any alignment (common.h, row_load)
template <typename T, int ACT, int VEC, bool RAGGED = false, class Pre = Stored>
__device__ __forceinline__ void dx_vec(const T* delta, const T* out, const T* pre, size_t off, float (&dx)[VEC], const Pre& pre_of = Pre()) {
    float d[VEC], o[VEC], p[VEC];
    if constexpr (VEC == 1) {
        d[0] = ld(delta + off);
        if constexpr (ACT != LUXHIP_ACT_IDENTITY && !Act<ACT>::needs_pre) o[0] = ld(out + off);
        if constexpr (Act<ACT>::needs_pre) p[0] = pre_of(ld(pre + off), 0);
    } else {
        row_load<T, VEC, RAGGED>(delta, off, d);
        if constexpr (ACT != LUXHIP_ACT_IDENTITY && !Act<ACT>::needs_pre) row_load<T, VEC, RAGGED>(out, off, o);
        if constexpr (Act<ACT>::needs_pre) {
            row_load<T, VEC, RAGGED>(pre, off, p);
#pragma unroll
            for (int k = 0; k < VEC; ++k) p[k] = pre_of(p[k], k);
        }
    }
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        if constexpr (ACT == LUXHIP_ACT_IDENTITY) dx[k] = d[k];
        else if constexpr (Act<ACT>::needs_pre) dx[k] = d[k] * Act<ACT>::d(Act<ACT>::f(p[k]), p[k]);
        else dx[k] = d[k] * Act<ACT>::d(o[k], 0.0f);
    }
}

template <typename T, int VEC>
__device__ __forceinline__ void store_vec(T* p, size_t off, const float (&v)[VEC]) {
    if constexpr (VEC == 1) st(p + off, v[0]);
    else Vec<T>::store(p + off, v);
}

}  // namespace luxhip
