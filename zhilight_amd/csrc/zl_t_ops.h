// zl_t_ops.h -- arithmetic on 16-bit numbers with a rounding to T per step, shared by the elementwise kernels and the products' epilogues
#pragma once
#include "zl_common.h"

template <int DT>
__device__ __forceinline__ uint16_t t_add(uint16_t a, uint16_t b) {  // one rounding to T (exact sum in fp32*)
    // fp16: the fp32 sum of two halfs is exact; bf16: may round in fp32 first (documented)
    return ZT<DT>::from_f32(ZT<DT>::to_f32(a) + ZT<DT>::to_f32(b));
}
template <int DT>
__device__ __forceinline__ uint16_t t_mul(uint16_t a, uint16_t b) {  // product of two T is exact in fp32
    return ZT<DT>::from_f32(ZT<DT>::to_f32(a) * ZT<DT>::to_f32(b));
}
// act(g) u in fp32, one rounding; act 0: silu, 1: gelu (tanh form)
template <int DT>
__device__ __forceinline__ uint16_t t_gate(uint16_t g, uint16_t u, int act) {
    const float x = ZT<DT>::to_f32(g);
    float a;
    if (act == 0) a = x / (1.0f + expf(-x));
    else a = 0.5f * x * (1.0f + tanhf(0.7978845608028654f * x * (1.0f + 0.044715f * x * x)));
    return ZT<DT>::from_f32(a * ZT<DT>::to_f32(u));
}
