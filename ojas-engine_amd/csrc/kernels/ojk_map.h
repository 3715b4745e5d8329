// Grid-stride maps shared by the conversion kernels and the decoders that convert activations beside their work.
#pragma once
#include "ojk_common.h"

// The element-wise kernels are grid-stride loops over groups of 8 elements (128-bit accesses when
// both pointers are 16-byte aligned), plus a scalar tail: any grid of 256-thread blocks is valid.
template <class In, class Out, class F>
__device__ __forceinline__ void map8_at(const In* __restrict__ x, Out* __restrict__ y, uint n, F f, uint t, uint stride) {
    uint done = 0;
    if ((((size_t)x | (size_t)y) & 15u) == 0) {
        const uint n8 = n >> 3;
        for (uint i = t; i < n8; i += stride) {
            In v[8];
            Out o[8];
            if (sizeof(In) == 4) { *(uint4*)v = ((const uint4*)x)[2 * i]; *(uint4*)(v + 4) = ((const uint4*)x)[2 * i + 1]; }
            else *(uint4*)v = ((const uint4*)x)[i];
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = f(v[e]);
            if (sizeof(Out) == 4) { ((uint4*)y)[2 * i] = *(uint4*)o; ((uint4*)y)[2 * i + 1] = *(uint4*)(o + 4); }
            else ((uint4*)y)[i] = *(uint4*)o;
        }
        done = n8 << 3;
    }
    for (uint i = done + t; i < n; i += stride) y[i] = f(x[i]);
}
__device__ __forceinline__ void fill_zero_at(uint* __restrict__ y, uint n, uint t, uint stride) {
    uint done = 0;
    if (((size_t)y & 15u) == 0) {
        const uint n4 = n >> 2;
        for (uint i = t; i < n4; i += stride) ((uint4*)y)[i] = make_uint4(0u, 0u, 0u, 0u);
        done = n4 << 2;
    }
    for (uint i = done + t; i < n; i += stride) y[i] = 0u;
}
