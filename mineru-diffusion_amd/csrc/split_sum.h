// A row of a linear layer's output as the K-split partial sums that mdx_decode_linear_partials leaves: eight consecutive
// columns, summed in fp32 and rounded to the storage type as the layer's own output would be.
#pragma once
#include "mdx_common.h"

namespace mdx_split {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ bf16x8 sum8(const float* __restrict__ p, int splits, int64_t stride) {
    f32x4 lo = f32x4{0.f, 0.f, 0.f, 0.f}, hi = lo;
    int s = 0;
    for (; s + 4 <= splits; s += 4) {               // four splits' loads in flight together
        f32x4 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] = *reinterpret_cast<const f32x4*>(p + (s + i) * stride);
            b[i] = *reinterpret_cast<const f32x4*>(p + (s + i) * stride + 4);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) { lo += a[i]; hi += b[i]; }
    }
    for (; s < splits; ++s) {
        lo += *reinterpret_cast<const f32x4*>(p + s * stride);
        hi += *reinterpret_cast<const f32x4*>(p + s * stride + 4);
    }
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) { out[e] = (__bf16)lo[e]; out[4 + e] = (__bf16)hi[e]; }
    return out;
}

}  // namespace mdx_split
