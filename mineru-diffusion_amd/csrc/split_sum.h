// A row of a linear layer's output as the K-split partial sums that mdx_linear_partials leaves: eight consecutive
// columns, summed in fp32 and rounded to the storage type as the layer's own output would be.
#pragma once
#include "mdx_common.h"
#include <type_traits>

namespace mdx_split {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// A kernel's SLICES: how many there are, with their loads in flight together and with whatever else the caller asks for before it takes
// the sum; kAnySlices, known at run time only, two at a time; kNoSlices, the row itself in bf16.
constexpr int kNoSlices = 0, kAnySlices = -1;

template <int SLICES> struct Eight {
    static constexpr int N = SLICES > 0 ? SLICES : 1;
    bf16x8 row;
    f32x4 lo[N], hi[N];
    const float* p; int n; int64_t stride;
    // x: the columns in bf16; or partials: the columns in the first of n slices, `between` elements apart.
    __device__ __forceinline__ void load(const __bf16* x, const float* partials, int slices, int64_t between) {
        p = partials; n = slices; stride = between;
        if constexpr (SLICES == kNoSlices) row = *reinterpret_cast<const bf16x8*>(x);
        if constexpr (SLICES > 0) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                lo[i] = *reinterpret_cast<const f32x4*>(p + i * stride);
                hi[i] = *reinterpret_cast<const f32x4*>(p + i * stride + 4);
            }
        }
    }
    __device__ __forceinline__ bf16x8 value() const {
        if constexpr (SLICES == kNoSlices) return row;
        f32x4 l = f32x4{0.f, 0.f, 0.f, 0.f}, h = l;
        if constexpr (SLICES > 0) {
#pragma unroll
            for (int i = 0; i < N; ++i) { l += lo[i]; h += hi[i]; }
        } else {
#pragma unroll 2
            for (int i = 0; i < n; ++i) {
                l += *reinterpret_cast<const f32x4*>(p + i * stride);
                h += *reinterpret_cast<const f32x4*>(p + i * stride + 4);
            }
        }
        bf16x8 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) { out[e] = (__bf16)l[e]; out[4 + e] = (__bf16)h[e]; }
        return out;
    }
};

// The linear layers of few rows are cut into 2, 4 or 8 slices mostly.
template <typename Launch> void with_slices(int slices, Launch launch) {
    if (slices == 2) launch(std::integral_constant<int, 2>());
    else if (slices == 4) launch(std::integral_constant<int, 4>());
    else if (slices == 8) launch(std::integral_constant<int, 8>());
    else launch(std::integral_constant<int, kAnySlices>());
}

}  // namespace mdx_split
