// Noise of the sampled unmask step, drawn inside the kernels: a counter-based generator and its transform to Gumbel noise.
#pragma once
#include "mdx_common.h"

namespace mdx_noise {

// --- Gumbel noise drawn in the kernel ------------------------------------------------------------
// Sampler.prepare draws gumbel = -log(Exponential(1)) per logit (sampler.py:15-16).  Here the draw is
// a pure function of (seed, offset, row, column): Philox-4x32-10 (Salmon et al., "Parallel random
// numbers: as easy as 1, 2, 3", 2011) with key = seed and counter = (column / 4, row, offset), whose
// four 32-bit outputs serve columns 4*(column/4) .. +3.  So the noise does not depend on the launch
// geometry, a caller reproduces a step from three integers, and nothing is read from memory.
struct NoiseSpec {
    const float* noise; int64_t noise_row_stride;      // explicit noise tensor, or
    bool philox; uint32_t key0, key1;                   // noise from the generator: seed,
    uint64_t offset; const int64_t* offset_dev;         // offset (+ *offset_dev when given: a counter a graph replay can advance),
    const int64_t* row_ids;                             // and the row coordinate of each logits row (NULL: the row's own index)
};

struct U4 { uint32_t x, y, z, w; };

// a ^ b ^ c as one instruction (the compiler makes two of it); 0x96 is the truth table of the three-way exclusive or.  The sampled step,
// us, with two / one: 96 rows 27.5 / 26.1, 256 rows 46.2 / 42.5, 384 rows 62.1 / 56.5, 1024 rows 127.5 / 114.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); }

__device__ __forceinline__ U4 philox4x32_10(U4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        // one 32 x 32 -> 64 multiply per product (v_mad_u64_u32) instead of a high and a low one: 32-bit integer
        // multiplies are what this generator costs, and the full-width form is 6.5 % faster over a logits pass
        const uint64_t p0 = (uint64_t)0xD2511F53u * (uint64_t)c.x, p1 = (uint64_t)0xCD9E8D57u * (uint64_t)c.z;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0, hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        c = U4{xor3(hi1, c.y, k0), lo1, xor3(hi0, c.w, k1), lo0};
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c;
}

// 32 random bits -> u = (top 23 bits + 1/2) / 2^23 in (0, 1) -> -ln(-ln u), the negated logarithm of a unit
// exponential.  With t = log2 u: -ln(-ln u) = -ln 2 * log2(-t) - ln(ln 2).  The largest noise values, the ones
// that decide an argmax, come from u next to 1, where t is tiny: the hardware logarithm keeps its relative
// accuracy there (over all 2^23 values of u the result is within 2e-6 of the fp64 one).
constexpr float kGumbelMax = 17.0f;      // above every value of gumbel_of (16.64 at u = 1 - 2^-24)
__device__ __forceinline__ float gumbel_of(uint32_t bits) {
    const float u = __builtin_fmaf((float)(bits >> 9), 1.1920928955078125e-07f, 5.9604644775390625e-08f);   // (k + 1/2) * 2^-23
    const float t = __builtin_amdgcn_logf(u);
    return __builtin_fmaf(-0.69314718055994531f, __builtin_amdgcn_logf(-t), 0.36651292058166435f);
}

struct RowNoise {                       // the generator's coordinates of one logits row
    uint32_t key0, key1, row, off_lo, off_hi;
    __device__ __forceinline__ U4 group(uint32_t column_group) const {
        return philox4x32_10(U4{column_group, row, off_lo, off_hi}, key0, key1);
    }
    __device__ __forceinline__ float at(int column) const {
        const U4 r = group((uint32_t)column >> 2);
        const uint32_t b[4] = {r.x, r.y, r.z, r.w};
        return gumbel_of(b[column & 3]);
    }
};

__device__ __forceinline__ RowNoise row_noise(const NoiseSpec& N, int64_t row) {
    const uint64_t off = N.offset + (N.offset_dev ? (uint64_t)*N.offset_dev : 0ull);
    const int64_t rid = N.row_ids ? N.row_ids[row] : row;
    return RowNoise{N.key0, N.key1, (uint32_t)rid, (uint32_t)off, (uint32_t)(off >> 32)};
}

inline NoiseSpec no_noise() { return NoiseSpec{nullptr, 0, false, 0, 0, 0, nullptr, nullptr}; }
inline NoiseSpec tensor_noise(const float* noise, int64_t stride) { NoiseSpec n = no_noise(); n.noise = noise; n.noise_row_stride = stride; return n; }
inline NoiseSpec generator_noise(uint64_t seed, uint64_t offset, const int64_t* offset_dev, const int64_t* row_ids) {
    NoiseSpec n = no_noise();
    n.philox = true; n.key0 = (uint32_t)seed; n.key1 = (uint32_t)(seed >> 32);
    n.offset = offset; n.offset_dev = offset_dev; n.row_ids = row_ids;
    return n;
}

}  // namespace mdx_noise
