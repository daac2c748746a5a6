// Rows of 16-bit logits as ordered keys: what the top-k / top-p filters of logit_filter.hip and filtered_pick.hip share.
#pragma once
#include "mdx_common.h"
#include <hip/hip_fp16.h>

namespace mdx_keys {

constexpr float kLog2e = 1.4426950408889634f;

template <typename T> struct Bits16;
template <> struct Bits16<__bf16> {
    static constexpr uint32_t kNegInf = 0xff80u;
    static __device__ __forceinline__ float value(uint32_t b) { return __uint_as_float(b << 16); }
};
template <> struct Bits16<__half> {
    static constexpr uint32_t kNegInf = 0xfc00u;
    static __device__ __forceinline__ float value(uint32_t b) { return __half2float(__ushort_as_half((unsigned short)b)); }
};

// Bit pattern -> key that grows with the value (-0 counts as +0); and back.
__device__ __forceinline__ uint32_t key_of(uint32_t b) {
    if (b == 0x8000u) b = 0;
    return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
}
__device__ __forceinline__ uint32_t bits_of(uint32_t k) { return (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu); }
template <typename T> __device__ __forceinline__ float value_of_key(uint32_t k) { return Bits16<T>::value(bits_of(k)); }

// The vocabulary pass takes no element at or below this for a row's largest: a row that holds no other has no confidence.
constexpr float kNoConfidence = -3.0e38f;

struct RowView {                        // a row as scalar head, aligned 16-byte chunks, scalar tail
    const uint16_t* p;
    const u32x4* chunks;
    int lead, nchunk, tail0, vocab;
};

__device__ __forceinline__ RowView row_view(const uint16_t* p, int vocab) {
    RowView r;
    r.p = p;
    r.vocab = vocab;
    r.lead = min((int)(((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / 2), vocab);
    r.nchunk = (vocab - r.lead) / 8;
    r.tail0 = r.lead + r.nchunk * 8;
    r.chunks = reinterpret_cast<const u32x4*>(p + r.lead);
    return r;
}

// f(bits, index) for every element of the row, shared out over a workgroup of THREADS; loads run four chunks ahead.
template <int THREADS, typename F>
__device__ __forceinline__ void scan_row(const RowView& r, int tid, F f) {
    constexpr int kAhead = 4;
    for (int e = tid; e < r.lead; e += THREADS) f((uint32_t)r.p[e], e);
    u32x4 next[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) if (tid + i * THREADS < r.nchunk) next[i] = r.chunks[tid + i * THREADS];
    for (int ch = tid; ch < r.nchunk; ch += THREADS) {
        const u32x4 u = next[0];
#pragma unroll
        for (int i = 0; i + 1 < kAhead; ++i) next[i] = next[i + 1];
        if (ch + kAhead * THREADS < r.nchunk) next[kAhead - 1] = r.chunks[ch + kAhead * THREADS];
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { f(w[i] & 0xffffu, r.lead + 8 * ch + 2 * i); f(w[i] >> 16, r.lead + 8 * ch + 2 * i + 1); }
    }
    for (int e = r.tail0 + tid; e < r.vocab; e += THREADS) f((uint32_t)r.p[e], e);
}

// Softmax terms relative to the row's maximum, at most 1 each, are summed as 64-bit integers in units of 2^-40: the sum does not
// depend on the order of the additions (candidate lists have none), is exact for rows of up to 2^23 elements, and a row of 2^18
// loses at most 2^-23 of its largest term to the rounding of its smallest.  NaN weighs nothing.
constexpr float kMassScale = 1099511627776.f;        // 2^40
typedef unsigned long long Mass;
__device__ __forceinline__ Mass mass_of(float term) { return term > 0.f ? (Mass)__builtin_rintf(term * kMassScale) : 0ull; }
// What a cumulative mass has to exceed for a share of the whole.
__device__ __forceinline__ Mass share_of(Mass total, float share) { return (Mass)((double)share * (double)total); }
// The terms are at most 1: neither an unbounded maximum nor a temperature that is zero, negative or not a number.
__device__ __forceinline__ bool has_masses(float m, float c) { return m > -INFINITY && m < INFINITY && c >= 0.f && c < INFINITY; }

template <typename V> __device__ __forceinline__ V wave_total(V v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += mdx::xor_lanes(v, off);
    return v;
}

// The sum over a workgroup, known to every thread; the order of the additions is fixed.  `slot`: one V per wavefront in LDS.
template <int THREADS, typename V> __device__ __forceinline__ V block_total(V v, V* slot, int tid) {
    v = wave_total(v);
    __syncthreads();                                            // earlier readers of the slots are done
    if ((tid & 63) == 0) slot[tid >> 6] = v;
    __syncthreads();
    V sum = slot[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) sum += slot[w];
    return sum;
}

// The filter's cut-off key of a row, bit by bit, a pass over the row for each: for rows that the fast forms do not hold (more
// than 65 535 equal values, or more ties at the k-th largest than a candidate list).  Every pass counts, or weighs, the
// elements at or above a trial key: the k-th largest key is the largest that k elements reach, the top-p cut-off the largest
// whose elements weigh more than the share asked for.  0 = everything is kept.
template <typename T, int THREADS>
__device__ uint32_t floor_by_bisection(const RowView& row, int tid, int top_k, float top_p, float c, Mass* mslot, int* islot) {
    uint32_t floor_key = 0, mk = 0;
    if (top_k > 0 && top_k < row.vocab) {
        for (int bit = 15; bit >= 0; --bit) {
            const uint32_t trial = floor_key | (1u << bit);
            int n = 0;
            scan_row<THREADS>(row, tid, [&](uint32_t b, int) { n += key_of(b) >= trial ? 1 : 0; });
            if (block_total<THREADS>(n, islot, tid) >= top_k) floor_key = trial;
        }
    }
    if (top_p < 1.0f) {
        scan_row<THREADS>(row, tid, [&](uint32_t b, int) { mk = max(mk, key_of(b)); });
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) mk = max(mk, (uint32_t)mdx::xor_lanes((int)mk, off));
        __syncthreads();
        if ((tid & 63) == 0) islot[tid >> 6] = (int)mk;
        __syncthreads();
        for (int w = 0; w < THREADS / 64; ++w) mk = max(mk, (uint32_t)islot[w]);
        const float m = value_of_key<T>(mk);
        if (has_masses(m, c)) {                                 // a row whose largest element is not finite has no softmax to take a share of
            auto mass_from = [&](uint32_t from) {
                Mass a = 0;
                scan_row<THREADS>(row, tid, [&](uint32_t b, int) { if (key_of(b) >= from) a += mass_of(__builtin_amdgcn_exp2f((Bits16<T>::value(b) - m) * c)); });
                return block_total<THREADS>(a, mslot, tid);
            };
            const Mass target = share_of(mass_from(floor_key), top_p);
            uint32_t key = 0;
            for (int bit = 15; bit >= 0; --bit) {
                const uint32_t trial = key | (1u << bit);
                if (trial <= mk && mass_from(max(trial, floor_key)) > target) key = trial;
            }
            floor_key = max(floor_key, key);
        }
    }
    return floor_key;
}

}  // namespace mdx_keys
