// One head row (q, k or v of a token) between the QKV projection and the attention: RMSNorm, rotary embedding and the cache store,
// shared by the kernel that reads the projection's output (qk_norm_rope_store.hip) and the projection itself (linear.hip).
//
// Eight lanes per row, each holding elements [8 j, 8 j + 8) and [64 + 8 j, 64 + 8 j + 8), which are exactly the pairs the
// rotation mixes, so no data crosses lanes except the 8-lane sum of squares.
//
// Rounding follows the reference: the normalised value is rounded to the storage type, then
// multiplied by the weight in the storage type (nanovllm/layers/layernorm.py:24-25); the rotation is done in
// fp32 and rounded once (layers/rotary_embedding.py:11-14).
#pragma once
#include "mdx_common.h"

namespace mdx_qk {

constexpr int kHeadDim = 128, kLanesPerRow = 8;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

struct RowParams {
    const __bf16* q_w; const __bf16* k_w; float eps;
    const float* cos_t; const float* sin_t; int64_t max_pos; const int64_t* positions;
    __bf16* q_out; int64_t q_out_stride;
    __bf16* k_out; int64_t k_out_stride;          // may be null
    __bf16* v_out; int64_t v_out_stride;          // may be null
    __bf16* k_cache; __bf16* v_cache;             // both may be null
    const int32_t* slot_mapping; int64_t num_slots;
    int hq, hkv;
};

struct TokenPlace { float cs[8], sn[8]; int64_t slot; };   // lane j's part of the token's rotation; its cache slot or -1

__device__ __forceinline__ TokenPlace place_of_token(const RowParams& P, int64_t tok, int j) {
    TokenPlace t;
    t.slot = -1;
    if (P.k_cache && P.slot_mapping) {
        const int64_t s = P.slot_mapping[tok];
        if (s >= 0 && s < P.num_slots) t.slot = s;
    }
    const int64_t pos = P.positions[tok];
    const bool pos_ok = pos >= 0 && pos < P.max_pos;        // out-of-table positions rotate by 0
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        t.cs[e] = pos_ok ? P.cos_t[pos * (kHeadDim / 2) + 8 * j + e] : 1.0f;
        t.sn[e] = pos_ok ? P.sin_t[pos * (kHeadDim / 2) + 8 * j + e] : 0.0f;
    }
    return t;
}

struct RowWeight { bf16x8 a, b; };      // the norm's weight for lane j's columns; of a v row, nothing

__device__ __forceinline__ RowWeight weight_of_row(const RowParams& P, int row, int j) {
    RowWeight w;
    if (row < P.hq + P.hkv) {
        const __bf16* src = (row < P.hq ? P.q_w : P.k_w) + 8 * j;
        w.a = *reinterpret_cast<const bf16x8*>(src);
        w.b = *reinterpret_cast<const bf16x8*>(src + 64);
    }
    return w;
}

// row: head row of the token, q | k | v.  The 8 lanes of a row call it together.
__device__ __forceinline__ void finish_row(const RowParams& P, int64_t tok, int row, int j, bf16x8 a, bf16x8 b, const TokenPlace& t,
                                           const RowWeight& w) {
    const bool is_q = row < P.hq, is_k = !is_q && row < P.hq + P.hkv;
    if (is_q || is_k) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) { const float x = (float)a[e], y = (float)b[e]; ss += x * x + y * y; }
        ss += mdx::xor_lanes(ss, 1);
        ss += mdx::xor_lanes(ss, 2);
        ss += mdx::xor_lanes(ss, 4);
        const float inv = rsqrtf(ss * (1.0f / kHeadDim) + P.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x1 = (float)(__bf16)((float)(__bf16)((float)a[e] * inv) * (float)w.a[e]);
            const float x2 = (float)(__bf16)((float)(__bf16)((float)b[e] * inv) * (float)w.b[e]);
            a[e] = (__bf16)(x1 * t.cs[e] - x2 * t.sn[e]);
            b[e] = (__bf16)(x2 * t.cs[e] + x1 * t.sn[e]);
        }
    }
    auto store = [&](__bf16* dst) {
        *reinterpret_cast<bf16x8*>(dst + 8 * j) = a;
        *reinterpret_cast<bf16x8*>(dst + 64 + 8 * j) = b;
    };
    if (is_q) { store(P.q_out + tok * P.q_out_stride + (int64_t)row * kHeadDim); return; }
    const int kvrow = is_k ? row - P.hq : row - P.hq - P.hkv;
    if (is_k && P.k_out) store(P.k_out + tok * P.k_out_stride + (int64_t)kvrow * kHeadDim);
    if (!is_k && P.v_out) store(P.v_out + tok * P.v_out_stride + (int64_t)kvrow * kHeadDim);
    if (t.slot >= 0) store((is_k ? P.k_cache : P.v_cache) + (t.slot * P.hkv + kvrow) * kHeadDim);
}

}  // namespace mdx_qk
