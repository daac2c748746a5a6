// Fused producer of the attention inputs: per-head q/k RMSNorm, rotary embedding and the
// KV-cache store in one pass over the fused QKV projection output.
//
// Replaces, for one token, the chain
//   q = q_norm(q); k = k_norm(k)          nanovllm/models/sdar.py:79-81, layers/layernorm.py:16-26
//   q, k = rotary_emb(positions, q, k)    nanovllm/layers/rotary_embedding.py:6-14,37-48
//   store_kvcache(k, v, ...)              nanovllm/layers/sdar_attention.py:37-38, layers/attention.py:10-40
// which in the engine is about a dozen element-wise launches per layer.  It is a pure
// bandwidth op (reads 8 KiB of QKV per token, writes q, k and the two cache rows), so: a
// workgroup per token (for few tokens, several), 8 lanes per head row (qk_row.h).
#include "mdx_common.h"
#include "qk_row.h"
#include "split_sum.h"

namespace {

using namespace mdx_qk;

struct FusedParams {
    const __bf16* qkv; int64_t qkv_stride;        // or, with PARTIALS,
    const float* partials; int splits;            // [splits][tokens][rows * d]: the projection as K-split partial sums
    RowParams rows; int64_t n_tokens;
};

// A workgroup: THREADS / 8 head rows of one token at a time.  Everything that a head row waits for is asked for together.
template <int SLICES, int THREADS>
__global__ __launch_bounds__(THREADS) void qk_norm_rope_store_kernel(const FusedParams P)
{
    constexpr int kRows = THREADS / kLanesPerRow;
    const int64_t tok = (int)blockIdx.x + mdx::fetch_arguments<sizeof(FusedParams)>(gridDim.y);
    const int n_rows = P.rows.hq + 2 * P.rows.hkv;             // head rows of this token: q | k | v
    const int j = threadIdx.x % kLanesPerRow;
    const int64_t width = (int64_t)n_rows * kHeadDim;
    mdx_split::Eight<SLICES> a, b;
    RowWeight w;
    auto load = [&](int row) {
        const int64_t at = (int64_t)row * kHeadDim + 8 * j;
        const __bf16* x = P.qkv + tok * P.qkv_stride + at;
        const float* p = P.partials + tok * width + at;
        a.load(x, p, P.splits, P.n_tokens * width);
        b.load(x + 64, p + 64, P.splits, P.n_tokens * width);
        w = weight_of_row(P.rows, row, j);
    };
    int row = blockIdx.y * kRows + threadIdx.x / kLanesPerRow;
    if (row >= n_rows) return;
    load(row);
    const TokenPlace place = place_of_token(P.rows, tok, j);
    while (true) {
        finish_row(P.rows, tok, row, j, a.value(), b.value(), place, w);
        row += gridDim.y * kRows;
        if (row >= n_rows) return;
        load(row);
    }
}

}  // namespace

namespace {

int qk_norm_rope_store(const void* qkv, int64_t qkv_row_stride, const float* partials, int splits,
                                      const void* q_weight, const void* k_weight, float eps,
                                      const float* cos_table, const float* sin_table, int64_t max_positions,
                                      const int64_t* positions,
                                      void* q_out, int64_t q_out_row_stride,
                                      void* k_out, int64_t k_out_row_stride,
                                      void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_slots,
                                      int64_t n_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                      int32_t dtype, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(n_tokens >= 0 && num_q_heads > 0 && num_kv_heads > 0, MDX_EINVAL, "qk_norm_rope_store: bad size");
    MDX_REQUIRE(dtype == MDX_BF16, MDX_EUNSUPPORTED, "qk_norm_rope_store: dtype %d (only bf16)", dtype);
    MDX_REQUIRE(head_dim == kHeadDim, MDX_EUNSUPPORTED, "qk_norm_rope_store: head_dim %d (only 128)", head_dim);
    if (n_tokens == 0) return MDX_OK;
    MDX_REQUIRE((qkv || partials) && q_weight && k_weight && cos_table && sin_table && positions && q_out, MDX_EINVAL,
                "qk_norm_rope_store: null pointer");
    MDX_REQUIRE((k_cache == nullptr) == (v_cache == nullptr), MDX_EINVAL, "qk_norm_rope_store: give both caches or neither");
    MDX_REQUIRE(!k_cache || slot_mapping, MDX_EINVAL, "qk_norm_rope_store: caches without slot_mapping");
    MDX_REQUIRE(n_tokens < ((int64_t)1 << 31), MDX_EUNSUPPORTED, "qk_norm_rope_store: too many tokens");
    MDX_REQUIRE(mdx::aligned16(qkv) && mdx::aligned16(partials) && mdx::aligned16(q_out) && mdx::aligned16(q_weight) && mdx::aligned16(k_weight) &&
                (!k_out || mdx::aligned16(k_out)) && (!k_cache || (mdx::aligned16(k_cache) && mdx::aligned16(v_cache))) &&
                qkv_row_stride % 8 == 0 && q_out_row_stride % 8 == 0 && k_out_row_stride % 8 == 0,
                MDX_EUNSUPPORTED, "qk_norm_rope_store: tensors must be 16-byte aligned with row strides that are multiples of 8");
    MDX_REQUIRE(partials ? splits > 0 : qkv_row_stride >= (int64_t)(num_q_heads + 2 * num_kv_heads) * kHeadDim, MDX_EINVAL,
                "qk_norm_rope_store: qkv row stride shorter than a QKV row");
    FusedParams P;
    P.qkv = (const __bf16*)qkv; P.qkv_stride = qkv_row_stride; P.partials = partials; P.splits = splits;
    P.rows = RowParams{(const __bf16*)q_weight, (const __bf16*)k_weight, eps, cos_table, sin_table, max_positions, positions,
                       (__bf16*)q_out, q_out_row_stride, (__bf16*)k_out, k_out_row_stride, nullptr, 0,
                       (__bf16*)k_cache, (__bf16*)v_cache, slot_mapping, num_slots, num_q_heads, num_kv_heads};
    P.n_tokens = n_tokens;
    // A wavefront per workgroup while the chip has more CUs than there are tokens: 32 tokens of four slices are read by 128 CUs, not by 32
    // (one request through the engine, with the loads in flight together: 69.9 -> 69.3 ms).
    const int n_rows = num_q_heads + 2 * num_kv_heads;
    const dim3 spread((unsigned)n_tokens, (unsigned)std::min((n_rows + 7) / 8, 64));
    auto launch = [&](auto slices) {
        constexpr int N = decltype(slices)::value;
        if (n_tokens < mdx::compute_units()) qk_norm_rope_store_kernel<N, 64><<<spread, 64, 0, stream>>>(P);
        else qk_norm_rope_store_kernel<N, 256><<<(unsigned)n_tokens, 256, 0, stream>>>(P);
    };
    if (partials) mdx_split::with_slices(splits, launch);
    else launch(std::integral_constant<int, mdx_split::kNoSlices>());
    return mdx::check_launch("qk_norm_rope_store");
}

}  // namespace

extern "C" int mdx_qk_norm_rope_store(const void* qkv, int64_t qkv_row_stride,
                                      const void* q_weight, const void* k_weight, float eps,
                                      const float* cos_table, const float* sin_table, int64_t max_positions,
                                      const int64_t* positions,
                                      void* q_out, int64_t q_out_row_stride,
                                      void* k_out, int64_t k_out_row_stride,
                                      void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_slots,
                                      int64_t n_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                      int32_t dtype, mdx_stream_t stream_)
{
    return qk_norm_rope_store(qkv, qkv_row_stride, nullptr, 0, q_weight, k_weight, eps, cos_table, sin_table, max_positions, positions,
                              q_out, q_out_row_stride, k_out, k_out_row_stride, k_cache, v_cache, slot_mapping, num_slots,
                              n_tokens, num_q_heads, num_kv_heads, head_dim, dtype, stream_);
}

extern "C" int mdx_qk_norm_rope_store_partials(const float* partials, int32_t splits,
                                               const void* q_weight, const void* k_weight, float eps,
                                               const float* cos_table, const float* sin_table, int64_t max_positions,
                                               const int64_t* positions, void* q_out, int64_t q_out_row_stride,
                                               void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_slots,
                                               int64_t n_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                               int32_t dtype, mdx_stream_t stream)
{
    return qk_norm_rope_store(nullptr, 0, partials, splits, q_weight, k_weight, eps, cos_table, sin_table, max_positions, positions,
                              q_out, q_out_row_stride, nullptr, 0, k_cache, v_cache, slot_mapping, num_slots,
                              n_tokens, num_q_heads, num_kv_heads, head_dim, dtype, stream);
}
