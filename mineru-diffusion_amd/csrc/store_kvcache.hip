// store_kvcache: scatter of K/V rows into the paged cache.
//
// Pure HBM-bound copy (read 2 rows, write 2 rows per token), so there is no
// MFMA here: every lane moves 16 bytes, one small workgroup per row (a token's
// K row or its V row: one fully coalesced 2-KiB stream in, one out), loads and
// stores both nontemporal.  Measured on 38 k tokens of 2 x 2 KiB: this runs at
// the rate of a plain contiguous copy written the same way (6.0 TB/s read +
// written); four tokens per 256-thread workgroup with ordinary stores, the
// layout this replaced, reached 4.9, and the runtime's own device copy 5.2-5.4.
//
// Semantics follow engines/nano_dvlm/nanovllm/layers/attention.py:10-40.
#include "mdx_common.h"

namespace {

constexpr int kThreads = 256;

// Fast path: rows are multiples of 16 B, all bases and strides 16-B aligned.
// grid = (tokens, 2): blockIdx.y 0 copies the token's K row, 1 its V row.
// EARLY: the row is on its way before its slot is known, one trip to memory instead of two; rows that no slot takes are read in vain.  For launches whose workgroups
// are all on the chip at once, where that trip is what counts and such rows keep nobody waiting.  (us, the slot first / so: the store and the attention of one block behind 16 x 2300
// keys 43.2 / 43.0, fp32, 1056 keys 20.1 / 19.8; 1024 tokens 3.36 / 3.25, half of them without a slot 2.83 / 2.90, none with one 2.16 / 2.25; but 2048 tokens 4.73 / 4.56,
// 3.74 / 3.78, 2.50 / 2.84, and 38 434 57.9 / 58.2, 31.4 / 44.7, 17.8 / 26.2.)
constexpr int64_t kEarlyTokens = 1024;
template <bool EARLY>
__global__ __launch_bounds__(kThreads) void store_kvcache_vec16(
    const u32x4* __restrict__ key, const u32x4* __restrict__ value,
    int64_t k_stride16, int64_t v_stride16,
    u32x4* __restrict__ k_cache, u32x4* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping,
    int row16, int64_t num_slots)
{
    const int64_t tok = blockIdx.x;
    const bool is_v = blockIdx.y != 0;
    const u32x4* src = is_v ? value + tok * v_stride16 : key + tok * k_stride16;
    int c = threadIdx.x;
    u32x4 x{0, 0, 0, 0};
    if (EARLY && c < row16) x = __builtin_nontemporal_load(src + c);
    const int64_t s = slot_mapping[tok];
    if (s < 0 || s >= num_slots) return;
    if (!EARLY && c < row16) x = __builtin_nontemporal_load(src + c);
    u32x4* dst = (is_v ? v_cache : k_cache) + s * row16;
    while (c < row16) {
        __builtin_nontemporal_store(x, dst + c);
        c += blockDim.x;
        if (c < row16) x = __builtin_nontemporal_load(src + c);
    }
}

// Fallback for unaligned bases/strides or odd row sizes: element-wise copy.
template <typename E>
__global__ __launch_bounds__(kThreads) void store_kvcache_elem(
    const E* __restrict__ key, const E* __restrict__ value,
    int64_t k_stride, int64_t v_stride,
    E* __restrict__ k_cache, E* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping,
    int64_t n_tokens, int64_t row_elems, int64_t num_slots)
{
    const int64_t tok = blockIdx.x;
    if (tok >= n_tokens) return;
    const int64_t s = slot_mapping[tok];
    if (s < 0 || s >= num_slots) return;
    for (int64_t c = threadIdx.x; c < row_elems; c += kThreads) {
        k_cache[s * row_elems + c] = key[tok * k_stride + c];
        v_cache[s * row_elems + c] = value[tok * v_stride + c];
    }
}

}  // namespace

extern "C" int mdx_store_kvcache(const void* key, const void* value,
                                 int64_t k_row_stride, int64_t v_row_stride,
                                 void* k_cache, void* v_cache,
                                 const int32_t* slot_mapping,
                                 int64_t n_tokens, int64_t row_elems, int32_t elem_size,
                                 int64_t num_slots, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(n_tokens >= 0 && row_elems > 0 && num_slots >= 0, MDX_EINVAL,
                "store_kvcache: negative size (n_tokens=%lld row_elems=%lld num_slots=%lld)",
                (long long)n_tokens, (long long)row_elems, (long long)num_slots);
    MDX_REQUIRE(elem_size == 1 || elem_size == 2 || elem_size == 4 || elem_size == 8, MDX_EUNSUPPORTED,
                "store_kvcache: elem_size %d not in {1,2,4,8}", elem_size);
    if (n_tokens == 0) return MDX_OK;
    MDX_REQUIRE(key && value && k_cache && v_cache && slot_mapping, MDX_EINVAL, "store_kvcache: null pointer");
    MDX_REQUIRE(n_tokens < (int64_t)1 << 31, MDX_EUNSUPPORTED, "store_kvcache: n_tokens %lld too large", (long long)n_tokens);
    // key.stride(0) may be anything >= 0 for a broadcast, but rows are dense (attention.py:36-37).
    MDX_REQUIRE(k_row_stride >= 0 && v_row_stride >= 0, MDX_EUNSUPPORTED, "store_kvcache: negative row stride");

    const int64_t row_bytes = row_elems * elem_size;
    const bool vec_ok = row_bytes % 16 == 0 && (k_row_stride * elem_size) % 16 == 0 &&
                        (v_row_stride * elem_size) % 16 == 0 && mdx::aligned16(key) && mdx::aligned16(value) &&
                        mdx::aligned16(k_cache) && mdx::aligned16(v_cache) && row_bytes / 16 < (1 << 30);
    if (vec_ok) {
        const int row16 = (int)(row_bytes / 16);
        const int64_t ks16 = k_row_stride * elem_size / 16, vs16 = v_row_stride * elem_size / 16;
        // one lane per 16-byte chunk of the row, in whole wavefronts, up to 256 lanes (longer rows loop)
        int threads = (row16 + mdx::kWave - 1) / mdx::kWave * mdx::kWave;
        if (threads > kThreads) threads = kThreads;
        (n_tokens <= kEarlyTokens ? store_kvcache_vec16<true> : store_kvcache_vec16<false>)<<<dim3((unsigned)n_tokens, 2), threads, 0, stream>>>(
            (const u32x4*)key, (const u32x4*)value, ks16, vs16, (u32x4*)k_cache, (u32x4*)v_cache,
            slot_mapping, row16, num_slots);
    } else {
#define MDX_STORE_ELEM(E)                                                                         \
        store_kvcache_elem<E><<<(unsigned)n_tokens, kThreads, 0, stream>>>(                       \
            (const E*)key, (const E*)value, k_row_stride, v_row_stride, (E*)k_cache, (E*)v_cache, \
            slot_mapping, n_tokens, row_elems, num_slots)
        switch (elem_size) {
            case 1: MDX_STORE_ELEM(uint8_t); break;
            case 2: MDX_STORE_ELEM(uint16_t); break;
            case 4: MDX_STORE_ELEM(uint32_t); break;
            default: MDX_STORE_ELEM(uint64_t); break;
        }
#undef MDX_STORE_ELEM
    }
    return mdx::check_launch("store_kvcache");
}
