// Staircase block-prefill attention in fp32 arithmetic: the form of mdx_staircase_attn_varlen for fp32
// q/k/v/o and for heads that the 16-bit kernels of staircase_attn.hip do not take (wider than 128 columns,
// up to 256, or not a multiple of 16).  The reference's kernel accepts any q.dtype and any head_dim
// (engines/nano_dvlm/nanovllm/kernels/triton/attention/block_prefill_attention_v2.py:16-199:
// BLOCK_DMODEL = head_dim, o = empty_like(q)); the model itself runs bf16 with d = 128, so this is the path
// for callers outside the model's own configuration.  Arithmetic and layout: attn_f32_tile.h.
//
// A workgroup of 4 wavefronts owns 128 / KW padded query rows of one (sequence, head), KW wavefronts every 32 of them: each takes
// every KW-th tile of 32 keys, KW tiles (K and V as fp32) are staged through LDS at a time, and the KW states fold at the end.
// The matrix instruction bounds it, 8192 cycles per wavefront and tile, and its last row group sees all keys, so a launch
// that does not fill the chip lasts as long as that group's chain of tiles: KW divides the chain.
//
// The mask is the reference's (:98-102,137-139): with nb = ceil(L / S) blocks right-aligned, pad = nb S - L,
// query row i sees key j iff j <= ((i + pad) / S + 1) S - 1 - pad.
#include "attn_f32_tile.h"
#include <atomic>

namespace {

using namespace mdx_attn_f32;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

struct WideParams {
    const void* q; const void* k; const void* v; void* o;
    int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh;    // strides in elements
    const int32_t* cu_seqlens;
    int batch, total_tokens, n_row_groups, num_q_heads, num_kv_heads, head_dim, log2_s;
    float c;                                                   // scale * log2(e)
};

// T: element type of q/k/v/o.  D: 128 or 256, the head width that registers and LDS are laid out for.
template <typename T, int D, int KW>
__global__ __launch_bounds__(kThreads, D <= 128 && KW <= 2 ? 2 : 1) void staircase_attn_f32_kernel(const WideParams P)
{
    constexpr int kRowsPerWg = 32 * kWaves / KW;
    extern __shared__ __attribute__((aligned(16))) float lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kw = wave % KW;
    const int H = lane >> 5, r = lane & 31;
    const int head = blockIdx.x;
    const int rg = P.n_row_groups - 1 - (int)blockIdx.y;       // the heaviest row groups start first
    const int b = (int)blockIdx.z + mdx::fetch_arguments<sizeof(WideParams)>();

    // bounds that do not describe a range inside the packed tensors (decreasing, negative, past total_tokens) are clipped
    // to one, so that no row outside q/k/v/o is ever touched
    const int seq0 = min(max(P.cu_seqlens[b], 0), P.total_tokens);
    const int L = min(max(P.cu_seqlens[b + 1], seq0), P.total_tokens) - seq0;
    if (L <= 0) return;
    const int S = 1 << P.log2_s;
    const int Lp = ((L + S - 1) >> P.log2_s) << P.log2_s;      // padded length
    const int pad = Lp - L;
    const int row_g0 = rg * kRowsPerWg;                        // first padded row of the workgroup
    if (row_g0 >= Lp) return;
    const int kvh = head / (P.num_q_heads / P.num_kv_heads);
    const int width = P.head_dim;

    const T* kb = static_cast<const T*>(P.k) + (int64_t)kvh * P.k_sh;
    const T* vb = static_cast<const T*>(P.v) + (int64_t)kvh * P.v_sh;

    // ---- this lane's query ----
    const int row_w0 = row_g0 + wave / KW * 32;
    const int ip = row_w0 + r;                                 // padded query row
    const bool row_ok = ip >= pad && ip < Lp;
    const int64_t tok = (int64_t)seq0 + (ip - pad);
    float q[D / 2];
    const T* qb = static_cast<const T*>(P.q) + ((int64_t)seq0 - pad) * P.q_st + (int64_t)head * P.q_sh;      // padded row 0
    QueryRegs<T, D, kWaves / KW, kThreads> queries;
    if constexpr (KW == 1) load_q<T, D>(q, row_ok ? qb + ip * P.q_st : nullptr, H, width);                   // (more of them than tiles in LDS)
    else queries.fetch(tid, width, [&](int row) { const int i = row_g0 + row; return i >= pad && i < Lp ? qb + i * P.q_st : nullptr; });

    // exclusive key limit (padded coordinates) of a row
    auto limit_of = [&](int row) { return min(Lp, ((row >> P.log2_s) + 1) << P.log2_s); };
    const int key_hi = limit_of(ip);
    const int wave_hi = (row_w0 < Lp) ? limit_of(min(row_w0 + 31, Lp - 1)) : 0;    // 0: idle wavefront
    const int wg_hi = limit_of(min(row_g0 + kRowsPerWg - 1, Lp - 1));
    const int n_tiles = (wg_hi + kTileKeys - 1) / kTileKeys;

    State<D> st;
    st.init();
    // the next tile is on its way (its first batch, in registers) while this one is multiplied; rows outside the sequence: its
    // first one, zeroed later
    TileRegs<T, D, kThreads> regs;
    auto fetch = [&](int t, int batch) {
        auto tok_of = [&](int row) { const int jp = t * kTileKeys + row; return (int64_t)seq0 + (jp >= pad && jp < Lp ? jp - pad : 0); };
        regs.fetch(batch, tid, width, [&](int row) { return kb + tok_of(row) * P.k_st; }, [&](int row) { return vb + tok_of(row) * P.v_st; });
    };
    fetch(0, 0);
    if constexpr (KW > 1) {
        static_assert(queries.kBytes <= KW * Lds<D>::kBytes, "queries exceed the tile region");
        queries.write(lds, tid);
        __syncthreads();
        queries.read(q, lds, wave / KW, H, r, width);
    }
    for (int t = 0; t < n_tiles; t += KW) {
        __syncthreads();                                       // the previous tiles have been read by everybody
#pragma unroll
        for (int i = 0; i < KW; ++i) {
#pragma unroll
            for (int batch = 0; batch < regs.kBatches; ++batch) {
                if (i + batch > 0) fetch(t + i, batch);
                regs.write(batch, lds + i * Lds<D>::kFloats, tid, width, [&](int row) { const int jp = (t + i) * kTileKeys + row; return jp >= pad && jp < Lp; });
            }
        }
        if (t + KW < n_tiles) fetch(t + KW, 0);
        __syncthreads();
        const int key0 = (t + kw) * kTileKeys;
        if (key0 >= wave_hi || key0 + kTileKeys <= pad) continue;        // nothing of this tile is visible to this wavefront
        tile_step<D>(lds + kw * Lds<D>::kFloats, q, st, P.c, width, lane, [&](int key) { const int kj = key0 + key; return kj >= pad && kj < key_hi; });
    }
    static_assert(KW == 1 || kWaves * kStateBytes<D> <= KW * Lds<D>::kBytes, "merge buffer exceeds the tile region");
    T* orow = static_cast<T*>(P.o) + tok * P.o_st + (int64_t)head * P.o_sh;
    fold_states<D, KW>(lds, st, wave, lane, width, [&](int d, f32x4 acc) {
        const float inv = st.l > 0.f ? 1.0f / st.l : 0.f;
        if (row_ok) store4(orow + d, f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv});
    });
}

template <typename T, int D, int KW>
int launch_split(WideParams P, int64_t max_l, hipStream_t stream)
{
    constexpr int kRowsPerWg = 32 * kWaves / KW, kLdsBytes = KW * Lds<D>::kBytes;
    max_l = max_l < P.total_tokens ? max_l : P.total_tokens;
    P.n_row_groups = (int)((max_l + (1 << P.log2_s) - 1 + kRowsPerWg - 1) / kRowsPerWg);
    MDX_REQUIRE(P.batch <= 65535 && P.n_row_groups <= 65535, MDX_EUNSUPPORTED,
                "staircase_attn: fp32 arithmetic takes up to 65535 sequences of up to 8 M tokens");
    // the kernel's LDS limit is raised once per device
    static std::atomic<bool> raised[64];
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "staircase_attn: no current device (%s)", hipGetErrorString(e));
    if (!raised[device].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(staircase_attn_f32_kernel<T, D, KW>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
        MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "staircase_attn: cannot reserve %d bytes of LDS (%s)", kLdsBytes, hipGetErrorString(e));
        raised[device].store(true, std::memory_order_release);
    }
    const dim3 grid((unsigned)P.num_q_heads, (unsigned)P.n_row_groups, (unsigned)P.batch);
    staircase_attn_f32_kernel<T, D, KW><<<grid, kThreads, kLdsBytes, stream>>>(P);
    return mdx::check_launch("staircase_attn (fp32 arithmetic)");
}

// How many wavefronts share a row tile's keys, from the number of row tiles R (all heads) and the longest prompt.  While the
// launch leaves compute units idle the longest chain of tiles counts: four, as soon as there are tiles for them and their
// workgroups (135 KB of LDS, one per CU) come in one round, or in three if the chain is long enough to pay for those.  Then
// two, as long as the row groups' unequal chains leave a ragged end (to 16 row tiles per CU); prompts of two tiles have nothing
// to share once the chip is full, and the fold at the end costs about one tile.  Measured (1 / 2 / 4 wavefronts, 16 query
// heads, us): 100 tokens 25 / 16 / 12, 500 85 / 50 / 33, 1024 164 / 94 / 71, 2000 320 / 235 / 244, 4096 855 / 694 / 916,
// 8192 2539 / 2452 / 3527, 8 x 250 59 / 44 / 64, 16 x 64 15 / 18 / 23, 4 x 2048 788 / 680 / 970, 4 x 4096 2438 / 2519 / 3680.
template <typename T>
int launch(const WideParams& P, int64_t max_l, hipStream_t stream)
{
    if (P.head_dim > 128) return launch_split<T, 256, 1>(P, max_l, stream);
    const int64_t row_tiles = ((int64_t)P.total_tokens / 32 + P.batch) * P.num_q_heads, cus = mdx::compute_units();
    if (max_l > 64 && row_tiles <= (max_l < 384 ? cus : 3 * cus)) return launch_split<T, 128, 4>(P, max_l, stream);
    if (row_tiles <= (max_l <= 64 ? cus : 16 * cus)) return launch_split<T, 128, 2>(P, max_l, stream);
    return launch_split<T, 128, 1>(P, max_l, stream);
}

}  // namespace

namespace mdx {

// Called by mdx_staircase_attn_varlen, which has checked sizes, head counts, staircase size and scale, for
// dtype MDX_F32 and for head widths outside the 16-bit kernels'.
int launch_staircase_f32(const void* q, const void* k, const void* v, void* o,
                         int64_t q_stride_t, int64_t q_stride_h, int64_t k_stride_t, int64_t k_stride_h,
                         int64_t v_stride_t, int64_t v_stride_h, int64_t o_stride_t, int64_t o_stride_h,
                         const int32_t* cu_seqlens, int32_t batch, int64_t max_l, int64_t total_tokens,
                         int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                         int32_t log2_s, float scale, int32_t dtype, hipStream_t stream)
{
    MDX_REQUIRE(head_dim >= 4 && head_dim <= 256 && head_dim % 4 == 0, MDX_EUNSUPPORTED,
                "staircase_attn: head_dim %d (fp32 arithmetic: multiples of 4 up to 256)", head_dim);
    const uintptr_t align = dtype == MDX_F32 ? 15u : 7u;       // four elements per access
    MDX_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) & align) == 0 &&
                q_stride_t % 4 == 0 && q_stride_h % 4 == 0 && k_stride_t % 4 == 0 && k_stride_h % 4 == 0 &&
                v_stride_t % 4 == 0 && v_stride_h % 4 == 0 && o_stride_t % 4 == 0 && o_stride_h % 4 == 0,
                MDX_EUNSUPPORTED, "staircase_attn: q/k/v/o must be aligned to four elements with strides that are multiples of 4 elements");
    WideParams P;
    P.q = q; P.k = k; P.v = v; P.o = o;
    P.q_st = q_stride_t; P.q_sh = q_stride_h; P.k_st = k_stride_t; P.k_sh = k_stride_h;
    P.v_st = v_stride_t; P.v_sh = v_stride_h; P.o_st = o_stride_t; P.o_sh = o_stride_h;
    P.cu_seqlens = cu_seqlens;
    P.batch = batch;
    P.total_tokens = (int)total_tokens;
    P.n_row_groups = 0;                                        // with the split
    P.num_q_heads = num_q_heads; P.num_kv_heads = num_kv_heads; P.head_dim = head_dim; P.log2_s = log2_s;
    P.c = scale * kLog2e;
    switch (dtype) {
    case MDX_F32:  return launch<float>(P, max_l, stream);
    case MDX_F16:  return launch<_Float16>(P, max_l, stream);
    case MDX_BF16: return launch<__bf16>(P, max_l, stream);
    }
    return mdx::fail(MDX_EUNSUPPORTED, "staircase_attn: dtype %d", dtype);
}

}  // namespace mdx
