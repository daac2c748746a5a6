// Paged single-block ("decode") attention in fp32 arithmetic: the form of mdx_paged_block_attn for fp32
// tensors and for heads that the 16-bit kernel of paged_attn.hip does not take (wider than 128 columns,
// up to 256, or not a multiple of 16).  flash_attn_with_kvcache, which this call replaces
// (engines/nano_dvlm/nanovllm/layers/sdar_attention.py:48-56), takes heads of up to 256 columns; the model
// itself runs bf16 with d = 128, so this is the path for callers outside the model's own configuration.
// Arithmetic and layout: attn_f32_tile.h.
//
// What bounds it is the fp32 matrix instruction: 128 of them, 64 cycles each, per wavefront, head and tile of 32 keys.  So
// the contexts are cut into pieces of keys until the chip's wavefront slots are filled (one sequence of 1056 keys is 16 x 33
// such steps for 1024 SIMDs), the pieces' states go to fp32 partials in the workspace, and a second, small launch folds
// them.  (One workgroup per sequence and query head walking the whole context, the form this replaced, left 240 of 256 CUs
// idle on that shape: 84 us.)
//
// A workgroup serves one (sequence, piece, group of HPW query heads that share a KV head, tile of 32 queries): HPW x KW
// wavefronts, each on one head and every KW-th tile of 32 keys, KW tiles staged at a time.  Two query heads per workgroup
// halve what is staged per product, and with 68 KB of LDS two workgroups share a CU, so that one stages while the other
// multiplies.
// The semantics are those of the 16-bit kernel: non-causal, the first min(context_lens[b], max_pages x
// page_size) keys through block_table[b]; keys on a page id outside [0, num_pages) are left out; a sequence
// without any key yields zeros.
#include "attn_f32_tile.h"
#include <atomic>

namespace {

using namespace mdx_attn_f32;

struct PagedWideParams {
    const void* q; void* o; const void* k_cache; const void* v_cache;
    int64_t q_sb, q_ss, q_sh, o_sb, o_ss, o_sh;     // element strides
    int64_t c_sp, c_st, c_sh;                       // cache strides: page, token, head
    const int32_t* block_table; int64_t bt_stride;
    const int32_t* context_lens;
    int bs, sq, nqt, num_q_heads, heads_per_kv, page_size, page_shift, max_pages, head_dim;   // page_shift: log2(page_size) or -1
    int64_t num_pages;
    float c;                                        // scale * log2(e)
    int nsplit, pieces;                             // partial slots per sequence; pieces the whole launch should be cut into per (head group, query tile)
    float* part_o; float* part_ml;                  // [bs, Hq, nqt, nsplit, 32, D] and [bs, Hq, nqt, nsplit, 2, 32]
};

constexpr int kLeastKeys = 64;                      // keys of a piece: a multiple of this
constexpr int kMaxSplits = 64;

__device__ __forceinline__ int keys_of(const PagedWideParams& P, int b) {
    const int64_t room = (int64_t)P.max_pages * P.page_size;
    const int raw = P.context_lens[b];
    return max(0, (int)(raw < room ? raw : room));
}

// Keys per piece of sequence b (all wavefronts of both kernels find the same).  Pieces of one size for all sequences, so that a
// long sequence gets more of them and all workgroups run equally long: total keys / pieces, but never more pieces of a
// sequence than it has slots.  Beyond 64 sequences, whose lengths no wavefront holds, a sequence is cut evenly.
// QUICK: the sum by DPP shifts, 1200 cycles less of a workgroup's start.  Not in launches of several rounds per piece: there it is up to 2 % slower where all workgroups are equal
// (us, by shuffles / by shifts: 1 x 16 300 keys 65.4 / 67.2, 1 x 14 000 63.8 / 64.9, 4 x 4000 73.6 / 74.5; but 8 x 300-2000 64.2 / 62.4).  Probably the two
// workgroups of a CU stay in step then, stage at the same time and multiply at the same time; a wave priority for one of them undid that there and cost 1 % elsewhere.
template <bool QUICK>
__device__ __forceinline__ int keys_per_piece(const PagedWideParams& P, int ctx, int lane) {
    int want = (ctx + P.nsplit - 1) / P.nsplit;
    if (P.bs <= 64) {
        int total = lane < P.bs ? keys_of(P, lane) : 0;
        if (QUICK) total = mdx::wave_sum(total);
#pragma unroll
        for (int off = 32; !QUICK && off >= 1; off >>= 1) total += __shfl_xor(total, off);
        want = max(want, (total + P.pieces - 1) / P.pieces);
    }
    return max(1, (want + kLeastKeys - 1) / kLeastKeys) * kLeastKeys;
}

// ONE_ROUND: pieces of KW tiles at most, whose loads are on their way before the queries go through LDS and their pages are looked up in a register.  (Where there
// are more rounds the same start, or the next round's loads ahead of the products, is slower: 1 x 4000 keys 34.9 -> 35.5 us, 1 x 16 000 66 -> 67.5 and 70.)
template <typename T, int D, int HPW, int KW, bool ONE_ROUND>
__global__ __launch_bounds__(64 * HPW * KW, D <= 128 && KW <= 2 ? 2 : 1) void paged_attn_f32_kernel(const PagedWideParams P)
{
    constexpr int kThreads = 64 * HPW * KW;
    constexpr int kTileFloats = Lds<D>::kFloats;
    extern __shared__ __attribute__((aligned(16))) float lds[];          // KW tiles (K and V of 32 keys each), or the states to merge

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int H = lane >> 5, r = lane & 31;
    const int kw = wave % KW, hw = wave / KW;
    const int head = (blockIdx.x / P.nqt) * HPW + hw, qt = blockIdx.x % P.nqt, split = blockIdx.y, b = blockIdx.z;
    const int kvh = (blockIdx.x / P.nqt) * HPW / P.heads_per_kv;
    const int width = P.head_dim;

    QueryRegs<T, D, HPW, kThreads> queries;
    const int ctx = keys_of(P, b);
    const T* q0 = static_cast<const T*>(P.q) + (int64_t)b * P.q_sb + (int64_t)(qt * 32) * P.q_ss + (int64_t)(head - hw) * P.q_sh;
    queries.fetch(tid, width, [&](int row) { return qt * 32 + row % 32 < P.sq ? q0 + (int64_t)(row % 32) * P.q_ss + (int64_t)(row / 32) * P.q_sh : nullptr; });
    const int span = P.nsplit > 1 ? keys_per_piece<ONE_ROUND>(P, ctx, lane) : max(1, ctx);
    const int n_pieces = max(1, (ctx + span - 1) / span);
    if (split >= n_pieces) return;
    const int key_begin = split * span, key_end = min(ctx, key_begin + span);
    const int32_t* bt = P.block_table + (int64_t)b * P.bt_stride;
    const int n_tiles = (key_end - key_begin + kTileKeys - 1) / kTileKeys;

    const int qrow = qt * 32 + r;                   // this lane's query of the sequence's block
    const bool row_ok = qrow < P.sq;
    const T* kc = static_cast<const T*>(P.k_cache) + (int64_t)kvh * P.c_sh;
    const T* vc = static_cast<const T*>(P.v_cache) + (int64_t)kvh * P.c_sh;

    float q[D / 2];
    auto hand_out_queries = [&] {
        queries.write(lds, tid);
        __syncthreads();
        queries.read(q, lds, hw, H, r, width);
    };
    if (!ONE_ROUND) hand_out_queries();
    const int first_slot = P.page_shift >= 0 ? key_begin >> P.page_shift : key_begin / P.page_size;
    const int pages = ONE_ROUND ? bt[min(first_slot + lane, P.max_pages - 1)] : 0;
    State<D> st;
    st.init();
    for (int t0 = 0; t0 < (ONE_ROUND ? 1 : n_tiles); t0 += KW) {
        // ---- tiles t0 .. t0 + KW - 1 into LDS, all threads on each (a tile never straddles a page: page_size % 32 == 0, so that all
        //      its rows exist in memory, whatever they hold) ----
        unsigned tile_ok = 0;                                  // bit i: tile t0 + i exists and lies on a valid page (uniform)
        // tiles whose loads are in flight together: as registers allow (two instead of one at 128 columns: 8 x 4000-9000 keys
            // 192 -> 186 us, 1 x 4000 35.2 -> 34.4, 1 x 1056 and shorter level)
            constexpr int kTogether = KW == 4 ? 4 : D <= 128 ? KW : 1;
            static_assert(!ONE_ROUND || (kTogether == KW && TileRegs<T, D, kThreads>::kBatches == 1), "a round in registers");
        TileRegs<T, D, kThreads> regs[kTogether];
#pragma unroll
        for (int i0 = 0; i0 < KW; i0 += kTogether) {
            int64_t base[kTogether];
#pragma unroll
            for (int j = 0; j < kTogether; ++j) {
                const int key0 = key_begin + (t0 + i0 + j) * kTileKeys;
                const int page_slot = P.page_shift >= 0 ? key0 >> P.page_shift : key0 / P.page_size;
                const int64_t page = key0 >= key_end ? -1 : ONE_ROUND ? __builtin_amdgcn_readlane(pages, page_slot - first_slot) : bt[page_slot];
                if (page >= 0 && page < P.num_pages) tile_ok |= 1u << (i0 + j);
                base[j] = page * P.c_sp + (int64_t)(key0 - page_slot * P.page_size) * P.c_st;
            }
#pragma unroll 1
            for (int b = 0; b < regs[0].kBatches; ++b) {
#pragma unroll
                for (int j = 0; j < kTogether; ++j)
                    if ((tile_ok >> (i0 + j)) & 1u)
                        regs[j].fetch(b, tid, width, [&](int row) { return kc + base[j] + (int64_t)row * P.c_st; }, [&](int row) { return vc + base[j] + (int64_t)row * P.c_st; });
                if (ONE_ROUND) hand_out_queries();
                if (i0 == 0 && b == 0) __syncthreads();        // the queries or the previous tiles have been read by everybody
#pragma unroll
                for (int j = 0; j < kTogether; ++j)
                    if ((tile_ok >> (i0 + j)) & 1u)
                        regs[j].write(b, lds + (i0 + j) * kTileFloats, tid, width, [&](int row) { return key_begin + (t0 + i0 + j) * kTileKeys + row < key_end; });
            }
        }
        __syncthreads();
        if ((tile_ok >> kw) & 1u) {
            const int key0 = key_begin + (t0 + kw) * kTileKeys;
            tile_step<D>(lds + kw * kTileFloats, q, st, P.c, width, lane, [&](int key) { return key0 + key < key_end; });
        }
    }

    // ---- the KW states of a head fold through LDS; one piece: the result, else a partial ----
    static_assert(HPW * KW * kStateBytes<D> <= KW * Lds<D>::kBytes, "merge buffer exceeds the tile region");
    static_assert(QueryRegs<T, D, HPW, kThreads>::kBytes <= KW * Lds<D>::kBytes, "queries exceed the tile region");
    T* orow = static_cast<T*>(P.o) + (int64_t)b * P.o_sb + (int64_t)qrow * P.o_ss + (int64_t)head * P.o_sh;
    const int64_t slot = (((int64_t)b * P.num_q_heads + head) * P.nqt + qt) * P.nsplit + split;
    float* prow = P.part_o + (slot * 32 + r) * D;
    fold_states<D, KW>(lds, st, wave, lane, width, [&](int d, f32x4 acc) {
        if (!row_ok) return;
        if (n_pieces > 1) { *reinterpret_cast<f32x4*>(prow + d) = acc; return; }
        const float inv = st.l > 0.f ? 1.0f / st.l : 0.f;                      // no key at all: zeros
        store4(orow + d, f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv});
    });
    if (row_ok && n_pieces > 1 && kw == 0 && H == 0) {
        P.part_ml[(slot * 2 + 0) * 32 + r] = st.m;
        P.part_ml[(slot * 2 + 1) * 32 + r] = st.l;
    }
}

// Folds the pieces of a sequence: grid (head x query tile x 16, sequence), a thread takes four columns of one of two queries.
// A chain of memory latencies: the loads of the first AHEAD pieces are on their way before the lengths say how many there are
// (slots beyond them exist and are not used), the next AHEAD behind them; and a sequence's partials come in through many
// CUs.  (Eight queries per workgroup and eight pieces at a time, behind the lengths: 1 x 1056 keys 5.2 us of 20.8 for the whole call, which is
// 18.8 now together with the queries through LDS; 1 x 4000 37.3 -> 35.2, 1 x 12 000 58.5 -> 53.8, 2 x 900-2000 33.6 -> 31.1, 8 x 4000-9000
// 198 -> 190.)
constexpr int kFoldRows = 2, kFoldParts = 32 / kFoldRows;
template <typename T, int D, int AHEAD>
__global__ __launch_bounds__(kFoldRows * D / 4) void paged_combine_f32_kernel(const PagedWideParams P)
{
    const int part = blockIdx.x % kFoldParts, hq = blockIdx.x / kFoldParts, b = blockIdx.y;
    const int qt = hq % P.nqt, head = hq / P.nqt;
    const int s = part * kFoldRows + threadIdx.x / (D / 4), d = threadIdx.x % (D / 4) * 4;
    const int qrow = qt * 32 + s;
    const int64_t slot0 = (((int64_t)b * P.num_q_heads + head) * P.nqt + qt) * P.nsplit;
    float m[AHEAD], l[AHEAD];
    f32x4 po[AHEAD];
    auto load = [&](int i0, int n) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int64_t slot = slot0 + min(i0 + i, n - 1);
            m[i] = P.part_ml[(slot * 2 + 0) * 32 + s];
            l[i] = P.part_ml[(slot * 2 + 1) * 32 + s];
            po[i] = *reinterpret_cast<const f32x4*>(P.part_o + (slot * 32 + s) * D + d);
        }
    };
    load(0, P.nsplit);
    const int ctx = keys_of(P, b);
    const int span = keys_per_piece<true>(P, ctx, threadIdx.x & 63);
    const int n = __builtin_amdgcn_readfirstlane((ctx + span - 1) / span);
    if (n <= 1 || qrow >= P.sq || d >= P.head_dim) return;      // one piece: written by the attention kernel
    float M = kMinusBig, L = 0.f;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < n; i0 += AHEAD) {
        if (i0 > 0) load(i0, n);
#pragma unroll
        for (int g = 0; g < AHEAD; g += 8) {
            if (i0 + g >= n) break;
            float Mn = M;
#pragma unroll
            for (int i = g; i < g + 8; ++i) Mn = fmaxf(Mn, i0 + i < n ? m[i] : kMinusBig);
            const float keep = __builtin_amdgcn_exp2f(M - Mn);
            L *= keep;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] *= keep;
            M = Mn;
#pragma unroll
            for (int i = g; i < g + 8; ++i) {
                if (i0 + i >= n) break;                         // (nothing of the others: 0 x infinity is not 0)
                const float w = __builtin_amdgcn_exp2f(m[i] - M);
                L += w * l[i];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += w * po[i][e];
            }
        }
    }
    const float inv = L > 0.f ? 1.0f / L : 0.f;                 // every key on an invalid page: zeros
    store4(static_cast<T*>(P.o) + (int64_t)b * P.o_sb + (int64_t)qrow * P.o_ss + (int64_t)head * P.o_sh + d,
           f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv});
}

int64_t slot_bytes(int head_dim) { return 32 * ((head_dim > 128 ? 256 : 128) + 2) * (int64_t)sizeof(float); }

// Partial slots per sequence: pieces of at least kLeastKeys keys, and no more than fill the chip about four times over (2048
// slots of one head: 34 MB of partials at most, and pieces enough for the ragged end of a launch to be short).
int splits_wanted(int64_t bs, int nqt, int num_q_heads, int64_t max_keys) {
    int64_t n = 2048 / (bs * num_q_heads * nqt);
    if (n > (max_keys + kLeastKeys - 1) / kLeastKeys) n = (max_keys + kLeastKeys - 1) / kLeastKeys;
    if (n > kMaxSplits) n = kMaxSplits;
    return n < 1 ? 1 : (int)n;
}

template <typename T, int D, int HPW, int KW, bool ONE_ROUND = false>
int launch_groups(const PagedWideParams& P, hipStream_t stream)
{
    constexpr int kLdsBytes = KW * Lds<D>::kBytes;
    // the kernel's LDS limit is raised once per device
    static std::atomic<bool> raised[64];
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "paged_block_attn: no current device (%s)", hipGetErrorString(e));
    if (!raised[device].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(paged_attn_f32_kernel<T, D, HPW, KW, ONE_ROUND>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
        MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "paged_block_attn: cannot reserve %d bytes of LDS (%s)", kLdsBytes, hipGetErrorString(e));
        raised[device].store(true, std::memory_order_release);
    }
    const dim3 grid((unsigned)(P.num_q_heads / HPW * P.nqt), (unsigned)P.nsplit, (unsigned)P.bs);
    paged_attn_f32_kernel<T, D, HPW, KW, ONE_ROUND><<<grid, 64 * HPW * KW, kLdsBytes, stream>>>(P);
    const int rc = mdx::check_launch("paged_block_attn (fp32 arithmetic)");
    if (rc != MDX_OK || P.nsplit == 1) return rc;
    const dim3 fold((unsigned)(P.num_q_heads * P.nqt * kFoldParts), (unsigned)P.bs);
    constexpr int kFoldThreads = kFoldRows * D / 4;
    if (P.nsplit <= 8)       paged_combine_f32_kernel<T, D, 8><<<fold, kFoldThreads, 0, stream>>>(P);
    else if (P.nsplit <= 16) paged_combine_f32_kernel<T, D, 16><<<fold, kFoldThreads, 0, stream>>>(P);
    else                     paged_combine_f32_kernel<T, D, 24><<<fold, kFoldThreads, 0, stream>>>(P);     // (sixteen at a time: 1 x 4000 keys 36.8, 24: 35.2)
    return mdx::check_launch("paged_combine (fp32 arithmetic)");
}

// KW: tiles of 32 keys staged side by side, two workgroups' worth of LDS per CU.  Whole contexts for no more heads than there are
// CUs (a caller without a workspace) are chains of tiles with CUs to spare: a workgroup per head, one per CU with all of its LDS, and
// twice the wavefronts on the chain with the loads of four tiles in flight (us, two heads / one head per workgroup: d = 128, 4 x 2000
// keys 199 / 132, 16 x 2000 220 / 156, 1 x 1056 100 / 69; d = 256, 4 x 2000 746 / 455, 16 x 1000 408 / 252).  More heads than CUs are
// more than one round of such workgroups (24 x 2000, d = 128: 315, with two heads each 238).
template <typename T>
int launch(const PagedWideParams& P, hipStream_t stream)
{
    if (P.nsplit == 1 && (int64_t)P.bs * P.num_q_heads * P.nqt <= mdx::compute_units())
        return P.head_dim <= 128 ? launch_groups<T, 128, 1, 4>(P, stream) : launch_groups<T, 256, 1, 2>(P, stream);
    const bool pairs = P.heads_per_kv % 2 == 0;
    // pieces of the least size, whatever the lengths: no more keys in the tables than the pieces and the slots hold of it.  (Us: 1 x 1024 keys 20.0 / 19.4, 3 x 100-400
    // 19.0 / 18.4; a head per workgroup loads its tiles in two batches.)
    const int64_t max_keys = (int64_t)P.max_pages * P.page_size;
    const bool one_round = P.bs <= 64 && P.bs * max_keys <= (int64_t)kLeastKeys * P.pieces && max_keys <= (int64_t)kLeastKeys * P.nsplit;
    if (P.head_dim <= 128 && pairs && one_round && P.nsplit > 1) return launch_groups<T, 128, 2, 2, true>(P, stream);
    if (P.head_dim <= 128) return pairs ? launch_groups<T, 128, 2, 2>(P, stream) : launch_groups<T, 128, 1, 2>(P, stream);
    return pairs ? launch_groups<T, 256, 2, 1>(P, stream) : launch_groups<T, 256, 1, 1>(P, stream);
}

}  // namespace

extern "C" int64_t mdx_paged_block_attn_f32_workspace_bytes(int32_t bs, int32_t sq, int32_t num_q_heads, int32_t head_dim,
                                                            int32_t max_pages, int32_t page_size)
{
    if (bs <= 0 || sq <= 0 || num_q_heads <= 0 || head_dim <= 0 || max_pages <= 0 || page_size <= 0) return 0;
    const int nqt = (sq + 31) / 32;
    const int n = splits_wanted(bs, nqt, num_q_heads, (int64_t)max_pages * page_size);
    return n <= 1 ? 0 : (int64_t)bs * num_q_heads * nqt * n * slot_bytes(head_dim);
}

namespace mdx {

// Called by the launch behind every paged entry point, which has checked sizes, head counts, the page size
// (a multiple of 32), the scale and the pointers, for dtype MDX_F32 and for head widths outside the 16-bit kernel's.
int launch_paged_f32(const void* q, void* o, const void* k_cache, const void* v_cache,
                     int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                     int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                     int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                     const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                     int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                     int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                     float scale, int32_t dtype, void* workspace, int64_t workspace_bytes, hipStream_t stream)
{
    MDX_REQUIRE(head_dim >= 4 && head_dim <= 256 && head_dim % 4 == 0, MDX_EUNSUPPORTED,
                "paged_block_attn: head_dim %d (fp32 arithmetic: multiples of 4 up to 256)", head_dim);
    const uintptr_t align = dtype == MDX_F32 ? 15u : 7u;       // four elements per access
    MDX_REQUIRE((((uintptr_t)q | (uintptr_t)o | (uintptr_t)k_cache | (uintptr_t)v_cache) & align) == 0 &&
                q_stride_b % 4 == 0 && q_stride_s % 4 == 0 && q_stride_h % 4 == 0 &&
                o_stride_b % 4 == 0 && o_stride_s % 4 == 0 && o_stride_h % 4 == 0 &&
                cache_stride_page % 4 == 0 && cache_stride_tok % 4 == 0 && cache_stride_head % 4 == 0,
                MDX_EUNSUPPORTED, "paged_block_attn: tensors must be aligned to four elements with strides that are multiples of 4 elements");
    MDX_REQUIRE(bs <= 65535 && num_q_heads <= 65535, MDX_EUNSUPPORTED, "paged_block_attn: fp32 arithmetic takes up to 65535 sequences");
    PagedWideParams P;
    P.q = q; P.o = o; P.k_cache = k_cache; P.v_cache = v_cache;
    P.q_sb = q_stride_b; P.q_ss = q_stride_s; P.q_sh = q_stride_h;
    P.o_sb = o_stride_b; P.o_ss = o_stride_s; P.o_sh = o_stride_h;
    P.c_sp = cache_stride_page; P.c_st = cache_stride_tok; P.c_sh = cache_stride_head;
    P.block_table = block_table; P.bt_stride = bt_stride; P.context_lens = context_lens;
    P.bs = bs; P.sq = sq; P.nqt = (sq + 31) / 32;
    P.num_q_heads = num_q_heads; P.heads_per_kv = num_q_heads / num_kv_heads;
    P.page_size = page_size; P.max_pages = max_pages; P.head_dim = head_dim;
    P.page_shift = -1;
    for (int i = 0; i < 31; ++i) if (page_size == (1 << i)) P.page_shift = i;
    P.num_pages = num_pages;
    P.c = scale * kLog2e;
    // as many partial slots as the launch wants and the caller's workspace holds; none: whole contexts
    const int64_t n_rows = (int64_t)bs * num_q_heads * P.nqt, room = workspace && mdx::aligned16(workspace) ? workspace_bytes / (n_rows * slot_bytes(head_dim)) : 0;
    P.nsplit = splits_wanted(bs, P.nqt, num_q_heads, (int64_t)max_pages * page_size);
    if (P.nsplit > room) P.nsplit = room > 1 ? (int)room : 1;
    const int groups = num_q_heads / (P.heads_per_kv % 2 == 0 ? 2 : 1) * P.nqt;
    P.pieces = 1024 / groups > 0 ? 1024 / groups : 1;          // two pieces for each of the two workgroups that a CU holds
    P.part_o = static_cast<float*>(workspace);
    P.part_ml = P.nsplit > 1 ? P.part_o + n_rows * P.nsplit * 32 * (head_dim > 128 ? 256 : 128) : nullptr;
    switch (dtype) {
    case MDX_F32:  return launch<float>(P, stream);
    case MDX_F16:  return launch<_Float16>(P, stream);
    case MDX_BF16: return launch<__bf16>(P, stream);
    }
    return mdx::fail(MDX_EUNSUPPORTED, "paged_block_attn: dtype %d", dtype);
}

}  // namespace mdx
