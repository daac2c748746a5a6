// Paged single-block ("decode") attention: the Sq <= 128 queries of the current
// denoising block of every sequence attend, non-causally, to the first
// context_lens[b] keys of that sequence's paged KV cache.  A workgroup serves one
// tile of 32 queries; blocks of 64 or 128 positions (the reference's block length
// is a configuration field, nanovllm/config.py:48) run as 2 or 4 query tiles,
// each a workgroup with its own partials and arrival counter; they stream the
// same keys and are launched next to each other, 8 workgroups apart, so that
// they run on one XCD and the later ones find in its L2 what the first fetched.
//
// Replaces flash_attn_with_kvcache(..., causal=False) at
// engines/nano_dvlm/nanovllm/layers/sdar_attention.py:48-56.
//
// The op is HBM-bound (each K/V byte is used by only Sq * Hq/Hkv = 64 query
// rows), so the design goal is to keep the whole chip streaming pages:
//  * split-KV: a workgroup owns one split of consecutive keys of one sequence
//    for one group of query heads; the split size is chosen so that there are
//    one to two workgroups per CU at most (pick_chunk and the rule in the kernel), and with about a (sequence, KV head)
//    pair per CU sequences stay whole unless the longest is well above what
//    a resident workgroup's even share of all keys comes to (kWholeFactor).  Workgroups are numbered densely over the
//    (sequence, split) pairs that exist (lane b of each wavefront holds the
//    split count of sequence b), so the launch order has no holes: the
//    dispatcher deals consecutive workgroups round-robin to XCDs and shader
//    engines and stalls on a full one, which punishes interleaved no-op groups.
//  * a workgroup has 4 wavefronts, each owning 32 queries of ONE query head:
//    HPW heads that share a KV head (2 for grouped-query attention) times
//    KW = 4/HPW key slices of 32 keys.  Two workgroups share a CU.
//  * K/V tiles of 32*KW keys travel global -> registers -> LDS with 16-byte
//    coalesced loads into two register sets while a third tile is consumed from
//    the double-buffered LDS.  (As compiled, a stage waits for every load the
//    wavefront has outstanding, because the fetch of the younger tile sits under
//    a condition; making all fetches unconditional, so that the wait leaves the
//    younger tile in flight, was measured and changes nothing: the depth of the
//    load queue is not what bounds this kernel.)
//  * the KW wavefront states of a head are merged through LDS, then either
//    written as the final output (single split) or as an fp32 partial
//    (m, l, O) that the last split of the pair to arrive merges (single launch)
//    or a second, small kernel combines.
#include "mdx_common.h"
#include "attn_tile.h"
#include <type_traits>

namespace {

using namespace mdx_attn;

constexpr int kQTile = 32;          // queries per workgroup (one per lane pair of a wavefront)
constexpr int kMaxSq = 128;         // queries per sequence: up to four query tiles
constexpr int kChunkAlign = 256;   // the host's split sizes are multiples of this many keys

// Few sequences: the kernel's choice of pieces (PagedParams::fit_slots says why), and with the same figures the host's guess of it.
constexpr float kPieceRoot = 4.f;                       // keys of a piece: this times the root of the launch's keys, from kLeastPiece on
constexpr int kLeastPiece = 64;
// Sequences are only cut if that takes more off the longest workgroup than the partials of them all cost (8 x 300 and 16 x 600
// keys stay whole).
template <typename T> __host__ __device__ __forceinline__ bool stay_whole(T longest, T piece, int sequences) { return longest - piece < T(64 + 12 * sequences); }

// About a (sequence, head group) pair per CU and more: sequences are left whole -- no partials, nothing to merge -- unless the longest is kWholeFactor
// times what a resident workgroup's even share of the keys comes to (or 1.2 times the mean, where that is more); then all are cut into pieces
// of kShareFactor shares and kShareKeys keys.  The layer, us, cut at 1.25 times the mean only / by shares: 24 sequences of 1250-5000 keys 86 / 71, 550-2200
// 49 / 42, 32 of 375-1500 45 / 38, 825-3300 71 / 64, 33 of 1000-4000 100 / 78, 40 of 500-3500 93 / 76, 48 of 550-2200 85 / 68, 64 of 300-2300 89 / 78;
// equal lengths stay whole, level.  (Shares of 1.05 without the keys: 33 of 1000-4000 75, but 24 of 375-1500 38 instead of 33, 32 of those 43
// instead of 38: a second workgroup on a CU that holds one at a time costs its start and end.)
constexpr float kWholeFactor = 1.33f, kShareFactor = 1.2f;
constexpr int kShareKeys = 192;

using mdx::wave_sum;
using mdx::wave_max;

// Partials that another workgroup of the same launch reads (single-launch merge) travel with
// agent-scope accesses: such a store is written through to memory and such a load does not take a line
// that this XCD's L2 may still hold from an earlier launch.  That makes them visible across the XCDs'
// L2 caches without the release fence (a write-back walk of the whole L2) that ordinary stores would need.
typedef __attribute__((ext_vector_type(4))) float f32x4;
__device__ __forceinline__ void store_agent(float* p, f32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1" :: "v"(p), "v"(v) : "memory");
}
// (Not inline asm: the compiler takes such a load's registers for written while it is still on its way, and what it moved or spilled before the wait would be
// the old contents.  Two atomic loads of eight bytes: 16 sequences of 375-1500 keys 24.9 -> 25.5 us.)
constexpr int kAgentScope = 16;                      // sc1
constexpr int kRawBuffer = 0x27000;                  // last word of the descriptor: elements of 32 bits, not swizzled, out of range reads 0
__device__ __forceinline__ f32x4 load_agent(__amdgpu_buffer_rsrc_t from, int offset) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, offset, 0, kAgentScope));
}
__device__ __forceinline__ void wait_vector_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct PagedParams {
    const __bf16* q; __bf16* o; const __bf16* k_cache; const __bf16* v_cache;
    int64_t q_sb, q_ss, q_sh, o_sb, o_ss, o_sh;     // element strides
    int64_t c_sp, c_st, c_sh;                       // cache strides: page, token, head
    const int32_t* block_table; int64_t bt_stride;
    const int32_t* context_lens;
    int bs, sq, heads_per_kv, page_size, page_shift, max_pages;   // page_shift: log2(page_size) or -1
    int64_t num_pages;
    int chunk, nsplit;                              // keys per split, max splits per sequence
    int nqt;                                        // query tiles of 32 per sequence (grid z)
    int num_q_heads;
    mdx::Divisor by_bs;
    int head_dim;                                   // <= 128, a multiple of 16: columns beyond it are zeros in LDS and never stored
    float c;                                        // scale * log2(e)
    float* part_o; float* part_ml;                  // [bs, Hq, nqt, nsplit, (d tile, register quad), lane, 4] and [bs, Hq, nqt, nsplit, 32, (m, l)]
    // non-null: the attention kernel picks the split size (>= chunk) from the lengths and leaves it
    // here for the combine kernel.  A float on purpose: an int store in the attention kernel could
    // alias the int page table and lengths for the compiler, which would then stop fetching those
    // through the scalar cache and wait on the vector-memory counter for them, draining the K/V
    // prefetch queue (measured: 78 -> 120 us).  Split sizes are far below 2^24, so the value is exact.
    float* span_out;
    // > 0: fewer (sequence, head group) pairs than the chip holds workgroups.  The attention kernel, which sees the
    // lengths, picks the size of a piece, grows it by a tile at a time until the launch fits this
    // many resident workgroups -- one round, nobody starts late -- and leaves the size it settled on in span_out.  (Full tables: 16 sequences of 4128 keys 69 -> 60 us, 16 of
    // 1000 to 3000 keys in a table 12 pages wide 51 -> 42 us; no shape of the sweep slower.  Cutting each sequence
    // into equal pieces instead of full splits and a short remainder was measured too and loses: the remainders
    // start last and fill the tail.)
    // < 0: about a pair per CU or more, minus the workgroups that are resident (kWholeFactor).  (One field for both: with four bytes more of arguments
    // the launch with readers takes 0.2 us longer.)
    int fit_slots;
    // Single-launch mode: one arrival counter per (sequence, head group), zero between launches.  The
    // last split of a pair to arrive merges the pair's partials itself.  float for the same reason.
    float* arrive;
};

// Weights that the launches behind this one read.  An attention launch of a few sequences leaves most of the chip idle and HBM nearly
// so for 8 to 15 us, while the products behind it get W from HBM at half of its rate: a CU's loads come back in order, and
// rows of x from L2 wait behind rows of W.  Read once before, W is in the memory-side cache (256 MB), from where the gate/up projection of 128 rows takes
// 12.6 us instead of 19.6, of 32 rows 9.6 instead of 14.
struct ReadAhead {
    const u32x4* p[2]; int n[2];                    // 16-byte elements
    int first_y;                                    // blockIdx.y from which workgroups read
};
__device__ __forceinline__ bool is_reader(int block_y, const ReadAhead& A) { return block_y >= A.first_y; }
template <int THREADS> __device__ __forceinline__ void read_ahead(const ReadAhead& A) {
    constexpr int kTogether = 8;
    const int step = ((int)gridDim.y - A.first_y) * (int)gridDim.x * THREADS;
    u32x4 all = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int i = (((int)blockIdx.y - A.first_y) * (int)gridDim.x + (int)blockIdx.x) * THREADS + (int)threadIdx.x;
        for (; i + (kTogether - 1) * step < A.n[k]; i += kTogether * step) {
            u32x4 x[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) x[u] = A.p[k][i + u * step];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) all ^= x[u];
        }
        for (; i < A.n[k]; i += step) all ^= A.p[k][i];
    }
    asm volatile("" :: "v"(all));                   // (the loads have a use)
}

// The combine kernel's running fold of split partials over four columns of one query.  The merge at the end of paged_block_attn_kernel does the same
// operations in the same order on other columns per lane, and has to: a pair's result has the same bits either way.
struct Fold {
    float M, L, acc[4];
    __device__ __forceinline__ void init() {
        M = kMinusBig; L = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = 0.f;
    }
    // Four slots, of which the first `on` exist (the others hold leftovers).
    __device__ __forceinline__ void take4(const float (&m_in)[4], const float (&l)[4], const f32x4 (&po)[4], int on) {
        float m[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = i < on ? m_in[i] : kMinusBig;
        const float Mn = fmaxf(fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])), M);
        const float keep = __builtin_amdgcn_exp2f(M - Mn);
        L *= keep;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] *= keep;
        M = Mn;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float w = i < on ? __builtin_amdgcn_exp2f(m[i] - M) : 0.f;
            L = i < on ? __builtin_fmaf(w, l[i], L) : L;                   // (explicit: a contraction that the compiler picked could differ from the merge's)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = i < on ? __builtin_fmaf(w, po[i][e], acc[e]) : acc[e];
        }
    }
    __device__ __forceinline__ float inverse() const { return L > 0.f ? 1.0f / L : 0.f; }   // no valid key at all (every page id invalid): zeros, like a context of 0
};

// WAVES = 4 (two workgroups per CU) or 8 (one workgroup per CU, 128-key tiles: for launches with about
// one workgroup per CU, where a CU would otherwise hold four wavefronts only).  Tiles hold 32 keys per
// key slice (WAVES / HPW slices); two 64-key tile buffers fit a CU twice, two 128-key ones once.
// MERGE: single launch, the last split of a pair merges them (a kernel of its own: one sequence's launch is 0.3 us longer with that code in it).
// AHEAD: none, or ReadAhead: workgroups behind those of the attention read what the launches behind it need.
template <typename E, int HPW, int DEPTH, int WAVES, bool MERGE, typename... AHEAD>
__global__ __launch_bounds__(64 * WAVES, (WAVES / HPW == 2) ? 2 : 1) void paged_block_attn_kernel(const PagedParams P, const AHEAD... ahead)
{
    const int zero = mdx::fetch_arguments<sizeof(PagedParams)>(gridDim.x);
    const unsigned block_x = blockIdx.x + zero;
    if constexpr (sizeof...(AHEAD) > 0) {
        if (is_reader((int)blockIdx.y + zero, ahead...)) { read_ahead<64 * WAVES>(ahead...); return; }
    }
    constexpr int kThreads = 64 * WAVES;
    constexpr int kRowsPerPass = kThreads / 16;     // LDS rows one pass of the workgroup stages
    constexpr int kPassesPerSlice = 32 / kRowsPerPass;
    constexpr int KW = WAVES / HPW;                 // key slices (wavefronts per head)
    constexpr int kTileKeys = 32 * KW;
    constexpr int kTileBytes = kTileKeys * kLdsPitch;
    constexpr int kPasses = TileRegs<kTileKeys, kThreads>::kPasses;   // 16 rows per pass
    // [buffer][K tile, V tile]; the region is reused for the cross-wavefront merge at the end.
    __shared__ __attribute__((aligned(16))) char lds[2][2 * kTileBytes];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int H = lane >> 5, r = lane & 31;
    // launch order: head group fastest, then the query tiles of a (sequence, split), then the pairs -- the tiles of a
    // block longer than 32 queries stream the same keys, so they start next to each other and on the same XCD
    const int n_groups = P.num_q_heads / HPW;
    const int qt = mdx::quotient(block_x, n_groups);           // this workgroup's tile of 32 queries
    const int hg = block_x - qt * n_groups;
    const int kw = wave % KW;                       // this wavefront's key slice
    const int head = hg * HPW + wave / KW;          // and query head

    // ---- workgroup -> (sequence b, split) ------------------------------------------------------
    int b, split, span = P.chunk;
    bool paced = false;
    typedef __attribute__((address_space(4))) const int32_t ConstantEntry;
    int ctx_all = 0;                                // (up to 64 sequences) the clipped length of sequence `lane`
    if (P.bs <= 64) {
        // lengths beyond the page table name keys that do not exist: clipped here and below
        const int ctx_l = lane < P.bs ? min(max(0, P.context_lens[lane]), P.max_pages * P.page_size) : 0;
        ctx_all = ctx_l;
        bool cut = true;                            // false: every sequence is known to be one piece
        auto splits_of_lane = [&]() { return lane < P.bs ? max(1, (ctx_l + span - 1) / span) : 0; };   // (padding rows get one)
        int n = 0;
        if (P.fit_slots > 0) {
            // One size of piece for all sequences.  A launch of few keys is a chain of latencies as long as its longest
            // workgroup, one of many keys a stream that more and shorter workgroups only disturb: over batches of 1 to 20
            // sequences and contexts of 300 to 16 000 keys the best size follows 4 sqrt(total keys) up to 512 (300 keys: 64,
            // 1100: 128, 4 x 1100: 192 to 256, 8 x 1100: 384, 16 x 1100, 4 x 8000: 512).  At least what fills the chip once, total / (resident
            // workgroups per head group - a remainder of half a piece per sequence), and no more pieces of a sequence than
            // the launch has room for (the "+ 1" keeps the longest within nsplit pieces whatever the rounding of the
            // reciprocals; every workgroup makes the same estimate).
            const int total = wave_sum(ctx_l), longest = wave_max(ctx_l), live = __popcll(__ballot(ctx_l > 0));
            const float per_group = (float)P.fit_slots * __builtin_amdgcn_rcpf((float)gridDim.x);      // resident workgroups per head group and query tile
            const float room = fmaxf(1.f, per_group - 0.5f * (float)live);
            const int best = min(512, ((int)(kPieceRoot * __builtin_amdgcn_sqrtf((float)total)) + 32) & ~63);
            const float least = fmaxf((float)total * __builtin_amdgcn_rcpf(room), (float)longest * __builtin_amdgcn_rcpf((float)P.nsplit) + 1.f);
            span = max(max(kLeastPiece, best), ((int)least + 63) & ~63);
            if (stay_whole(longest, span, live)) span = max(span, longest);
            n = splits_of_lane();
            // a tile more per step (24 steps double the smallest split); a few workgroups beyond what is resident
            // may stay: the last to start are remainders, which fill the tail
            for (int it = 0; it < 24 && wave_sum(n) * (int)gridDim.x > P.fit_slots + P.fit_slots / 32; ++it) {
                span += 64;
                n = splits_of_lane();
            }
            // more than three quarters of the resident workgroups have a whole piece (fetch_by says why; launches that merge themselves have no more than 2560 keys a
            // sequence and were level)
            paced = !MERGE && 4.f * (float)total * (float)gridDim.x > 3.f * (float)P.fit_slots * (float)span;
            if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *P.span_out = (float)span;
        } else {
            if (P.fit_slots < 0) {
                // (kWholeFactor above says why; the host's split is what keeps the longest within nsplit pieces)
                const int total = wave_sum(ctx_l), longest = wave_max(ctx_l), live = __popcll(__ballot(ctx_l > 0));
                const float share = (float)total * (float)gridDim.x * __builtin_amdgcn_rcpf((float)-P.fit_slots);
                const float mean = (float)total * __builtin_amdgcn_rcpf((float)max(live, 1));
                span = max(span, ((int)(kShareFactor * share) + kShareKeys + 63) & ~63);
                if ((float)longest <= kWholeFactor * fmaxf(share, 0.9f * mean)) span = max(span, longest);
                cut = longest > span;
                if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *P.span_out = (float)span;
            }
            if (!MERGE) n = splits_of_lane();
        }
        // the j-th (sequence, split) pair in launch order; `has`: the lanes (sequences) that own a pair of the kind that is next in it
        int j = blockIdx.y, level = 0;
        b = -1;
        auto among = [&](unsigned long long has) {
            const int c = __popcll(has);
            if (j < c) {
                const int before = __popcll(has & ((1ull << lane) - 1ull));
                const unsigned long long hit = __ballot(((has >> lane) & 1ull) != 0 && before == j);
                b = __ffsll((long long)hit) - 1;
                return true;
            }
            j -= c;
            return false;
        };
        if (MERGE && !cut && P.bs * (int)gridDim.x <= -P.fit_slots) {
            // Whole sequences that are all resident at once: any order will do, and the search for a pair is part of every workgroup's start.  (32 equal
            // sequences of 1088-3136 keys, average under the profiler: 52.6 us with the search below, 51.6 without; a decode pass of them is 0.9 % shorter.)
            if (j >= P.bs) return;
            b = j;
            level = 0;
        } else if constexpr (MERGE) {
            // Heaviest first: all whole pieces, then the remainders (and sequences shorter than a piece) by eighths of a piece, so that
            // those which start late, when there are more workgroups than the chip holds at once, are the short ones of all.  (16 sequences of
            // 375-1500 keys 30.3 us in the order below, 26.2 in this one.)
            const int whole = cut ? ctx_l / span : ctx_l == span && ctx_l > 0, rest = ctx_l - whole * span;
            if (j >= (cut ? wave_sum(lane < P.bs ? whole + (rest > 0 || whole == 0) : 0) : P.bs)) return;
            bool found = false;
            for (; !found && level < P.nsplit; ++level) found = among(__ballot(whole > level));
            if (found) {
                --level;
            } else {
                const int eighth = lane < P.bs && (rest > 0 || whole == 0) ? min(7, (int)((float)rest * 8.f * __builtin_amdgcn_rcpf((float)span))) : -1;
                for (int e = 7; !found && e >= 0; --e) found = among(__ballot(eighth == e));
                if (found) level = __builtin_amdgcn_readlane(whole, b);
            }
        } else {
            // the first split of every sequence, then the second of those that have one, ...: the last split of a sequence is its remainder
            // (from the level that the pair would have if all of them had that many: those below it hold a sum)
            if (j >= P.bs) {
                level = mdx::quotient(j, P.by_bs);
                j -= wave_sum(min(n, level));
            }
            for (; level < P.nsplit; ++level) if (among(__ballot(n > level))) break;
        }
        if (b < 0) return;                          // past the last (sequence, split) pair
        split = level;
    } else {
        b = blockIdx.y / P.nsplit;
        split = blockIdx.y % P.nsplit;
    }
    const int ctx = P.bs <= 64 ? __builtin_amdgcn_readlane(ctx_all, b)       // lane b read it above: no second trip to memory
                               : min(P.context_lens[b], P.max_pages * P.page_size);
    const int n_valid_splits = (ctx + span - 1) / span;
    if (ctx <= 0) {
        // graph-padding row: defined output (zeros), written by its split 0
        if (split == 0 && qt == 0) {
            for (int e = tid; e < P.sq * HPW * (kHeadDim / 8); e += kThreads) {
                const int d8 = e % (kHeadDim / 8), h = (e / (kHeadDim / 8)) % HPW, s = e / (kHeadDim / 8) / HPW;
                if (d8 * 8 < P.head_dim) *reinterpret_cast<u32x4*>(P.o + (int64_t)b * P.o_sb + (int64_t)s * P.o_ss + (int64_t)(hg * HPW + h) * P.o_sh + d8 * 8) = u32x4{0, 0, 0, 0};
            }
        }
        return;
    }
    // (uniform in the compiler's eyes too, or the page table comes through vector loads)
    const int key_begin = __builtin_amdgcn_readfirstlane(split * span);
    if (key_begin >= ctx) return;
    const int key_end = __builtin_amdgcn_readfirstlane(min(ctx, key_begin + span));
    const int kvh = mdx::quotient(hg * HPW, P.heads_per_kv);

    // (by itself the compiler takes the table for constant only in some forms of this kernel)
    auto table_row = [&] {
        const int32_t* row = P.block_table + (int64_t)__builtin_amdgcn_readfirstlane(b) * P.bt_stride;
        return (ConstantEntry*)(uintptr_t)row;
    };
    const auto bt = table_row();
    const int chunk = tid & 15, trow = tid >> 4;    // one pass stages kRowsPerPass rows
    const int n_tiles = (key_end - key_begin + kTileKeys - 1) / kTileKeys;
    // The loads of a fetch are unconditional (rows past the context or on an invalid page id read row `trow` of page 0 instead and are zeroed when they reach LDS).
    // Each pass of kRowsPerPass keys, which never straddles a page (page_size % 32 == 0), looks its page up: in the first tiles, whose lookups, through the constant address
    // space, are all on their way at once.  (Through an ordinary pointer each was waited for before its pass's loads: 4800 cycles of a workgroup's start, and the first tile had
    // landed before the second was asked for.  From a register that holds the piece's first 64 pages, as behind the first tiles, the start is slower: one sequence of 1337
    // keys 14.1 us, so 13.3, 17 of 120 13.4 / 12.4.)  Behind them, where a tile lies in one page (paged_tiles), its page comes from that register: a scalar load that is
    // waited for among the reads from LDS holds them all up.  K's rows of a tile are asked for before V's, which HBM prefers (32 of 600-2400 56.5 / 56.1).  The layer, us, before both / now: one
    // sequence of 300 keys 11.9 / 11.0, 1337 14.6 / 13.3, 12 000 27.4 / 24.6, four of 1000-3000 23.0 / 21.3, 12 of 500-2500 34.8 / 32.4.  Not where the launch fills most of the resident
    // workgroups (`paced`): HBM is the bound there, workgroups that ask for their tiles as soon as they can crowd out each other, and a lookup per pass spreads the loads
    // (16 of 512-4096: 42.9 before, 44.4 without the rule, 41.8 with it); nor beside readers: that launch lasts as long as those do (generating with one request 61.7 ms, 62.1 with it,
    // eight 57.5 / 58.5); nor with eight wavefronts (32 of 600-2400 56.4 / 56.0).
    struct Staged {
        TileRegs<kTileKeys, kThreads> regs;
        unsigned row_ok;       // bit p: this thread's row of pass p holds a real key
        unsigned pass_ok;      // bit p (uniform): pass p lies on a valid page inside the context
    };
    // (a thread whose 16-byte chunk lies beyond a narrow head reads the head's last chunk instead; zeroed like a row past the end)
    const bool col_ok = chunk * 8 < P.head_dim;
    const int64_t safe_off = (int64_t)trow * P.c_st + (int64_t)kvh * P.c_sh + min(chunk * 8, P.head_dim - 8);
    const bool tile_in_page = sizeof...(AHEAD) == 0 && WAVES == 4 && P.page_shift >= 0 && P.page_size >= kTileKeys && (key_begin & (kTileKeys - 1)) == 0;
    const bool paged_tiles = tile_in_page && !paced;
    auto slot_of = [&](int key) { return P.page_shift >= 0 ? key >> P.page_shift : key / P.page_size; };
    const int first_slot = slot_of(key_begin), pages = bt[min(first_slot + lane, P.max_pages - 1)];
    auto load_k = [&](Staged& sg, int p, int64_t off) { sg.regs.k[p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(P.k_cache + off)); };
    auto load_v = [&](Staged& sg, int p, int64_t off, bool ok, int key0) {
        sg.regs.v[p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(P.v_cache + off));
        sg.pass_ok |= (ok ? 1u : 0u) << p;
        sg.row_ok |= ((ok && col_ok && key0 + kRowsPerPass * p + trow < key_end) ? 1u : 0u) << p;
    };
    auto fetch_by = [&](auto first, Staged& sg, int t) {
        const int key0 = key_begin + t * kTileKeys;
        sg.row_ok = 0;
        sg.pass_ok = 0;
        if (!first && paged_tiles) {
            const int ahead = slot_of(key0) - first_slot, page = ahead < 64 ? __builtin_amdgcn_readlane(pages, ahead) : bt[first_slot + ahead];
            const bool valid = page >= 0 && page < P.num_pages;
            const int64_t base = valid ? page * P.c_sp + (int64_t)(key0 & (P.page_size - 1)) * P.c_st : 0;
            auto ok = [&](int p) { return valid && key0 + kRowsPerPass * p < key_end; };
            auto offset = [&](int p) { return (ok(p) ? base + (int64_t)(kRowsPerPass * p) * P.c_st : 0) + safe_off; };
#pragma unroll
            for (int p = 0; p < kPasses; ++p) load_k(sg, p, offset(p));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < kPasses; ++p) load_v(sg, p, offset(p), ok(p), key0);
        } else {
#pragma unroll
            for (int p = 0; p < kPasses; ++p) {
                const int kp = key0 + kRowsPerPass * p, page_slot = slot_of(kp);
                const bool inside = kp < key_end && page_slot < P.max_pages;
                const int64_t page = bt[inside ? page_slot : 0];
                const bool ok = inside && page >= 0 && page < P.num_pages;             // uniform
                const int64_t off = ok ? page * P.c_sp + (int64_t)(kp - page_slot * P.page_size) * P.c_st + safe_off : safe_off;
                load_k(sg, p, off);
                load_v(sg, p, off, ok, key0);
            }
        }
    };
    typename Elem16<E>::vec8 q[1][8];
    WaveState<1> st;
    auto fetch = [&](Staged& sg, int t) { fetch_by(std::false_type(), sg, t); };
    unsigned tile_pass_ok[2] = {0, 0};                 // pass_ok of the tile sitting in LDS buffer 0 / 1
    auto stage = [&](int buf, Staged& sg) {
#pragma unroll
        for (int p = 0; p < kPasses; ++p)
            if (!((sg.row_ok >> p) & 1u)) { sg.regs.k[p] = u32x4{0, 0, 0, 0}; sg.regs.v[p] = u32x4{0, 0, 0, 0}; }
        store_tile<kTileKeys, kThreads>(lds[buf], lds[buf] + kTileBytes, sg.regs, tid);
        tile_pass_ok[buf] = sg.pass_ok;
    };
    auto compute = [&](int t) {
        const char* lk = lds[t & 1];
        const int key0 = key_begin + t * kTileKeys + kw * 32;        // this wavefront's 32 keys = passes 2kw, 2kw+1
        // keys of an invalid page are excluded (not merely zeroed): the owning wavefront skips them
        if ((tile_pass_ok[t & 1] >> (kPassesPerSlice * kw)) & 1u) {
            if (key0 + 32 <= key_end)
                attn_step<E, 1, 1, false>(lk, lk + kTileBytes, kw * 32, q, st, P.c, lane, key0, 0, key_end);
            else
                attn_step<E, 1, 1, true>(lk, lk + kTileBytes, kw * 32, q, st, P.c, lane, key0, 0, key_end);
        }
    };

    // Register sets ra / rb hold the tiles after the one in LDS; tile t+1 sits in set (t+1)%2.
    Staged ra, rb;
    const int qrow = qt * kQTile + r;               // this lane's query of the sequence's block
    const bool row_ok = qrow < P.sq;
    load_q(q[0], row_ok ? P.q + (int64_t)b * P.q_sb + (int64_t)qrow * P.q_ss + (int64_t)head * P.q_sh : nullptr, H, P.head_dim);

    st.init();
    fetch_by(std::true_type(), ra, 0);
    if (DEPTH == 2 && n_tiles > 1) fetch_by(std::true_type(), rb, 1);
    stage(0, ra);
    if (DEPTH == 2) { if (n_tiles > 2) fetch(ra, 2); } else { if (n_tiles > 1) fetch(ra, 1); }
    __syncthreads();
    for (int t = 0; t < n_tiles; t += 2) {
        // even tile t from buffer 0; stage tile t+1 into buffer 1
        compute(t);
        if (t + 1 < n_tiles) {
            if (DEPTH == 2) {
                stage(1, rb);
                if (t + 3 < n_tiles) fetch(rb, t + 3);
            } else {
                stage(1, ra);
                if (t + 2 < n_tiles) fetch(ra, t + 2);
            }
        }
        __syncthreads();
        if (t + 1 >= n_tiles) break;
        // odd tile t+1 from buffer 1; stage tile t+2 into buffer 0
        compute(t + 1);
        if (t + 2 < n_tiles) {
            stage(0, ra);
            if (DEPTH == 2) { if (t + 4 < n_tiles) fetch(ra, t + 4); } else { if (t + 3 < n_tiles) fetch(ra, t + 3); }
        }
        __syncthreads();
    }

    // ---- merge the KW key-slice states of each head through LDS ---------------------------------
    // Slice kw folds, and stores, the d tiles kw, kw + KW, ... of its head: it leaves the other d tiles of its state in LDS as 16-byte lanes (of four slices: all of them),
    // and behind one barrier takes its own from the others'.  (A tree of pairwise merges with 4-byte LDS accesses and three barriers, all output from one wavefront, took
    // 2.7 us of every workgroup's end.)  All slices sum in the same order, so they agree on the head's m and l bit for bit.
    // (single launch: how many splits of this pair have counted themselves in -- asked for here, needed behind the merge)
    __shared__ int counted;
    float* const counter = MERGE ? P.arrive + ((int64_t)b * n_groups + hg) * P.nqt + qt : nullptr;
    if (MERGE && n_valid_splits > 1 && tid == 0) counted = (int)__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    st.l[0] = both_halves_sum(st.l[0]);          // a state is now (m, l, O) per query
    // Exchange layout per wavefront: O as [d tile][group][64 lanes][4] floats, then m, l as [64].
    constexpr int kStateFloats = 4 * 16 * 64 + 2 * 64;
    static_assert(HPW * KW * kStateFloats * 4 <= (int)sizeof(lds), "merge buffer exceeds the tile region");
    float* xch = reinterpret_cast<float*>(&lds[0][0]) + (wave / KW) * KW * kStateFloats;   // this head's slots
    // (the loop's last barrier already separates the tile reads from these writes; what a slice folds itself stays in its registers: with all of every state written and read,
    // 128 KB through LDS, the merge took 1960 cycles of a workgroup's 14 500 of one sequence, so 1400)
    f32x4 own[4 / KW][4];                           // what this slice folds: d tiles kw, kw + KW, ...
    auto exchange = [&](auto slice) {
        constexpr int MINE = decltype(slice)::value;
        auto quad = [&](int t, int g) { return f32x4{st.o[0][t][4 * g], st.o[0][t][4 * g + 1], st.o[0][t][4 * g + 2], st.o[0][t][4 * g + 3]}; };
        float* dst = xch + MINE * kStateFloats;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (t % KW != MINE) *reinterpret_cast<f32x4*>(dst + ((t * 4 + g) * 64 + lane) * 4) = quad(t, g);
        dst[4 * 16 * 64 + lane] = st.m[0];
        dst[4 * 16 * 64 + 64 + lane] = st.l[0];
        __syncthreads();
        float w[KW];                                // weights of the KW states: 2^(m_s - M)
        float M = kMinusBig;
#pragma unroll
        for (int s = 0; s < KW; ++s) { w[s] = xch[s * kStateFloats + 4 * 16 * 64 + lane]; M = fmaxf(M, w[s]); }
        float l = 0.f;
#pragma unroll
        for (int s = 0; s < KW; ++s) {
            w[s] = __builtin_amdgcn_exp2f(w[s] - M);
            l += xch[s * kStateFloats + 4 * 16 * 64 + 64 + lane] * w[s];
        }
        st.m[0] = M;
        st.l[0] = l;
#pragma unroll
        for (int t = 0; t < 4 / KW; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                own[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < KW; ++s)
                    own[t][g] += (s == MINE ? quad(MINE + KW * t, g) : *reinterpret_cast<const f32x4*>(xch + s * kStateFloats + (((MINE + KW * t) * 4 + g) * 64 + lane) * 4)) * w[s];
            }
    };
    // (kw is the same throughout a wavefront; each meets one barrier, whichever branch it takes.  Of four slices each keeps a quarter only: 32 sequences of 1150 keys,
    // whose merge is all through LDS, 42.6 us, with four branches 42.9.)
    if constexpr (KW == 2) {
        if (__builtin_amdgcn_readfirstlane(kw) == 0) exchange(std::integral_constant<int, 0>());
        else exchange(std::integral_constant<int, 1>());
    } else {
        {
            float* dst = xch + kw * kStateFloats;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<f32x4*>(dst + ((t * 4 + g) * 64 + lane) * 4) =
                        f32x4{st.o[0][t][4 * g], st.o[0][t][4 * g + 1], st.o[0][t][4 * g + 2], st.o[0][t][4 * g + 3]};
            dst[4 * 16 * 64 + lane] = st.m[0];
            dst[4 * 16 * 64 + 64 + lane] = st.l[0];
        }
        __syncthreads();
        {
            float w[KW];                                // weights of the KW states: 2^(m_s - M)
            float M = kMinusBig;
#pragma unroll
            for (int s = 0; s < KW; ++s) { w[s] = xch[s * kStateFloats + 4 * 16 * 64 + lane]; M = fmaxf(M, w[s]); }
            float l = 0.f;
#pragma unroll
            for (int s = 0; s < KW; ++s) {
                w[s] = __builtin_amdgcn_exp2f(w[s] - M);
                l += xch[s * kStateFloats + 4 * 16 * 64 + 64 + lane] * w[s];
            }
            st.m[0] = M;
            st.l[0] = l;
#pragma unroll
            for (int t = 0; t < 4 / KW; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    own[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < KW; ++s)
                        own[t][g] += *reinterpret_cast<const f32x4*>(xch + s * kStateFloats + (((kw + KW * t) * 4 + g) * 64 + lane) * 4) * w[s];
                }
        }
    }

    // ---- output: slice kw holds, and stores, the d tiles kw, kw + KW, ... of its head ----------------
    constexpr int kMine = 4 / KW;                // d tile kw + KW * t is `t` below
    auto store_rows = [&](const f32x4 (&acc)[kMine][4], float l) {
        if (!row_ok) return;
        const float inv = l > 0.f ? 1.0f / l : 0.f;              // no valid key at all: zeros
        __bf16* orow = P.o + (int64_t)b * P.o_sb + (int64_t)qrow * P.o_ss + (int64_t)head * P.o_sh;
#pragma unroll
        for (int t = 0; t < kMine; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d = d_of_reg(kw + KW * t, 4 * g, H);
                typename Elem16<E>::vec4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) out[e] = (E)(acc[t][g][e] * inv);
                if (d < P.head_dim) *reinterpret_cast<typename Elem16<E>::vec4*>(orow + d) = out;
            }
    };
    if (n_valid_splits == 1) { store_rows(own, st.l[0]); return; }
    const int64_t slot0 = (((int64_t)b * P.num_q_heads + head) * P.nqt + qt) * P.nsplit;
    if constexpr (!MERGE) {                      // two launches: the combine kernel follows
        if (row_ok) {
            float* po = P.part_o + ((slot0 + split) * 16 * 64 + lane) * 4;
#pragma unroll
            for (int t = 0; t < kMine; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(po + ((kw + KW * t) * 4 + g) * 64 * 4) = own[t][g];
            if (kw == 0 && H == 0) *reinterpret_cast<float2*>(P.part_ml + ((slot0 + split) * kQTile + r) * 2) = float2{st.m[0], st.l[0]};
        }
    } else {

    // ---- single launch: the last split of this (sequence, head group) to arrive merges them ----
    // A split that finds all others counted in is the last, keeps its state in its registers and folds theirs into the result.  Any other
    // writes its partials (in the order of its registers, 1 KB per store: nobody but this kernel reads them), waits until they have reached
    // memory, and counts itself in; it may still turn out to be the last by that count, and folds then.  No cache-wide
    // fence on either side, and nobody waits for anybody.  What this costs falls at the end of a launch: one trip to memory for
    // the other splits' partials, four at a time, by the workgroup that has just finished, where every split used to write its own, wait, count,
    // and the last to read them all back in two rounds of smaller loads (32 sequences of 375-1500 keys, same cuts: 45 -> 39 us).
    __shared__ int i_am_last;
    auto part = [&](int sp, int t, int g) { return P.part_o + (((slot0 + sp) * 16 + (kw + KW * t) * 4 + g) * 64 + lane) * 4; };
    if (counted != n_valid_splits - 1) {
#pragma unroll
        for (int t = 0; t < kMine; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) store_agent(part(split, t, g), own[t][g]);
        if (kw == 0 && H == 0) {
            float* ml = P.part_ml + ((slot0 + split) * kQTile + r) * 2;
            __hip_atomic_store(ml, st.m[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(ml + 1, st.l[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        wait_vector_memory();
        __syncthreads();
        if (tid == 0) i_am_last = atomicAdd(counter, 1.0f) == (float)(n_valid_splits - 1) ? 1 : 0;
        __syncthreads();
        if (!i_am_last) return;
    }
    const int64_t sequence_floats = (int64_t)P.num_q_heads * P.nqt * P.nsplit * kQTile * kHeadDim;       // (below 2^31 bytes: the launch)
    const __amdgpu_buffer_rsrc_t of_sequence =
        __builtin_amdgcn_make_buffer_rsrc(P.part_o + __builtin_amdgcn_readfirstlane(b) * sequence_floats, 0, (int)(sequence_floats * 4), kRawBuffer);
    // the operations of Fold::take4 in its order, split by split in groups of four, whoever is last: the bits of the combine kernel (change both or neither)
    float M = kMinusBig, L = 0.f;
    f32x4 acc[kMine][4];
#pragma unroll
    for (int t = 0; t < kMine; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[t][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < n_valid_splits; i0 += 4) {
        float m[4], l[4];
        f32x4 po[4][kMine][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int sp = min(i0 + i, n_valid_splits - 1);
            const float* ml = P.part_ml + ((slot0 + sp) * kQTile + r) * 2;
            m[i] = __hip_atomic_load(ml, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            l[i] = __hip_atomic_load(ml + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (i0 + i < n_valid_splits && i0 + i != split) {
#pragma unroll
                for (int t = 0; t < kMine; ++t)
#pragma unroll
                    for (int g = 0; g < 4; ++g) po[i][t][g] = load_agent(of_sequence, ((((head * P.nqt + qt) * P.nsplit + sp) * 16 + (kw + KW * t) * 4 + g) * 64 + lane) * 16);
            }
        }
        float Mn = M;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i0 + i == split) { m[i] = st.m[0]; l[i] = st.l[0]; }
            if (i0 + i < n_valid_splits) Mn = fmaxf(Mn, m[i]);
        }
        const float keep = __builtin_amdgcn_exp2f(M - Mn);
        M = Mn;
        L *= keep;
#pragma unroll
        for (int t = 0; t < kMine; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) acc[t][g] *= keep;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i0 + i >= n_valid_splits) break;
            const float w = __builtin_amdgcn_exp2f(m[i] - M);
            L = __builtin_fmaf(w, l[i], L);
#pragma unroll
            for (int t = 0; t < kMine; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[t][g][e] = __builtin_fmaf(w, i0 + i == split ? own[t][g][e] : po[i][t][g][e], acc[t][g][e]);
        }
    }
    store_rows(acc, L);
    if (tid == 0) __hip_atomic_store(counter, 0.f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
    }
}

// Folds the split partials: a workgroup takes ROWS queries of a (sequence, head), a thread four columns of one of them.  The
// kernel is a chain of memory latencies (length -> partials -> output), not of bytes: the loads of the first AHEAD slots are
// on their way before the lengths say how many of them exist (where a slot lies does not depend on it; what lies
// beyond is masked out), and a thread's share of a slot is one load.  (A workgroup per head with 16 columns per thread, the form this
// replaced, took 0.6 us per four pieces of a sequence, which kept the pieces long.)
template <typename E, int AHEAD, int ROWS>
__global__ __launch_bounds__(32 * ROWS) void paged_combine_kernel(const PagedParams P)
{
    constexpr int kParts = kQTile / ROWS;
    const unsigned block = blockIdx.x + mdx::fetch_arguments<sizeof(PagedParams)>();
    const int part = block % kParts, rest = block / kParts;
    const int row_tile = mdx::quotient(rest, P.nqt), qt = rest - row_tile * P.nqt, b = mdx::quotient(row_tile, P.num_q_heads), hq = row_tile - b * P.num_q_heads;
    const int unit = part * (ROWS / 2) + (threadIdx.x >> 6), lane = threadIdx.x & 63;       // a register quad of the attention's wavefronts, and the lane that held it
    const int c = d_of_reg(unit >> 2, 4 * (unit & 3), lane >> 5), s = lane & 31;
    if (c >= P.head_dim || qt * kQTile + s >= P.sq) return;
    const int64_t slot0 = (((int64_t)b * P.num_q_heads + hq) * P.nqt + qt) * P.nsplit;
    const float* part_o = P.part_o + ((slot0 * 16 + unit) * 64 + lane) * 4;
    const float2* part_ml = reinterpret_cast<const float2*>(P.part_ml) + slot0 * kQTile + s;
    int nv = P.nsplit;                         // until the lengths are in: every slot that exists
    Fold F;
    F.init();
    for (int i0 = 0; i0 < nv; i0 += AHEAD) {
        float m[AHEAD / 4][4], l[AHEAD / 4][4];
        f32x4 po[AHEAD / 4][4];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int slot = min(i0 + i, P.nsplit - 1);
            const float2 ml = part_ml[slot * kQTile];
            m[i / 4][i % 4] = ml.x;
            l[i / 4][i % 4] = ml.y;
            po[i / 4][i % 4] = *reinterpret_cast<const f32x4*>(part_o + (int64_t)slot * kQTile * kHeadDim);
        }
        if (i0 == 0) {
            const int ctx = min(P.context_lens[b], P.max_pages * P.page_size);
            const int span = P.span_out ? (int)*P.span_out : P.chunk;     // the attention kernel's choice
            nv = (ctx + span - 1) / span;
            if (nv <= 1) return;               // written directly by the attention kernel
        }
#pragma unroll
        for (int g = 0; g < AHEAD / 4; ++g)
            if (i0 + 4 * g < nv) F.take4(m[g], l[g], po[g], nv - i0 - 4 * g);
    }
    const float inv = F.inverse();
    typename Elem16<E>::vec4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (E)(F.acc[e] * inv);
    *reinterpret_cast<typename Elem16<E>::vec4*>(P.o + (int64_t)b * P.o_sb + (int64_t)(qt * kQTile + s) * P.o_ss + (int64_t)hq * P.o_sh + c) = out;
}

// Reading ahead: rows of a pass, and what is read at most.
constexpr int64_t kReadAheadFewRows = 32, kReadAheadRows = 256;
constexpr int64_t kReadAheadFewBytes = (int64_t)32 << 20, kReadAheadBytes = (int64_t)64 << 20;

// Keys per split.  Measured over batches of 4 to 64 sequences and contexts of 300 to 8000 keys, the
// kernel is fastest with 1.5 to 1.8 workgroups per CU in total (just under the two per CU that are
// resident at once: one round, no tail of late workgroups), with splits of at least 512 keys (a
// workgroup's fixed cost is worth some 300 keys of streaming) and with whole sequences once there
// are about as many (sequence, head group) pairs as CUs (from 192 pairs on) (in the engine's decode pass at batch 32 that beats two
// splits per sequence by 4 %: no partials to write, nothing to combine).  The host knows the
// page-table width, not the lengths: tables are taken to be about 65 % full, and the last split of
// a sequence to be half a split (the attention kernel, which sees the lengths, corrects the split
// both ways: PagedParams::fit_slots).  In the pair-per-CU case up to four splits per sequence are allowed
// and the kernel itself, which sees the lengths, cuts by even shares where the longest is well above one: kWholeFactor
// (*device_span; the dense workgroup numbering that this needs exists for up to 64 sequences).
//
// The counts behind those rules (1.95 workgroups per CU, pairs per CU) are taken from the current device's
// number of compute units, read once per device; 256 on the MI355X that the rules were measured on, and
// where no device can be asked (a shape query in a process without a GPU).
int cu_count() { return mdx::compute_units(); }

// head_groups counts the workgroups that one (sequence, split) pair launches: head groups x query tiles.
int pick_chunk(int bs, int head_groups, int max_pages, int page_size, bool* device_span) {
    *device_span = false;
    const int cus = cu_count();
    const int64_t max_keys = (int64_t)max_pages * page_size;
    const int64_t whole = (max_keys + kChunkAlign - 1) / kChunkAlign * kChunkAlign;   // one split per sequence
    const double per_pair = 1.953 * cus / ((double)bs * head_groups) - 0.5;           // workgroups per pair
    if ((int64_t)bs * head_groups >= (cus * 3) / 4 || per_pair <= 1.0) {
        if (bs > 64 || whole < 4 * kChunkAlign) return (int)whole;
        *device_span = true;
        return (int)((whole / 4 + kChunkAlign - 1) / kChunkAlign * kChunkAlign);
    }
    int64_t chunk = (int64_t)(0.65 * (double)max_keys / per_pair / kChunkAlign + 0.5) * kChunkAlign;
    if (chunk < 2 * kChunkAlign) chunk = 2 * kChunkAlign;
    if (2 * chunk >= max_keys && (int64_t)bs * head_groups >= (cus * 25) / 32) chunk = whole;   // two short splits only to fill CUs
    return (int)chunk;
}

// Where the kernel picks the pieces of few sequences: whether the last split of a pair merges them (single launch) or a combine launch does.  One
// workgroup reads what the combine launch reads through many, so it is for enough pairs to be done next to each other, and for
// sequences of few pieces.  The layer, us, combine launch / merging: tables of 768 keys 8 sequences 22.2 / 19.9, 16: 27.1 / 22.8, 20: 30.3 / 25.8; of 1280 keys 16 of
// a quarter to all of that 29.7 / 24.2; of 2304 keys 8: 31.1 / 28.0, 16: 42.2 / 41.0, 6: 26.8 / 25.5; but 4 of 1280 20.2 / 20.9, one 15.8 / 19.3, 12 of 3328 41.9 / 43.8,
// 16 of 832-3288 41.7 / 42.8.
constexpr int64_t kMergeKeys = 2560;
bool merges_itself(int64_t pairs, int64_t max_keys, int cus) { return pairs >= cus * 3 / 16 && max_keys <= kMergeKeys; }

// Partial slots per sequence: what the host's split needs and, where the kernel cuts by the lengths (up to 64 sequences, not
// device_span), what its own choice of 4 sqrt(total keys) can need, sqrt(longest) / 4 (beyond 16 K keys the pieces grow) -- as far as that keeps the launch's partials
// below 17 MB (1024 slots).
int nsplit_of(int bs, int64_t heads_and_tiles, int max_pages, int page_size, int chunk, bool device_span) {
    const int64_t max_keys = (int64_t)max_pages * page_size;
    const int64_t n = (max_keys + chunk - 1) / chunk;
    if (device_span || bs > 64) return (int)n;
    // sequences that the kernel would leave whole even in tables that are 65 % full need no slots, and no combine launch
    const double longest = 0.65 * (double)max_keys, best = kPieceRoot * sqrt(longest * bs);
    if (n == 1 && stay_whole(longest, best > kLeastPiece ? best : (double)kLeastPiece, bs)) return 1;
    int64_t own = 2;
    while ((own - 1) * (own - 1) * 16 < max_keys) ++own;
    if (own > 1024 / (bs * heads_and_tiles)) own = 1024 / (bs * heads_and_tiles);
    return (int)(own > n ? own : n);
}

}  // namespace

extern "C" int64_t mdx_paged_block_attn_workspace_bytes(int32_t bs, int32_t sq, int32_t num_q_heads,
                                                        int32_t num_kv_heads, int32_t head_dim,
                                                        int32_t max_pages, int32_t page_size)
{
    if (bs <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || max_pages <= 0 || page_size <= 0) return 0;
    if (head_dim > kHeadDim || head_dim % 16 != 0) return 0;       // the fp32-arithmetic kernel: no split, no partials
    const int G = num_q_heads / num_kv_heads;
    const int HPW = (G % 2 == 0) ? 2 : 1;
    const int nqt = sq <= kQTile ? 1 : (sq + kQTile - 1) / kQTile;
    bool device_span;
    const int chunk = pick_chunk(bs, num_q_heads / HPW * nqt, max_pages, page_size, &device_span);
    const int nsplit = nsplit_of(bs, (int64_t)num_q_heads * nqt, max_pages, page_size, chunk, device_span);
    if (nsplit <= 1) return 0;
    return (int64_t)bs * num_q_heads * nqt * nsplit * kQTile * (kHeadDim + 2) * (int64_t)sizeof(float) + 16;   // + the split size
}

namespace mdx {

int launch_paged_f32(const void* q, void* o, const void* k_cache, const void* v_cache,
                     int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                     int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                     int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                     const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                     int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                     int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                     float scale, int32_t dtype, void* workspace, int64_t workspace_bytes, hipStream_t stream);   // paged_attn_f32.hip

// The launch behind every paged entry point of the library.  next, then: what the launches behind it read.
int launch_paged_ahead(const void* q, void* o, const void* k_cache, const void* v_cache,
                 int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                 int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                 int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                 const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                 int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                 int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                 float scale, int32_t dtype,
                 void* workspace, int64_t workspace_bytes, bool single_launch, void* counters, int64_t counter_bytes,
                 const void* next, int64_t next_bytes, const void* then, int64_t then_bytes, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(next_bytes >= 0 && then_bytes >= 0 && (next || next_bytes == 0) && (then || then_bytes == 0) && next_bytes % 16 == 0 &&
                then_bytes % 16 == 0 && mdx::aligned16(next) && mdx::aligned16(then), MDX_EINVAL,
                "paged_block_attn: what is read ahead starts at and is a multiple of 16 bytes");
    MDX_REQUIRE(bs >= 0 && sq >= 0 && max_pages >= 0 && num_pages >= 0, MDX_EINVAL, "paged_block_attn: negative size");
    MDX_REQUIRE(dtype == MDX_BF16 || dtype == MDX_F16 || dtype == MDX_F32, MDX_EUNSUPPORTED, "paged_block_attn: dtype %d (bf16, fp16 or fp32)", dtype);
    // 16-bit elements and heads of 16, 32, ..., 128 columns run on the 16-bit matrix instructions; fp32 tensors and
    // the other head widths up to 256 on the fp32 one (paged_attn_f32.hip: cut into as many pieces as the workspace has room for)
    const bool f32_arithmetic = dtype == MDX_F32 || head_dim > kHeadDim || head_dim % 16 != 0;
    MDX_REQUIRE(head_dim >= 4 && head_dim <= 256 && head_dim % 4 == 0, MDX_EUNSUPPORTED,
                "paged_block_attn: head_dim %d (multiples of 4 up to 256)", head_dim);
    MDX_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0, MDX_EINVAL,
                "paged_block_attn: Hq %d not a multiple of Hkv %d", num_q_heads, num_kv_heads);
    MDX_REQUIRE(sq <= kMaxSq, MDX_EUNSUPPORTED, "paged_block_attn: %d queries per sequence (max %d)", sq, kMaxSq);
    MDX_REQUIRE(page_size > 0 && page_size % 32 == 0, MDX_EUNSUPPORTED,
                "paged_block_attn: page_size %d not a multiple of 32", page_size);
    MDX_REQUIRE(scale > 0.f, MDX_EINVAL, "paged_block_attn: scale must be positive");
    if (bs == 0 || sq == 0) return MDX_OK;
    MDX_REQUIRE(max_pages > 0, MDX_EINVAL, "paged_block_attn: empty block table");
    MDX_REQUIRE(q && o && k_cache && v_cache && block_table && context_lens, MDX_EINVAL, "paged_block_attn: null pointer");
    MDX_REQUIRE(bt_stride >= max_pages, MDX_EINVAL, "paged_block_attn: bt_stride < max_pages");
    if (f32_arithmetic)
        return launch_paged_f32(q, o, k_cache, v_cache, q_stride_b, q_stride_s, q_stride_h, o_stride_b, o_stride_s, o_stride_h,
                                cache_stride_page, cache_stride_tok, cache_stride_head, block_table, bt_stride, context_lens,
                                bs, sq, num_q_heads, num_kv_heads, head_dim, max_pages, page_size, num_pages, scale, dtype, workspace, workspace_bytes, stream);
    MDX_REQUIRE(mdx::aligned16(q) && mdx::aligned16(o) && mdx::aligned16(k_cache) && mdx::aligned16(v_cache) &&
                q_stride_b % 8 == 0 && q_stride_s % 8 == 0 && q_stride_h % 8 == 0 &&
                o_stride_b % 8 == 0 && o_stride_s % 8 == 0 && o_stride_h % 8 == 0 &&
                cache_stride_page % 8 == 0 && cache_stride_tok % 8 == 0 && cache_stride_head % 8 == 0,
                MDX_EUNSUPPORTED, "paged_block_attn: tensors must be 16-byte aligned with strides that are multiples of 8 elements");

    const int G = num_q_heads / num_kv_heads;
    const int HPW = (G % 2 == 0) ? 2 : 1;
    PagedParams P;
    P.q = (const __bf16*)q; P.o = (__bf16*)o; P.k_cache = (const __bf16*)k_cache; P.v_cache = (const __bf16*)v_cache;
    P.q_sb = q_stride_b; P.q_ss = q_stride_s; P.q_sh = q_stride_h;
    P.o_sb = o_stride_b; P.o_ss = o_stride_s; P.o_sh = o_stride_h;
    P.c_sp = cache_stride_page; P.c_st = cache_stride_tok; P.c_sh = cache_stride_head;
    P.block_table = block_table; P.bt_stride = bt_stride; P.context_lens = context_lens;
    P.bs = bs; P.sq = sq; P.heads_per_kv = G; P.page_size = page_size; P.max_pages = max_pages;
    P.page_shift = -1;
    for (int i = 0; i < 31; ++i) if (page_size == (1 << i)) P.page_shift = i; P.num_pages = num_pages;
    bool device_span;
    P.nqt = (sq + kQTile - 1) / kQTile;
    const int64_t wg_per_pair = (int64_t)(num_q_heads / HPW) * P.nqt;               // workgroups of one (sequence, split)
    const int cus = cu_count();
    P.chunk = pick_chunk(bs, (int)wg_per_pair, max_pages, page_size, &device_span);
    P.nsplit = nsplit_of(bs, (int64_t)num_q_heads * P.nqt, max_pages, page_size, P.chunk, device_span);
    P.num_q_heads = num_q_heads;
    P.by_bs = mdx::divisor(bs, (uint64_t)bs * P.nsplit);
    P.head_dim = head_dim;
    P.c = scale * kLog2e;
    P.part_o = nullptr; P.part_ml = nullptr; P.span_out = nullptr; P.arrive = nullptr; P.fit_slots = 0;
    // Up to one (sequence, head group) pair per CU: workgroups of 8 wavefronts on 128-key tiles, so that a
    // CU that holds a single workgroup still has two wavefronts per SIMD (batch 32 x 8 KV heads: 79 -> 69 us
    // on equal lengths); with more pairs than CUs the second round costs more than that gains.
    const bool eight = device_span && (int64_t)bs * wg_per_pair <= cus;
    const int resident = cus * (HPW == 2 && !eight ? 2 : 1);           // workgroups at once
    if (P.nsplit > 1) {
        const int64_t n_slots = (int64_t)bs * num_q_heads * P.nqt * P.nsplit;
        const int64_t need = n_slots * kQTile * (kHeadDim + 2) * (int64_t)sizeof(float) + 16;
        MDX_REQUIRE(workspace && workspace_bytes >= need, MDX_EWORKSPACE,
                    "paged_block_attn: workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
        MDX_REQUIRE(mdx::aligned16(workspace), MDX_EWORKSPACE, "paged_block_attn: workspace not 16-byte aligned");
        P.part_o = static_cast<float*>(workspace);
        P.part_ml = P.part_o + n_slots * kQTile * kHeadDim;
        if (device_span) P.fit_slots = -resident;
        else if (bs <= 64) P.fit_slots = resident;
        if (P.fit_slots != 0) P.span_out = P.part_ml + n_slots * kQTile * 2;
        // Single launch: the partials are written through with agent-scope stores and read back with
        // agent-scope loads, so counting in costs a workgroup the wait for its own stores and one atomic,
        // not a device-wide release (a write-back walk of its XCD's L2).  With about a pair per CU that always beats the combine launch (24 sequences of
        // 1250-5000 keys 75 / 72 us, 48 of 550-2200 74 / 68, and sequences that stay whole pay nothing); with fewer it does for enough pairs
        // whose sequences come to few pieces (merges_itself).  Those launches take two where there are no counters to use.
        const int64_t pairs = (int64_t)bs * wg_per_pair, need_c = pairs * (int64_t)sizeof(float);
        const bool have_counters = counters && counter_bytes >= need_c && ((uintptr_t)counters & 3) == 0;
        // (a sequence's partials: 31 bits of bytes, or two launches)
        const bool addressable = (int64_t)num_q_heads * P.nqt * P.nsplit * kQTile * kHeadDim * 4 < ((int64_t)1 << 31);
        if (single_launch && device_span) {
            MDX_REQUIRE(counters && counter_bytes >= need_c, MDX_EWORKSPACE,
                        "paged_block_attn: %lld bytes of arrival counters needed, %lld given", (long long)need_c, (long long)counter_bytes);
            MDX_REQUIRE(((uintptr_t)counters & 3) == 0, MDX_EWORKSPACE, "paged_block_attn: counters not 4-byte aligned");
            if (addressable) P.arrive = static_cast<float*>(counters);
        } else if (single_launch && P.fit_slots > 0 && have_counters && addressable && merges_itself(pairs, (int64_t)max_pages * page_size, cus)) {
            P.arrive = static_cast<float*>(counters);
        }
    }
    // head group fastest, then the dense (sequence, split) index
    MDX_REQUIRE((int64_t)bs * P.nsplit <= 65535, MDX_EUNSUPPORTED, "paged_block_attn: bs * splits %lld > 65535", (long long)bs * P.nsplit);
    // With pieces of kShareFactor shares and more there are at most 1 / kShareFactor cuts per workgroup that is resident of a head group,
    // whatever nsplit allows.
    const int64_t most_pairs = bs + (int64_t)((double)resident / (kShareFactor * (double)wg_per_pair)) + 1;
    const int pairs_y = device_span && most_pairs < (int64_t)bs * P.nsplit ? (int)most_pairs : bs * P.nsplit;
    const dim3 grid((unsigned)(num_q_heads / HPW * P.nqt), (unsigned)pairs_y);
    const unsigned n_heads = (unsigned)(bs * num_q_heads * P.nqt);
    // Reading ahead, by rows of the pass (kReadAhead*).  Engine, ms per generation without / with, contexts of 1088 and more in tables of 2048: one request
    // 68.0 / 66.2, two 79.8 / 78.2, three 96.1 / 91.0, four 100.2 / 95.9, six 121.8 / 119.8, eight 132.8 / 130.7; of 32: one 61.6 / 60.7, four 82.2 / 77.9,
    // eight 98.1 / 96.7.  More rows: 16 requests 190.3 / 190.7 (the attention streams by itself then, and the products are bound by other things).  32 rows have
    // the shortest attention: all of 56 MB there 68.6, a workgroup on every other CU and 32 MB 66.2, and only where each reader has a CU to itself beside
    // all workgroups of the attention, with keys or without: us per decode pass without / with, one request of 1088 in tables of 2048 1808 / 1764, of 3072
    // 1814 / 1775, of 4096 1816 / 1817, of 8192 1817 / 1824 (of 4096 there 1943 / 1952).  Long contexts by themselves do no harm, although their K/V
    // passes through the same cache behind the readers: two of 4096 to 15000 in 16384 2257 / 2213 to 2724 / 2748, four of 15000 3607 / 3470, six 4605 / 4487, eight
    // of 8000 in 8192 4126 / 4061; only eight of 12000 to 15000 (390 MB and more per layer) are slower, 5189 / 5212.
    ReadAhead A{};
    int64_t budget = 0;
    int readers = 0;
    const int64_t pass_rows = (int64_t)bs * sq;
    if (next_bytes + then_bytes > 0 && dtype == MDX_BF16 && HPW == 2 && !eight && pass_rows <= kReadAheadRows) {
        const bool few = pass_rows <= kReadAheadFewRows;
        budget = few ? kReadAheadFewBytes : kReadAheadBytes;
        const int64_t attending = wg_per_pair * pairs_y, reading = few ? cus / 2 : cus;
        if (!few || attending + reading <= cus) readers = (int)(reading / wg_per_pair);
        const int64_t n0 = next_bytes < budget ? next_bytes : budget, n1 = then_bytes < budget - n0 ? then_bytes : budget - n0;
        A = ReadAhead{{static_cast<const u32x4*>(next), static_cast<const u32x4*>(then)}, {(int)(n0 / 16), (int)(n1 / 16)}, pairs_y};
    }
    if (pairs_y + readers > 65535) readers = 0;
    const bool two_launches = P.nsplit > 1 && !P.arrive;
    auto attend = [&](auto element, auto merge) {
        typedef decltype(element) E;
        constexpr bool M = decltype(merge)::value;
        if constexpr (std::is_same<E, __bf16>::value) {
            if (readers > 0) { paged_block_attn_kernel<E, 2, 2, 4, M, ReadAhead><<<dim3(grid.x, grid.y + readers), 256, 0, stream>>>(P, A); return; }
        }
        if (HPW == 2 && eight) paged_block_attn_kernel<E, 2, 2, 8, M><<<grid, 512, 0, stream>>>(P);
        else if (HPW == 2)     paged_block_attn_kernel<E, 2, 2, 4, M><<<grid, 256, 0, stream>>>(P);
        else                   paged_block_attn_kernel<E, 1, 1, 4, M><<<grid, 256, 0, stream>>>(P);
    };
    if (dtype == MDX_F16) { if (P.arrive) attend(_Float16(), std::true_type()); else attend(_Float16(), std::false_type()); }
    else                  { if (P.arrive) attend(__bf16(), std::true_type()); else attend(__bf16(), std::false_type()); }
    int rc = mdx::check_launch("paged_block_attn");
    if (rc != MDX_OK || !two_launches) return rc;
    // The slots asked for at once.  Many heads: four (sequences of so many have few pieces, and workgroups enough to wait beside each other;
    // with two queries per thread and half the workgroups, 9 x 1000-3000 keys took 34.8 us, this way 33.7, 16 x 512-4096 43.9 and 42.8).
    // Few: eight, or twelve where the sequences of tables that are 65 % full have about as many pieces or up to
    // half as many again.  (One sequence of 1337 keys, twelve against eight: 14.8 and 15.3 us, 1000: 14.2 and 14.7, two of 3000 to 3500:
    // 21.4 and 21.9, three of 3000 to 5000: 25.3 and 25.9; but one of 300: 12.3 and 12.1, of 2500: 17.2 and 16.9.)
    const double pieces = sqrt(0.65 * max_pages * page_size / bs) / kPieceRoot;
    // Up to 64 heads: two queries per workgroup, so that the partials come in through many CUs (one sequence of 1337 keys 14.6 -> 14.3 us, of
    // 4000 19.2 -> 18.5, four of 1000 to 3000 23.5 -> 23.2; eight of those 29.9 and 30.6).
    const bool twelve = pieces > 7 && pieces <= 9.5;
    auto combine = [&](auto element) {
        typedef decltype(element) E;
        if (n_heads <= 64) {
            if (twelve) paged_combine_kernel<E, 12, 2><<<kQTile / 2 * n_heads, 64, 0, stream>>>(P);
            else        paged_combine_kernel<E, 8, 2><<<kQTile / 2 * n_heads, 64, 0, stream>>>(P);
        } else {
            if (n_heads > 128) paged_combine_kernel<E, 4, 8><<<kQTile / 8 * n_heads, 256, 0, stream>>>(P);
            else if (twelve)   paged_combine_kernel<E, 12, 8><<<kQTile / 8 * n_heads, 256, 0, stream>>>(P);
            else               paged_combine_kernel<E, 8, 8><<<kQTile / 8 * n_heads, 256, 0, stream>>>(P);
        }
    };
    if (dtype == MDX_F16) combine(_Float16()); else combine(__bf16());
    return mdx::check_launch("paged_combine");
}

int launch_paged(const void* q, void* o, const void* k_cache, const void* v_cache,
                 int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                 int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                 int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                 const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                 int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                 int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                 float scale, int32_t dtype,
                 void* workspace, int64_t workspace_bytes, bool single_launch, void* counters, int64_t counter_bytes,
                 mdx_stream_t stream)
{
    return launch_paged_ahead(q, o, k_cache, v_cache, q_stride_b, q_stride_s, q_stride_h, o_stride_b, o_stride_s, o_stride_h,
                              cache_stride_page, cache_stride_tok, cache_stride_head, block_table, bt_stride, context_lens,
                              bs, sq, num_q_heads, num_kv_heads, head_dim, max_pages, page_size, num_pages, scale, dtype,
                              workspace, workspace_bytes, single_launch, counters, counter_bytes, nullptr, 0, nullptr, 0, stream);
}

}  // namespace mdx

extern "C" int mdx_paged_block_attn(const void* q, void* o, const void* k_cache, const void* v_cache,
                                    int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                                    int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                                    int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                                    const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                                    int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                                    int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                                    float scale, int32_t dtype,
                                    void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return mdx::launch_paged(q, o, k_cache, v_cache, q_stride_b, q_stride_s, q_stride_h, o_stride_b, o_stride_s, o_stride_h,
                        cache_stride_page, cache_stride_tok, cache_stride_head, block_table, bt_stride, context_lens,
                        bs, sq, num_q_heads, num_kv_heads, head_dim, max_pages, page_size, num_pages, scale, dtype,
                        workspace, workspace_bytes, false, nullptr, 0, stream);
}

extern "C" int64_t mdx_paged_block_attn_counter_bytes(int32_t bs, int32_t num_q_heads, int32_t num_kv_heads)
{
    if (bs <= 0 || num_q_heads <= 0 || num_kv_heads <= 0) return 0;
    const int G = num_q_heads / num_kv_heads;
    // one counter per (sequence, head group, query tile), sized for the largest block (four tiles of 32 queries)
    return (int64_t)bs * (num_q_heads / ((G % 2 == 0) ? 2 : 1)) * (kMaxSq / kQTile) * (int64_t)sizeof(float);
}

extern "C" int32_t mdx_paged_block_attn_needs_counters(int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads, int32_t max_pages, int32_t page_size)
{
    if (bs <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || max_pages <= 0 || page_size <= 0) return 0;
    const int hpw = (num_q_heads / num_kv_heads) % 2 == 0 ? 2 : 1, nqt = sq <= kQTile ? 1 : (sq + kQTile - 1) / kQTile;
    bool device_span;
    pick_chunk(bs, num_q_heads / hpw * nqt, max_pages, page_size, &device_span);
    return device_span;
}

extern "C" int mdx_paged_block_attn_single_launch(const void* q, void* o, const void* k_cache, const void* v_cache,
                                                  int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                                                  int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                                                  int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                                                  const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                                                  int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                                                  int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                                                  float scale, int32_t dtype,
                                                  void* workspace, int64_t workspace_bytes,
                                                  void* counters, int64_t counter_bytes, mdx_stream_t stream)
{
    return mdx::launch_paged(q, o, k_cache, v_cache, q_stride_b, q_stride_s, q_stride_h, o_stride_b, o_stride_s, o_stride_h,
                        cache_stride_page, cache_stride_tok, cache_stride_head, block_table, bt_stride, context_lens,
                        bs, sq, num_q_heads, num_kv_heads, head_dim, max_pages, page_size, num_pages, scale, dtype,
                        workspace, workspace_bytes, true, counters, counter_bytes, stream);
}

extern "C" int mdx_paged_block_attn_read_ahead(const void* q, void* o, const void* k_cache, const void* v_cache,
                                               int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                                               int64_t o_stride_b, int64_t o_stride_s, int64_t o_stride_h,
                                               int64_t cache_stride_page, int64_t cache_stride_tok, int64_t cache_stride_head,
                                               const int32_t* block_table, int64_t bt_stride, const int32_t* context_lens,
                                               int32_t bs, int32_t sq, int32_t num_q_heads, int32_t num_kv_heads,
                                               int32_t head_dim, int32_t max_pages, int32_t page_size, int64_t num_pages,
                                               float scale, int32_t dtype,
                                               void* workspace, int64_t workspace_bytes, void* counters, int64_t counter_bytes,
                                               const void* next, int64_t next_bytes, const void* then, int64_t then_bytes,
                                               mdx_stream_t stream)
{
    return mdx::launch_paged_ahead(q, o, k_cache, v_cache, q_stride_b, q_stride_s, q_stride_h, o_stride_b, o_stride_s, o_stride_h,
                                   cache_stride_page, cache_stride_tok, cache_stride_head, block_table, bt_stride, context_lens,
                                   bs, sq, num_q_heads, num_kv_heads, head_dim, max_pages, page_size, num_pages, scale, dtype,
                                   workspace, workspace_bytes, counters != nullptr, counters, counter_bytes,
                                   next, next_bytes, then, then_bytes, stream);
}
