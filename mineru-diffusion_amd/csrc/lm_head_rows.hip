// The fused vocabulary projection for up to 32 rows of 2048 columns, and of 512 and 1024 for large vocabularies (a decode pass of one sequence, or what is left masked of
// more): logits x . W^T, rounded to bf16, reduced to (max, sum of exp, first argmax) in registers.  With so few rows it is a read of W (622 MB at 151 936 x 2048): fragments of W straight
// from memory into registers, x whole in LDS (at most 128 KB).  One workgroup per CU walks the vocabulary in tiles of
// 128 rows without a pause between tiles; the wavefronts share nothing but x and need no barrier: each streams its own rows of W, three steps of 256 columns (24 KB)
// ahead of the product.  A lane keeps the running state of its rows of x over all its logits, so that a
// workgroup leaves one record per row at its end and the fold over the records is short.
//
// Rows of W are mostly a power of two apart, so that what all workgroups ask for at the same column meets in few of the memory's channels.  Workgroup b therefore takes
// part i ^ (b % parts) of its rows as its i-th (four parts of 2048 columns, two of the others: parts of 1 KB, or half a row), and adds the parts' sums as (0th + 1st) + (2nd + 3rd): the
// same two meet whatever b is, so that equal rows have equal logits wherever they stand and the first of them is taken.  (us, all from column 0 on / so: 12 rows 119.1 / 109.0, 32 rows
// 120.5 / 110.5.  Eighths 114; each wavefront in an order of its own 115; a loop without the fixed parts, whose sums are moved at run time, 165; 1024 columns in four parts of 512
// bytes 69, in two 60.)  The loads ahead are asked for without a condition: behind one that might not have been, the compiler waits for all of them (512 columns 68 us, so 36).
//
// W is read with ordinary loads: marked nontemporal, the two loads that share a 128-byte line fetch it twice now and then (139
// against 129 us at 32 rows).  Bound: HBM.  us at 12 / 32 rows: 109 / 110 (5.6 TB/s); tiles of 64 x 128 (lm_head_unmask.hip) 124 / 124, the library's product and a vocabulary
// pass 213 / 155.  More rows are better served by those tiles: 64 rows of 2048 through LDS step by step, a barrier each, 141 against 127, 128 rows 170 against 154.  So are other widths,
// but where a workgroup has more than four tiles of 512 or 1024 columns (32 rows, here / there, us: 151 936 entries, 512 columns 35.6 / 38.3, 1024 60.2 / 64.1; 100 000 31 / 30, 50 / 49;
// 48 000 21.6 / 18.0, 31 / 28.5; 32 000 16 / 13.4, 22.7 / 19.7).  1536 columns: level at 151 936 (90 / 91), 70 / 68 at 100 000, 29.8 / 27.3 at 32 000.
#include "lm_head.h"
#include "linear_tile.h"

namespace {

using namespace mdx_head;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kWaves = 8, kThreads = 64 * kWaves, kTileRows = 16 * kWaves;

__device__ __forceinline__ void load_to_lds(unsigned lds, const void* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(lds), "v"(p) : "memory");
}

struct State { float m, s; int idx; };
// Two states of disjoint columns; on equal maxima the lower index.
__device__ __forceinline__ void merge(State& a, float m, float s, int idx, float c) {
    const float M = fmaxf(a.m, m);
    if (!(M > -INFINITY)) return;
    a.s = (a.m > -INFINITY ? a.s * __builtin_amdgcn_exp2f((a.m - M) * c) : 0.f) + (m > -INFINITY ? s * __builtin_amdgcn_exp2f((m - M) * c) : 0.f);
    a.idx = m > a.m ? idx : m == a.m ? min(a.idx, idx) : a.idx;
    a.m = M;
}

// A lane's rows of x over the columns of W that it has seen: row l16 of each of the MT tiles, columns 4 g .. 4 g + 3 of a
// wavefront's 16 per tile of W.
template <int MT> struct Rows {
    float c[MT];
    State st[MT];
    __device__ __forceinline__ void init(const LmHeadParams& P, int l16) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            c[mt] = row_scale(P, mt * 16 + l16);
            st[mt] = State{-INFINITY, 0.f, 0x7fffffff};
        }
    }
    // The sums of a tile, which are cleared for the next; n0: this lane's first column.
    __device__ __forceinline__ void take(f32x4 (&acc)[MT], int n0, int vocab) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float x[4], top = -INFINITY;
            int first = 0;
#pragma unroll
            for (int i = 3; i >= 0; --i) {
                x[i] = n0 + i < vocab ? (float)(__bf16)acc[mt][i] : -INFINITY;
                if (x[i] >= top) { top = x[i]; first = i; }
                acc[mt][i] = 0.f;
            }
            if (top > st[mt].m) {
                st[mt].s = st[mt].m > -INFINITY ? st[mt].s * __builtin_amdgcn_exp2f((st[mt].m - top) * c[mt]) : 0.f;
                st[mt].m = top;
                st[mt].idx = n0 + first;
            }
            if (st[mt].m > -INFINITY) {
#pragma unroll
                for (int i = 0; i < 4; ++i) st[mt].s += __builtin_amdgcn_exp2f((x[i] - st[mt].m) * c[mt]);
            }
        }
    }
    // One record per row: the four lanes of a row, then the wavefronts through LDS (whose x tiles are done with).
    __device__ __forceinline__ void finish(const LmHeadParams& P, char* lds, int tid) {
        const int lane = tid & 63, wave = tid >> 6, l16 = lane & 15;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int off = 16; off <= 32; off <<= 1)
                merge(st[mt], mdx::xor_lanes(st[mt].m, off), mdx::xor_lanes(st[mt].s, off), mdx::xor_lanes(st[mt].idx, off), c[mt]);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the x tiles have been read by everybody
        State* states = reinterpret_cast<State*>(lds);                       // [wave][16 MT]
        if (lane < 16) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) states[wave * 16 * MT + mt * 16 + l16] = st[mt];
        }
        __syncthreads();
        if (tid >= P.rows || tid >= 16 * MT) return;
        State a = states[tid];
        const float cr = row_scale(P, tid);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) { const State b = states[w * 16 * MT + tid]; merge(a, b.m, b.s, b.idx, cr); }
        P.records[(int64_t)tid * P.n_slices + blockIdx.x] = Record{a.m, a.s, a.idx, 0};
    }
};

template <int PAIRS> struct Weights { bf16x8 w[PAIRS][2]; };
// A lane's fragments of PAIRS pairs of matrix steps: 32 consecutive bytes per pair, the four lanes of a row cover a line.
template <int PAIRS> __device__ __forceinline__ void load_weights(Weights<PAIRS>& d, const LmHeadParams& P, int tile, int k, int wave, int lane) {
    const int row = min(tile * kTileRows + wave * 16 + (lane & 15), P.vocab - 1);            // (past the vocabulary: its last row again)
    const __bf16* wp = P.w + (int64_t)row * P.w_stride + k + (lane >> 4) * 16;
#pragma unroll
    for (int p = 0; p < PAIRS; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) d.w[p][h] = *reinterpret_cast<const bf16x8*>(wp + p * 64 + h * 8);
}

// Rows [16 MT] x columns [k, k + KC) of x to LDS: position p of row m holds the 16-byte chunk p ^ (m % 16).
template <int MT, int KC> __device__ __forceinline__ void load_x(const LmHeadParams& P, unsigned lds, int k, int wave, int lane) {
    constexpr int kRowLanes = KC / 8, kRowsPerLoad = 64 / kRowLanes;
#pragma unroll
    for (int i = wave; i < 16 * MT / kRowsPerLoad; i += kWaves) {
        const int m = i * kRowsPerLoad + lane / kRowLanes, at = (lane % kRowLanes) ^ (m & 15);
        load_to_lds((unsigned)__builtin_amdgcn_readfirstlane((int)(lds + i * 1024)), P.x + (int64_t)min(m, P.rows - 1) * P.x_stride + k + at * 8);
    }
}

// PAIRS pairs of matrix steps of W against columns [first chunk..] of an x tile of [16 MT][KC] in LDS.
template <int MT, int KC, int PAIRS>
__device__ __forceinline__ void multiply(f32x4 (&acc)[MT], const Weights<PAIRS>& d, const char* x, int chunk0, int lane) {
    const int l16 = lane & 15, g = lane >> 4;
    const char* rows = x + l16 * (KC * 2);
#pragma unroll
    for (int p = 0; p < PAIRS; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = ((chunk0 + p * 8 + g * 2 + h) ^ l16) * 16;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d.w[p][h], *reinterpret_cast<const bf16x8*>(rows + mt * 16 * (KC * 2) + at), acc[mt], 0, 0, 0);
        }
}

__device__ __forceinline__ int tiles_of_workgroup(const LmHeadParams& P) { return (P.n_vocab_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x; }

// x in LDS as panels of 512 columns.  The ring's slots are fixed in the code, so that where a tile's steps are no multiple of the ring two tiles make one pass of the loop.
constexpr int kPanel = 512, kSub = 256, kRing = 4, kLeastRounds = 4;
template <int COLUMNS>
__global__ __launch_bounds__(kThreads, 1) void lm_head_few_rows_kernel(const LmHeadParams P)
{
    constexpr int MT = 2, kPanelBytes = 16 * MT * kPanel * 2, kSubs = COLUMNS / kSub, kParts = kSubs == 8 ? 4 : 2, kEach = kSubs / kParts, kFar = kRing - 1;
    constexpr int kTiles = kSubs % kRing == 0 ? 1 : 2;
    static_assert(kSubs % kParts == 0 && kTiles * kSubs % kRing == 0, "whole parts; a pass of the loop begins with the ring's first");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
    const int p = ((int)blockIdx.x & (kParts - 1)) * kEach, tiles = tiles_of_workgroup(P);
    auto sub_of = [&](int i) { return (i / kEach * kEach ^ p) + i % kEach; };
    Rows<MT> rows;
    rows.init(P, lane & 15);
#pragma unroll
    for (int k = 0; k < COLUMNS; k += kPanel) load_x<MT, kPanel>(P, lds0 + k / kPanel * kPanelBytes, k, wave, lane);
    Weights<kSub / 64> ring[kRing];
    int tile = blockIdx.x;
    auto load_step = [&](int slot, int i) { load_weights(ring[slot], P, tile + i / kSubs * (int)gridDim.x, sub_of(i % kSubs) * kSub, wave, lane); };      // step i from this tile's first on
#pragma unroll
    for (int r = 0; r < kFar; ++r) load_step(r, r);                              // (reading a tile too many is in bounds)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");                // x is in LDS for everybody
    for (int n = 0; n < tiles; n += kTiles) {
#pragma unroll
        for (int u = 0; u < kTiles; ++u) {
            if (n + u >= tiles) break;
            f32x4 part[kParts][MT];
#pragma unroll
            for (int i = 0; i < kSubs; ++i) {
                const int step = u * kSubs + i, sub = sub_of(i);
                load_step((step + kFar) % kRing, i + kFar);
                __builtin_amdgcn_sched_barrier(0);
                if (i % kEach == 0)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) part[i / kEach][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                multiply<MT, kPanel>(part[i / kEach], ring[step % kRing], lds + sub / 2 * kPanelBytes, (sub & 1) * (kSub / 8), lane);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                part[0][mt] += part[1][mt];
                if constexpr (kParts == 4) part[0][mt] += part[2][mt] + part[3][mt];
            }
            rows.take(part[0], tile * kTileRows + wave * 16 + 4 * (lane >> 4), P.vocab);
            tile += gridDim.x;
        }
    }
    rows.finish(P, lds, tid);
}

template <int COLUMNS> int launch(const LmHeadParams& P, hipStream_t stream)
{
    static std::atomic<bool> raised[64];
    constexpr int kLdsBytes = 32 * COLUMNS * 2;
    const int rc = mdx_tile::reserve_lds(reinterpret_cast<const void*>(lm_head_few_rows_kernel<COLUMNS>), kLdsBytes, raised, "lm_head_confidence");
    if (rc != MDX_OK) return rc;
    lm_head_few_rows_kernel<COLUMNS><<<(unsigned)P.n_slices, kThreads, kLdsBytes, stream>>>(P);
    return mdx::check_launch("lm_head_confidence");
}

}  // namespace

namespace mdx_head {

bool few_rows_covered(int64_t rows, int64_t vocab, int64_t hidden)
{
    if (rows > 32) return false;
    return hidden == 2048 || ((hidden == 512 || hidden == 1024) && vocab > (int64_t)kLeastRounds * kTileRows * mdx::compute_units());
}

int launch_few_rows(LmHeadParams& P, hipStream_t stream)
{
    P.n_vocab_tiles = (P.vocab + kTileRows - 1) / kTileRows;
    const int cus = mdx::compute_units();
    P.n_slices = P.n_vocab_tiles < cus ? P.n_vocab_tiles : cus;
    return P.hidden == 512 ? launch<512>(P, stream) : P.hidden == 1024 ? launch<1024>(P, stream) : launch<2048>(P, stream);
}

}  // namespace mdx_head
