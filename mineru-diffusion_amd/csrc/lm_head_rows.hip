// The fused vocabulary projection for few rows (up to 128: a decode pass of one to four sequences, or what is left masked of
// more): logits x . W^T, rounded to bf16, reduced to (max, sum of exp, first argmax) in registers.  With so few rows it is a read
// of W (622 MB at 151 936 x 2048): fragments of W straight
// from memory into registers, x through LDS without passing registers.  One workgroup per CU walks the vocabulary in tiles of
// 128 rows without a pause between tiles; a lane keeps the running state of its rows of x over all its logits, so that a
// workgroup leaves one record per row at its end and the fold over the records is short.
//
//  * up to 32 rows and 2048 columns x fits in LDS whole (128 KB), the wavefronts share nothing else and need no barrier: each
//    streams its own rows of W, three steps of 256 columns (24 KB) ahead of the product;
//  * otherwise x goes through LDS K step by K step with a barrier per step, W one step ahead.
//
// Rows of W are mostly a power of two apart, so that what all workgroups ask for at the same column meets in few of the memory's channels.  With x whole and
// rows of whole quarters (1024 and 2048 columns) workgroup b therefore takes quarter i ^ (b % 4) of its rows as its i-th, and adds the quarters' sums as (0th + 1st) + (2nd +
// 3rd): the same two meet whatever b is, so that equal rows have equal logits wherever they stand and the first of them is taken.  (us, 2048 columns, all from column 0 on / so: 12 rows
// 119.1 / 109.0, 32 rows 120.5 / 110.5; 1024 columns level.  Eighths 114; each wavefront in an order of its own 115.  A loop without the fixed quarters, whose sums are
// moved at run time, 165.  More rows hold too many sums: 64 rows 141 / 172.)
//
// W is read with ordinary loads: marked nontemporal, the two loads that share a 128-byte line fetch it twice now and then (139
// against 129 us at 32 rows).  Bound: HBM.  us at 16 / 32 / 64 / 128 rows: 109 / 110 / 140 / 170 (5.6 TB/s at 32 rows); tiles of 256 rows
// 200 / 199 / 208 / 200, the library's product and a vocabulary pass 213 / 155 / 161 / 175.
#include "lm_head.h"
#include <atomic>

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
                merge(st[mt], __shfl_xor(st[mt].m, off), __shfl_xor(st[mt].s, off), __shfl_xor(st[mt].idx, off), c[mt]);
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

// Up to 32 rows, x whole in LDS as panels of 512 columns.
constexpr int kPanel = 512, kSub = 256, kRing = 4, kMaxWhole = 2048;
__global__ __launch_bounds__(kThreads, 1) void lm_head_whole_kernel(const LmHeadParams P)
{
    constexpr int MT = 2, kPanelBytes = 16 * MT * kPanel * 2;
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
    const int subs = P.hidden / kSub, n_steps = tiles_of_workgroup(P) * subs;
    Rows<MT> rows;
    rows.init(P, lane & 15);
    f32x4 acc[MT] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};

    for (int k = 0; k < P.hidden; k += kPanel) load_x<MT, kPanel>(P, lds0 + k / kPanel * kPanelBytes, k, wave, lane);
    Weights<kSub / 64> ring[kRing];
    int f_tile = blockIdx.x, f_sub = 0, m_tile = blockIdx.x, m_sub = 0;           // the step being fetched, and the one being multiplied
    auto fetch = [&](Weights<kSub / 64>& d) {
        load_weights(d, P, f_tile, f_sub * kSub, wave, lane);
        if (++f_sub == subs) { f_sub = 0; f_tile += gridDim.x; }
    };
#pragma unroll
    for (int r = 0; r < kRing - 1; ++r) fetch(ring[r]);                          // (a tile has at least two steps, and reading a tile too many is in bounds)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");                // x is in LDS for everybody
    for (int t = 0; t < n_steps; t += kRing) {
#pragma unroll
        for (int r = 0; r < kRing; ++r) {
            if (t + r + kRing - 1 < n_steps) fetch(ring[(r + kRing - 1) % kRing]);
            __builtin_amdgcn_sched_barrier(0);
            if (t + r < n_steps) {
                multiply<MT, kPanel>(acc, ring[r], lds + m_sub / 2 * kPanelBytes, (m_sub & 1) * (kSub / 8), lane);
                if (++m_sub == subs) {
                    rows.take(acc, m_tile * kTileRows + wave * 16 + 4 * (lane >> 4), P.vocab);
                    m_sub = 0;
                    m_tile += gridDim.x;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    rows.finish(P, lds, tid);
}

// The same where a row is SUBS steps, whole quarters: in an order of the workgroup's own.
constexpr int kParts = 4;
template <int SUBS>
__global__ __launch_bounds__(kThreads, 1) void lm_head_parts_kernel(const LmHeadParams P)
{
    constexpr int MT = 2, kPanelBytes = 16 * MT * kPanel * 2, kEach = SUBS / kParts, kFar = kRing - 1;
    static_assert(SUBS % kRing == 0 && SUBS % kParts == 0, "a tile begins with the ring's first");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
    const int p = ((int)blockIdx.x & (kParts - 1)) * kEach, tiles = tiles_of_workgroup(P);
    auto sub_of = [&](int i) { return (i / kEach * kEach ^ p) + i % kEach; };
    Rows<MT> rows;
    rows.init(P, lane & 15);
#pragma unroll
    for (int k = 0; k < SUBS * kSub; k += kPanel) load_x<MT, kPanel>(P, lds0 + k / kPanel * kPanelBytes, k, wave, lane);
    Weights<kSub / 64> ring[kRing];
    int tile = blockIdx.x;
#pragma unroll
    for (int r = 0; r < kFar; ++r) load_weights(ring[r], P, tile, sub_of(r) * kSub, wave, lane);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");                // x is in LDS for everybody
    for (int n = 0; n < tiles; ++n) {
        const int next = tile + (int)gridDim.x;
        f32x4 part[kParts][MT];
#pragma unroll
        for (int i = 0; i < SUBS; ++i) {
            if (i + kFar < SUBS || n + 1 < tiles) load_weights(ring[(i + kFar) % kRing], P, i + kFar < SUBS ? tile : next, sub_of((i + kFar) % SUBS) * kSub, wave, lane);
            __builtin_amdgcn_sched_barrier(0);
            const int sub = sub_of(i);
            if (i % kEach == 0)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) part[i / kEach][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            multiply<MT, kPanel>(part[i / kEach], ring[i % kRing], lds + sub / 2 * kPanelBytes, (sub & 1) * (kSub / 8), lane);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) part[0][mt] = (part[0][mt] + part[1][mt]) + (part[2][mt] + part[3][mt]);
        rows.take(part[0], tile * kTileRows + wave * 16 + 4 * (lane >> 4), P.vocab);
        tile = next;
    }
    rows.finish(P, lds, tid);
}

// MT: tiles of 16 rows of x.  KC: columns per step.
template <int MT, int KC>
__global__ __launch_bounds__(kThreads, 1) void lm_head_rows_kernel(const LmHeadParams P)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];            // two x tiles of [16 MT][KC]
    constexpr int kBufBytes = 16 * MT * KC * 2, kPairs = KC / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
    const int chunks = P.hidden / KC, n_steps = tiles_of_workgroup(P) * chunks;
    Rows<MT> rows;
    rows.init(P, lane & 15);
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    Weights<kPairs> a, b;
    int f_tile = blockIdx.x, f_chunk = 0, m_tile = blockIdx.x, m_chunk = 0;       // the step being fetched, and the one being multiplied
    auto fetch = [&](Weights<kPairs>& d, int buf) {
        load_x<MT, KC>(P, lds0 + buf * kBufBytes, f_chunk * KC, wave, lane);
        load_weights(d, P, f_tile, f_chunk * KC, wave, lane);
        if (++f_chunk == chunks) { f_chunk = 0; f_tile += gridDim.x; }
    };
    auto step = [&](const Weights<kPairs>& d, int buf) {
        multiply<MT, KC>(acc, d, lds + buf * kBufBytes, 0, lane);
        if (++m_chunk < chunks) return;
        rows.take(acc, m_tile * kTileRows + wave * 16 + 4 * (lane >> 4), P.vocab);
        m_chunk = 0;
        m_tile += gridDim.x;
    };
    // A step's x is in LDS for everybody once each wavefront has waited for its own loads; its W, issued after them, may still be on
    // its way (the compiler waits for that register by register).
    auto arrived = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(2 * kPairs) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch(a, 0);
    for (int t = 0; t < n_steps; t += 2) {
        arrived();
        if (t + 1 < n_steps) fetch(b, 1);
        __builtin_amdgcn_sched_barrier(0);
        step(a, 0);
        if (t + 1 >= n_steps) break;
        arrived();
        if (t + 2 < n_steps) fetch(a, 0);
        __builtin_amdgcn_sched_barrier(0);
        step(b, 1);
    }
    rows.finish(P, lds, tid);
}

// The kernel's LDS limit is raised once per device.
int launch(void (*kernel)(const LmHeadParams), int lds_bytes, std::atomic<bool>* raised, const LmHeadParams& P, hipStream_t stream)
{
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "lm_head_confidence: no current device (%s)", hipGetErrorString(e));
    if (!raised[device].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "lm_head_confidence: cannot reserve %d bytes of LDS (%s)", lds_bytes, hipGetErrorString(e));
        raised[device].store(true, std::memory_order_release);
    }
    kernel<<<(unsigned)P.n_slices, kThreads, lds_bytes, stream>>>(P);
    return mdx::check_launch("lm_head_confidence");
}

template <int MT, int KC> int launch_steps(const LmHeadParams& P, hipStream_t stream)
{
    static std::atomic<bool> raised[64];
    return launch(lm_head_rows_kernel<MT, KC>, 2 * 16 * MT * KC * 2, raised, P, stream);
}

}  // namespace

namespace mdx_head {

bool few_rows_covered(int64_t rows, int64_t hidden) { return rows <= 128 && hidden % (rows <= 64 ? 512 : 256) == 0; }

int launch_few_rows(LmHeadParams& P, hipStream_t stream)
{
    P.n_vocab_tiles = (P.vocab + kTileRows - 1) / kTileRows;
    const int cus = mdx::compute_units();
    P.n_slices = P.n_vocab_tiles < cus ? P.n_vocab_tiles : cus;
    if (P.rows <= 32 && P.hidden <= kMaxWhole) {
        static std::atomic<bool> raised[64], raised4[64], raised8[64];
        if (P.hidden == 4 * kSub) return launch(lm_head_parts_kernel<4>, 32 * 4 * kSub * 2, raised4, P, stream);
        if (P.hidden == 8 * kSub) return launch(lm_head_parts_kernel<8>, 32 * 8 * kSub * 2, raised8, P, stream);
        return launch(lm_head_whole_kernel, 32 * kMaxWhole * 2, raised, P, stream);
    }
    return P.rows <= 32 ? launch_steps<2, 512>(P, stream) : P.rows <= 64 ? launch_steps<4, 512>(P, stream) : launch_steps<8, 256>(P, stream);
}

}  // namespace mdx_head
