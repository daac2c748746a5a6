// Vocabulary projection fused with the confidence reduction of the unmask step: the logits
// x . W^T are produced on the matrix pipe, rounded to bf16 like the projection's output in the reference,
// and reduced to (max, sum of exp, first argmax) while still in registers, so the [rows, vocab] logits
// (311 MB at 1024 rows x 151 936) never travel to HBM and back.
//
// Replaces, for the rows of still-masked positions, ParallelLMHead.forward's F.linear
// (engines/nano_dvlm/nanovllm/layers/embed_head.py:61-67) followed by Sampler.prepare's softmax
// confidence and argmax without noise (layers/sampler.py:11-22).
//
// A workgroup computes a tile of 64 x 128 to 256 x 256 (x rows by vocabulary rows) over the whole hidden dimension
// (linear_tile.h) and leaves one 16-byte record per x row; a second, small kernel folds a row's records (about vocab / 256 or / 128 of them) into x0 /
// x0_p.  What bounds it: the matrix pipe under the board's power limit (at 1024 rows 522 us on data, 441 on zeros, whose clock
// is higher, 380 without loads), 5 us of epilogue per tile, the last round of tiles (500 rows: 4.64 of 5).
#include "lm_head.h"
#include "linear_tile.h"

namespace {

using namespace mdx_head;
using namespace mdx_tile;

constexpr int kFoldThreads = 256;
constexpr float kClamp = -1.0e30f;

struct Best { float m, s; int idx; };                     // max logit, sum of exp2((x - m) c), first index of the max

// (0 where a lane saw nothing: its stand-in maximum must not meet an infinite factor)
__device__ __forceinline__ Best merge(const Best& a, const Best& b, float c) {
    const float A = fmaxf(a.m, kClamp), B = fmaxf(b.m, kClamp), M = fmaxf(A, B);
    Best r;
    r.m = fmaxf(a.m, b.m);
    r.s = a.s * __builtin_amdgcn_exp2f((A - M) * c) + b.s * __builtin_amdgcn_exp2f((B - M) * c);
    r.idx = a.m > b.m ? a.idx : b.m > a.m ? b.idx : min(a.idx, b.idx);
    return r;
}

__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

template <typename T>
__global__ __launch_bounds__(T::kThreads, T::kWaves / 4) void lm_head_confidence_kernel(const LmHeadParams P, const Places places)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const T tile;
    const Place at = place_of(blockIdx.x, places);
    const int xr0 = at.m * T::BM, v0 = at.n * T::BN;
    const int row0 = tile.wm * (T::BM / T::WM) + tile.l16;        // this lane's first x row in the tile
    float c[T::TM];
#pragma unroll
    for (int i = 0; i < T::TM; ++i) c[i] = row_scale(P, xr0 + row0 + 16 * i);
    typename T::Sums acc;
    tile.product(Operands{P.x, P.w, P.x_stride, P.w_stride, P.rows, P.vocab}, xr0, v0, 0, P.hidden / kStepK, lds, acc);

    wait_loads_and_meet<0>();                              // the tile's steps have been read by everybody
    Best* parts = reinterpret_cast<Best*>(lds);            // [WN][BM]
    const int v_lane = v0 + tile.wn * (T::BN / T::WN) + 4 * tile.g;                 // vocabulary index of this lane's first logit
    const bool edge = v0 + T::BN > P.vocab;
#pragma unroll
    for (int i = 0; i < T::TM; ++i) {
        // the lane's logits in ascending vocabulary order, rounded to the projection's bf16; beyond the vocabulary: -inf
        float v[4 * T::TN];
#pragma unroll
        for (int j = 0; j < T::TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[4 * j + e] = (float)(__bf16)acc[i][j][e];
                if (edge && v_lane + 16 * j + e >= P.vocab) v[4 * j + e] = -INFINITY;
            }
        float m = v[0];
#pragma unroll
        for (int k = 1; k < 4 * T::TN; k += 2) m = max3(m, v[k], v[k + 1 < 4 * T::TN ? k + 1 : k]);
        int first = 0;
#pragma unroll
        for (int k = 4 * T::TN - 1; k >= 0; --k) first = v[k] == m ? k : first;
        // one FMA per exponent: the product m c is rounded once and its error taken out of the sum afterwards
        const float ms = fmaxf(m, kClamp), h = ms * c[i];
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4 * T::TN; ++k) s[k & 3] += __builtin_amdgcn_exp2f(__builtin_fmaf(v[k], c[i], -h));
        float sum = ((s[0] + s[1]) + (s[2] + s[3])) * __builtin_amdgcn_exp2f(-__builtin_fmaf(ms, c[i], -h));
        if (m == -INFINITY) sum = 0.f;                     // all of it beyond the vocabulary: 0, not 0 x the correction's infinity
        // (nothing but NaN: no maximum, so that no other lane's loses its index to this one's; the sum stays NaN)
        Best b = Best{fmaxf(m, -INFINITY), sum, v_lane + 16 * (first >> 2) + (first & 3)};
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1)
            b = merge(b, Best{__shfl_xor(b.m, off), __shfl_xor(b.s, off), __shfl_xor(b.idx, off)}, c[i]);
        if (tile.g == 0) parts[tile.wn * T::BM + row0 + 16 * i] = b;
    }
    __syncthreads();
    const int r = threadIdx.x, row = xr0 + r;
    if (r >= T::BM || row >= P.rows) return;
    const float cr = row_scale(P, row);
    Best b = parts[r];
#pragma unroll
    for (int w = 1; w < T::WN; ++w) b = merge(b, parts[w * T::BM + r], cr);
    P.records[(int64_t)row * P.n_slices + at.n] = Record{b.m, b.s, b.idx, 0};
}

// ---- 128 columns: two steps, which leave a tile's epilogue most of the time.  Tiles of 256 x 256 on the generated core of lm_head_core.inc
//      (one wavefront per SIMD), two records per row and tile.  151 936 entries, us, this core / a 256 x 256 tile of linear_tile.h with two steps in LDS: 256 rows 38 / 40,
//      500 57 / 60, 1024 101 / 110, 4096 349 / 392. ----
#include "lm_head_core.inc"

constexpr int kThreads = 256;
constexpr int kTile = 256;                     // vocab rows and x rows per workgroup
constexpr int kSlice = 128;                    // vocab rows per record (one wavefront's share)
constexpr int kLdsBytes = 2 * 2 * kTile * 128; // two stages of (W tile + x tile), 128-byte rows

// 32-bit LDS byte address of a pointer into shared memory (what ds_* instructions and M0 take).
__device__ __forceinline__ unsigned lds_address(const void* p) { return (unsigned)(uintptr_t)(const lds_char*)p; }

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ const void* uniform(const void* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const void*)(((uint64_t)hi << 32) | lo);
}

__global__ __launch_bounds__(kThreads, 1) void lm_head_two_steps_kernel(const LmHeadParams P)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int H = lane >> 5, r = lane & 31;
    const int wv = wave >> 1, wx = wave & 1;              // this wavefront's half of the vocab rows / of the x rows

    // workgroup -> (vocab tile, row tile): groups of 8 vocab tiles, the row tiles of one vocab tile 8 apart
    const int per_group = 8 * P.n_row_tiles;
    const int group = blockIdx.x / per_group, rem = blockIdx.x % per_group;
    const int vtile = group * 8 + (rem & 7), rtile = rem >> 3;
    if (vtile >= P.n_vocab_tiles) return;
    const int v0 = vtile * kTile, xr0 = rtile * kTile;

    const unsigned lds0 = lds_address(lds);
    LmHeadCoreArgs A;
    {
        const int f = (r >> 1) & 7;
        const unsigned pos0 = (unsigned)((f & 6) | ((H ^ f) & 1));
        A.aw = lds0 + (unsigned)((kSlice * wv + r) * 128) + (pos0 << 4);
        A.ax = lds0 + (unsigned)(kTile * 128) + (unsigned)((kSlice * wx + r) * 128) + (pos0 << 4);
    }
    A.row0 = (unsigned)(8 * wave + (lane >> 3));
    A.trow = (unsigned)tid;
    A.ch = (unsigned)((((lane & 7) ^ (((wave & 1) << 2) | (lane >> 4))) & 7) << 4);
    A.wlast = (unsigned)uniform(min(kTile - 1, P.vocab - 1 - v0));
    A.xlast = (unsigned)uniform(min(kTile - 1, P.rows - 1 - xr0));
    A.wsb = (unsigned)uniform((int)(P.w_stride * 2));
    A.xsb = (unsigned)uniform((int)(P.x_stride * 2));
    A.wb = uniform((const void*)(P.w + (int64_t)v0 * P.w_stride));
    A.xb = uniform((const void*)(P.x + (int64_t)xr0 * P.x_stride));
    A.ldsw = (unsigned)uniform((int)(lds0 + (unsigned)(wave * 1024)));
    A.nkb = (unsigned)uniform(P.hidden / 64);
    const int xrow = xr0 + kSlice * wx + r;               // this lane's x row in x tile 0
    A.c0 = row_scale(P, xrow);
    A.c1 = row_scale(P, xrow + 32);
    A.c2 = row_scale(P, xrow + 64);
    A.c3 = row_scale(P, xrow + 96);
    A.vlane = (unsigned)(v0 + kSlice * wv + 4 * H);
    A.vocab = (unsigned)uniform(P.vocab);
    A.edge = (unsigned)uniform(v0 + kTile > P.vocab ? 1 : 0);
    A.xrow = H == 0 ? (unsigned)xrow : 0x7fffffffu;
    A.rows = (unsigned)uniform(P.rows);
    A.pb = uniform((const void*)P.records);
    A.po = (unsigned)(((int64_t)xrow * P.n_slices + (2 * vtile + wv)) * (int64_t)sizeof(Record));
    A.postep = (unsigned)uniform((int)(32 * P.n_slices * (int)sizeof(Record)));
    lm_head_core(A);
}

// One wavefront per x row: folds the row's records (ascending vocabulary slices) into token and confidence.
__global__ __launch_bounds__(kFoldThreads) void lm_head_finalize_kernel(const LmHeadParams P)
{
    const int row = ((int)blockIdx.x + mdx::fetch_arguments<sizeof(LmHeadParams)>()) * (kFoldThreads / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= P.rows) return;
    const float c = row_scale(P, row);
    float m = -INFINITY, s = 0.f;
    int idx = 0x7fffffff;
    auto fold = [&](float m2, float s2, int i2) {
        if (!(m2 > -INFINITY)) return;                    // an empty slice (all of it beyond the vocabulary, or -inf logits)
        const float M = fmaxf(m, m2);
        const float a = fmaxf(m, kClamp) - fmaxf(M, kClamp), b = fmaxf(m2, kClamp) - fmaxf(M, kClamp);
        s = s * __builtin_amdgcn_exp2f(a * c) + s2 * __builtin_amdgcn_exp2f(b * c);
        idx = (m2 > m) ? i2 : ((m2 == m) ? min(idx, i2) : idx);
        m = M;
    };
    // the row's records, eight per lane in flight at a time (a fold per load would make this a chain of memory latencies)
    const u32x4* rec = reinterpret_cast<const u32x4*>(P.records + (int64_t)row * P.n_slices);
    for (int i0 = lane; i0 < P.n_slices; i0 += 64 * 8) {
        u32x4 q[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = i0 + 64 * k;
            q[k] = __builtin_nontemporal_load(rec + (i < P.n_slices ? i : lane));   // (lane < n_slices here: i0 = lane is)
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (i0 + 64 * k < P.n_slices) fold(__uint_as_float(q[k].x), __uint_as_float(q[k].y), (int)q[k].z);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float m2 = mdx::xor_lanes(m, off), s2 = mdx::xor_lanes(s, off);
        const int i2 = mdx::xor_lanes(idx, off);
        fold(m2, s2, i2);
    }
    if (lane == 0) {
        // a row without any finite logit reports token 0 with confidence 0, like the two-step path
        P.x0[row] = idx == 0x7fffffff ? 0 : idx;
        P.x0_p[row] = idx == 0x7fffffff ? 0.f : fminf(1.0f / s, 1.0f);
    }
}

// Records per row that the workspace has room for: the form for few rows and every tile below stay under it.
int slices_of(int64_t vocab) { return (int)((vocab + 255) / 256) * 2; }

template <int BM, int BN, int S, int SX>
int launch_tiles(LmHeadParams& P, hipStream_t stream)
{
    typedef Tile<BM, BN, 4, 2, 1, S, SX, false> T;
    static_assert(T::kStepsBytes <= 160 * 1024 && T::WN * BM * (int)sizeof(Best) <= T::kStepsBytes && BM <= T::kThreads, "LDS, a thread per row");
    static std::atomic<bool> raised[64];
    const int rc = reserve_lds(reinterpret_cast<const void*>(lm_head_confidence_kernel<T>), T::kStepsBytes, raised, "lm_head_confidence");
    if (rc != MDX_OK) return rc;
    P.n_row_tiles = (P.rows + BM - 1) / BM;
    P.n_vocab_tiles = P.n_slices = (P.vocab + BN - 1) / BN;
    const int64_t grid = (int64_t)P.n_row_tiles * P.n_vocab_tiles;
    lm_head_confidence_kernel<T><<<(unsigned)grid, T::kThreads, T::kStepsBytes, stream>>>(P, places_of(P.n_row_tiles, P.n_vocab_tiles, grid));
    return mdx::check_launch("lm_head_confidence");
}

int launch_two_steps(LmHeadParams& P, hipStream_t stream)
{
    static std::atomic<bool> raised[64];
    const int rc = reserve_lds(reinterpret_cast<const void*>(lm_head_two_steps_kernel), kLdsBytes, raised, "lm_head_confidence");
    if (rc != MDX_OK) return rc;
    P.n_row_tiles = (P.rows + kTile - 1) / kTile;
    P.n_vocab_tiles = (P.vocab + kTile - 1) / kTile;
    P.n_slices = slices_of(P.vocab);
    const int64_t grid = (int64_t)((P.n_vocab_tiles + 7) / 8) * 8 * P.n_row_tiles;
    lm_head_two_steps_kernel<<<(unsigned)grid, kThreads, kLdsBytes, stream>>>(P);
    return mdx::check_launch("lm_head_confidence");
}

// Which tile.  Up to 64 rows 64 x 128, of which two fit a CU (72 KB of LDS each), so that one's epilogue has the other's loads beside it; up to 128 rows 128 x 128.  151 936 entries, us,
// through LDS step by step, W straight to registers (which these two replaced) / here: 2048 columns, 40 rows 140 / 125, 64 141 / 127, 80 166 / 150, 128 171 / 154; 1024 columns 69 / 58, 71 / 61, 90 /
// 82, 91 / 85; 4096 256 / 234, 260 / 231, 314 / 258, 318 / 265.  (128 x 256: 40 rows 152, 128 159; 128 x 128 with two steps in LDS, two a CU, 128 rows 163; 64 x 128 with two steps 141.)
// Of 65 to 128 rows, 128 x 256 where it halves the rounds (100 rows, us, 128 x 128 / so: 50 000 entries, 512 columns 26.1 / 20.8, 2048 63.9 / 59.6; 100 000, 2048 114 / 104; 4096 191 / 172), and
// below kLongK columns, where the epilogue counts, 128 x 128 with two steps in LDS if there is more than a round of them (151 936, 100 rows, four steps / two: 256 columns 42.7 / 35.5, 384
// 51.1 / 43.4, 640 65.1 / 59.6, 1152 92.7 / 89.8, 1280 105.7 / 106.3, 2048 154 / 165; 32 000 entries, 512 columns 15.1 / 15.9, 1024 22.9 / 26.0).
// More rows: rounds of one workgroup per CU times what a round takes (us over 2048 columns: 256 x 256 53.5, 192 x 256 44.5, 128 x 256 33, 192 x 192 34; of other widths about the same to each
// other).  The two smaller ones are for vocabularies that the larger tiles have too few of for every CU (us, without / with them: 32 000 entries, 144 rows of 512 columns 19.9 / 18.6, 192 of
// 2048 51.1 / 44.2, 192 of 4096 87.2 / 75.5; 16 000, 192 of 2048 44.8 / 37.1).  151 936 entries, us, 256 x 256 / 192 x 256: 136 rows 186 / 170, 192 188 / 172, 256
// 188 / 226, 300 270 / 230, 384 270 / 229, 512 274 / 312, 640 373 / 418, 768 383 / 421, 1024 522 / 584.  (128 x 256: 183, 191, 194, 245, 246, 329, 388, 445, 599; 192 x 192: 175, 180, 243, 248, 253, 346, 437,
// 444, 620; 192 x 128, 192 rows 172; 256 x 192, 256 x 128 and 128 x 192 lie above the better of the two everywhere.)  With loads and reads in bursts behind the barriers (linear_tile.h): 136 rows 181, 192 185, 256 198,
// 384 263, 512 304, 768 418, 1024 560.  Whole rounds in the larger tile and the rest of the vocabulary in smaller ones is level (500 rows 273.5 / 274.9): the last round's tiles run faster by themselves.
constexpr int kLongK = 1280;
int launch_product(LmHeadParams& P, hipStream_t stream)
{
    if (P.hidden < 4 * kStepK) return launch_two_steps(P, stream);       // (128 columns)
    if (P.rows <= 64) return launch_tiles<64, 128, 3, 3>(P, stream);
    const int cus = mdx::compute_units();
    auto rounds = [&](int bm, int bn) {
        const int64_t tiles = (int64_t)((P.rows + bm - 1) / bm) * ((P.vocab + bn - 1) / bn);
        return (int)((tiles + cus - 1) / cus);
    };
    if (P.rows <= 128) {
        const int narrow = rounds(128, 128);
        if (narrow >= 2 * rounds(128, 256)) return launch_tiles<128, 256, 3, 3>(P, stream);
        return narrow > 1 && P.hidden < kLongK ? launch_tiles<128, 128, 2, 2>(P, stream) : launch_tiles<128, 128, 4, 4>(P, stream);
    }
    const float large = 53.5f * rounds(256, 256), middle = 44.5f * rounds(192, 256), half = 33.f * rounds(128, 256), square = 34.f * rounds(192, 192);
    if (half < large && half < middle && half <= square) return launch_tiles<128, 256, 3, 3>(P, stream);
    if (square < large && square < middle) return launch_tiles<192, 192, 3, 3>(P, stream);
    return middle < large ? launch_tiles<192, 256, 3, 2>(P, stream) : launch_tiles<256, 256, 3, 2>(P, stream);
}

}  // namespace

extern "C" int64_t mdx_lm_head_confidence_workspace_bytes(int64_t rows, int64_t vocab)
{
    if (rows <= 0 || vocab <= 0) return 0;
    return rows * slices_of(vocab) * (int64_t)sizeof(Record);
}

extern "C" int mdx_lm_head_confidence(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                      const float* temperatures, int32_t rows_per_temp, const int64_t* row_ids,
                                      int64_t* x0, float* x0_p,
                                      int64_t rows, int64_t vocab, int64_t hidden,
                                      void* workspace, int64_t workspace_bytes, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(rows >= 0 && vocab >= 0 && hidden >= 0, MDX_EINVAL, "lm_head_confidence: negative size");
    if (rows == 0) return MDX_OK;
    MDX_REQUIRE(vocab > 0, MDX_EINVAL, "lm_head_confidence: empty vocabulary");
    MDX_REQUIRE(x && w && x0 && x0_p, MDX_EINVAL, "lm_head_confidence: null pointer");
    MDX_REQUIRE(hidden >= 128 && hidden % 128 == 0, MDX_EUNSUPPORTED, "lm_head_confidence: hidden %lld (multiples of 128)", (long long)hidden);
    MDX_REQUIRE(rows <= 65536 && vocab < ((int64_t)1 << 24), MDX_EUNSUPPORTED,
                "lm_head_confidence: rows %lld (max 65536) or vocab %lld (below 2^24) out of range", (long long)rows, (long long)vocab);
    MDX_REQUIRE(mdx::aligned16(x) && mdx::aligned16(w) && x_row_stride % 8 == 0 && w_row_stride % 8 == 0 &&
                x_row_stride >= hidden && w_row_stride >= hidden, MDX_EUNSUPPORTED,
                "lm_head_confidence: x and W must be 16-byte aligned with row strides that are multiples of 8 elements and at least hidden");
    MDX_REQUIRE(x_row_stride * 2 * kTile < ((int64_t)1 << 31) && w_row_stride * 2 * kTile < ((int64_t)1 << 31) &&
                x_row_stride * 2 < (1 << 24) && w_row_stride * 2 < (1 << 24), MDX_EUNSUPPORTED, "lm_head_confidence: row stride too large");
    MDX_REQUIRE(!temperatures || rows_per_temp > 0, MDX_EINVAL, "lm_head_confidence: rows_per_temp must be positive");
    const int64_t need = mdx_lm_head_confidence_workspace_bytes(rows, vocab);
    MDX_REQUIRE(workspace && workspace_bytes >= need, MDX_EWORKSPACE,
                "lm_head_confidence: workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
    MDX_REQUIRE(mdx::aligned16(workspace), MDX_EWORKSPACE, "lm_head_confidence: workspace not 16-byte aligned");
    MDX_REQUIRE(need < ((int64_t)1 << 32), MDX_EUNSUPPORTED, "lm_head_confidence: too many records");

    LmHeadParams P;
    P.x = (const __bf16*)x; P.w = (const __bf16*)w; P.x_stride = x_row_stride; P.w_stride = w_row_stride;
    P.temperatures = temperatures; P.rows_per_temp = rows_per_temp; P.row_ids = row_ids;
    P.rows = (int)rows; P.vocab = (int)vocab; P.hidden = (int)hidden;
    P.n_row_tiles = P.n_vocab_tiles = P.n_slices = 0;      // with the launch
    P.records = static_cast<Record*>(workspace);
    P.x0 = x0; P.x0_p = x0_p;

    const int rc = few_rows_covered(rows, vocab, hidden) ? launch_few_rows(P, stream) : launch_product(P, stream);
    if (rc != MDX_OK) return rc;
    lm_head_finalize_kernel<<<(unsigned)((rows + kFoldThreads / 64 - 1) / (kFoldThreads / 64)), kFoldThreads, 0, stream>>>(P);
    return mdx::check_launch("lm_head_finalize");
}
