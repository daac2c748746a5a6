// Linear layers of the decoder, x . W^T for up to a few thousand rows of x: the QKV, output and down projections and the
// gate/up projection with the SiLU-and-multiply behind it (nanovllm/models/sdar.py:73-112, layers/linear.py,
// layers/activation.py:7-16).  The result is rounded to bf16, or left as fp32 partial sums over slices of K that the next
// kernel adds up (residual + RMSNorm; q/k norm + RoPE + store: they read every element once anyway).
//
// With 32 to 1500 rows the chip's 256 CUs can't all have a tile that the matrix pipe bounds (linear_tile.h); the plan below takes the
// largest tiles that still give every CU one, cutting K where that makes them larger.  Below 100 rows the read of W from HBM is
// the floor.
//
// Weights from HBM, us, here / the library's product (gate/up: with the SiLU kernel), QKV (4096 x 2048), output (2048 x 2048), gate/up
// (12288 x 2048) and down (2048 x 6144) projection:
//   rows    32    5.7   4.7  11.8   7.6 /   9.3   8.9  16.1  17.1
//   rows   128    7.8   6.0  16.0  11.7 /  12.6   9.0  20.9  17.9
//   rows   256    9.6   7.0  21.1  15.5 /  11.5   9.9  29.4  22.7
//   rows   512   12.9   9.1  27.3  21.4 /  15.7  11.3  34.8  27.6
//   rows  1024   18.7  13.1  43.6  28.1 /  20.9  15.1  53.1  41.6
//   rows  1536   25.2  16.6  67.0  40.3 /  25.8  18.3  89.3  47.1
//   rows  4096   56.5  33.2   154  80.3 /  49.8  33.2   167  81.8
//   rows  8192    106  55.6   323   140 /  93.5  49.7   337   129
//   rows 35840    485   262  1385   823 /   434   213  1501   668
// (Up to 1536 rows the better of rounded and partial sums.  Rounded where partial sums would be the faster, for a caller that doesn't take them, is slower than the library where K is long: down, whose
// chain of 96 steps few tiles share, 32 rows 25 / 17, 512 38 / 27.6, 1024 40 / 41.6: a caller that can't take partial sums
// there does better with the library.)
#include "linear_tile.h"
#include "qk_row.h"

namespace {

using namespace mdx_tile;

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
using mdx_qk::RowParams;
using mdx_qk::TokenPlace;

struct LinearParams {
    Operands in;
    __bf16* y; float* partials;                    // y: [M, N]; partials: [splits, M, N]
    int64_t y_stride;                              // elements between rows
    int k_split, splits;                           // elements of K per slice
    Places places;
    RowParams rows;                                // heads
};

// x / (1 + exp(-x)).  The division costs half of the epilogue's instructions (all eight wavefronts', with the matrix pipe idle); where nothing over- or underflows on the way, the
// quotient by the reciprocal and one correction from its exact remainder is the same but for its last place in rare cases, which the rounding to bf16
// behind it does not see.  Division / so, us: 1024 rows 45.5 / 45.2, 4096 164.7 / 162.2, 35 840 1385 / 1357;
// tiles of few rows, whose epilogue is one wait more than instructions, divide (32 rows 12.2 / 12.4).
constexpr float kTameGate = 80.f;
template <bool SHORT> __device__ __forceinline__ void silu(const float (&x)[4], float (&y)[4]) {
    const float most = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    if (SHORT && __builtin_amdgcn_ballot_w64(!(most <= kTameGate)) == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = 1.0f + __expf(-x[e]), r = __builtin_amdgcn_rcpf(d), q = x[e] * r;
            y[e] = __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-q, d, x[e]), r, q), x[e]);      // (of -0 the sums are +0)
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = x[e] / (1.0f + __expf(-x[e]));
    }
}

enum Form { kRounded = 0, kPartials = 1, kSilu = 2, kHeads = 3 };

template <typename T> constexpr int kSumsBytes = T::WK == 2 ? T::BM * T::BN * 4 : 0;      // where two wavefronts' sums meet
constexpr int kHeadPitch = mdx_qk::kHeadDim + 8;

template <typename T, int FORM>
__global__ __launch_bounds__(T::kThreads, T::kWaves / 4) void linear_kernel(const LinearParams A)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    constexpr int TM = T::TM, TN = T::TN;
    const T tile;
    const Place at = place_of(blockIdx.x + mdx::fetch_arguments<sizeof(LinearParams)>(), A.places);
    const int m0 = at.m * T::BM, n0 = at.n * T::kCols;
    // heads: a column tile is one head row of every token, eight lanes of this thread's go to a token's; its place in the rotation
    // and the cache is asked for ahead of the product
    constexpr int kTokens = T::kThreads / mdx_qk::kLanesPerRow, kPasses = FORM == kHeads ? T::BM / kTokens : 1;
    const int j8 = threadIdx.x % mdx_qk::kLanesPerRow, tok0 = m0 + (int)threadIdx.x / mdx_qk::kLanesPerRow;
    TokenPlace places[kPasses];
    mdx_qk::RowWeight weight;
    if constexpr (FORM == kHeads) {
#pragma unroll
        for (int p = 0; p < kPasses; ++p) places[p] = mdx_qk::place_of_token(A.rows, min(tok0 + p * kTokens, A.in.M - 1), j8);
        weight = mdx_qk::weight_of_row(A.rows, at.n, j8);
    }
    typename T::Sums acc;
    tile.product(A.in, m0, n0, (int64_t)at.split * A.k_split, A.k_split / kStepK, lds, acc);

    // where two wavefronts share a tile, each holds the sums over its halves of the steps, and finishes half of the rows
    constexpr int H = TM / T::WK;
    f32x4* sums = reinterpret_cast<f32x4*>(lds);             // [wave][H][TN][lane]
    if constexpr (T::WK == 2) {
        wait_loads_and_meet<0>();
        f32x4* mine = sums + tile.wave * H * TN * 64 + tile.lane;
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) mine[(i * TN + j) * 64] = tile.wk ? acc[i][j] : acc[H + i][j];
        __syncthreads();
    }
    const f32x4* theirs = sums + (tile.wave ^ (T::WM * T::WN)) * H * TN * 64 + tile.lane;
    const int mb = m0 + tile.wm * (T::BM / T::WM) + (T::WK == 2 ? tile.wk * H * 16 : 0) + tile.l16;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const int m = mb + i * 16;
        f32x4 sum[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (T::WK == 2) sum[j] = (tile.wk ? acc[H + i][j] : acc[i][j]) + theirs[(i * TN + j) * 64];
            else sum[j] = acc[i][j];
        }
        if constexpr (FORM == kHeads) {                      // the projection's rounding; rows of 128 bf16 and 16 bytes
            __bf16* row = reinterpret_cast<__bf16*>(lds + kSumsBytes<T>) + (m - m0) * kHeadPitch;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bf16x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) out[e] = (__bf16)sum[j][e];
                *reinterpret_cast<bf16x4*>(row + (tile.wn * TN + j) * 16 + 4 * tile.g) = out;
            }
            continue;
        }
        if (m >= A.in.M) continue;
        if (FORM == kSilu) {
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const int n = n0 + (tile.wn * TN + j) * 8 + 4 * tile.g;
                float gate[4], act[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) gate[e] = (float)(__bf16)sum[j][e];      // the projection's own rounding, then SiLU's
                silu<(T::BM >= 128)>(gate, act);
                bf16x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) out[e] = (__bf16)((float)(__bf16)act[e] * (float)(__bf16)sum[j + 1][e]);
                if (n < A.in.N) *reinterpret_cast<bf16x4*>(A.y + (int64_t)m * A.y_stride + n) = out;
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + (tile.wn * TN + j) * 16 + 4 * tile.g;
                if (n >= A.in.N) continue;
                if (FORM == kPartials) {
                    *reinterpret_cast<f32x4*>(A.partials + ((int64_t)at.split * A.in.M + m) * A.in.N + n) = sum[j];
                } else {
                    bf16x4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) out[e] = (__bf16)sum[j][e];
                    *reinterpret_cast<bf16x4*>(A.y + (int64_t)m * A.y_stride + n) = out;
                }
            }
        }
    }
    if constexpr (FORM == kHeads) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int tok = tok0 + p * kTokens;
            if (tok >= A.in.M) break;
            const __bf16* row = reinterpret_cast<const __bf16*>(lds + kSumsBytes<T>) + (tok - m0) * kHeadPitch;
            mdx_qk::finish_row(A.rows, tok, at.n, j8, *reinterpret_cast<const bf16x8*>(row + 8 * j8), *reinterpret_cast<const bf16x8*>(row + 64 + 8 * j8), places[p], weight);
        }
    }
}

template <int BM, int BN, int WM, int WN, int WK, int S, int SX, int FORM, bool WIDE = false>
int launch(LinearParams A, hipStream_t stream)
{
    typedef Tile<BM, BN, WM, WN, WK, S, SX, FORM == kSilu, WIDE> T;
    constexpr int kAfter = kSumsBytes<T> + (FORM == kHeads ? BM * kHeadPitch * 2 : 0), kLdsBytes = T::kStepsBytes > kAfter ? T::kStepsBytes : kAfter;
    static_assert(kLdsBytes <= 160 * 1024, "LDS");
    static_assert(FORM != kHeads || (BN == mdx_qk::kHeadDim && WK == 2 && BM % (T::kThreads / mdx_qk::kLanesPerRow) == 0), "a head per column tile");
    static std::atomic<bool> raised[64];
    const int rc = reserve_lds(reinterpret_cast<const void*>(linear_kernel<T, FORM>), kLdsBytes, raised, "linear");
    if (rc != MDX_OK) return rc;
    const int m_tiles = (A.in.M + BM - 1) / BM, n_tiles = (A.in.N + T::kCols - 1) / T::kCols;
    const int64_t grid = (int64_t)m_tiles * n_tiles * A.splits;
    MDX_REQUIRE(grid < ((int64_t)1 << 31), MDX_EUNSUPPORTED, "linear: %lld tiles", (long long)grid);
    A.places = places_of(m_tiles, n_tiles, grid);
    A.k_split /= A.splits;
    linear_kernel<T, FORM><<<(unsigned)grid, T::kThreads, kLdsBytes, stream>>>(A);
    return mdx::check_launch("linear");
}

// The tiles there are, and what a round of them costs: a step of K and what stands before and behind the steps, us, fitted to
// 1700 timings with cold weights (four projections of the decoder, 32 to 8192 rows, every tile, 1 to 32 slices of K) and held against 1486 shapes of other widths (K of 256 to 6144,
// 1024 to 12 288 columns, 16 to 1536 rows).  Small tiles that leave no room on the CU for the next round's, or share its intake with them, cost more from the second round
// on: 320 rows x 6144 x 2048 as 480 tiles of 64 x 64 with six steps 22.5 us, as 192 of 192 x 64 18.6; 160 x 6144 x 6144 as 480 of 32 x 64 42.3, as 192 of 128 x 64 35.0.
struct TileCost {
    int bm, bn, least_steps, steps_multiple;                // steps of 64 elements of K: at least, and a multiple of
    float step, around, again;                              // again: how much more every round costs where there are several
    int (*rounded)(LinearParams, hipStream_t);
    int (*partials)(LinearParams, hipStream_t);             // none for the tiles that only many rows fill
    int (*silu)(LinearParams, hipStream_t);
};
template <int BM, int BN, int WM, int WN, int WK, int S, int SX, bool PARTIALS>
constexpr TileCost tile(float step, float around, float again = 1.f) {
    typedef Tile<BM, BN, WM, WN, WK, S, SX, false> T;
    // (a slice has four steps at least: rows that are too far apart for the plan's tile go to one that loads four ahead, run_partials)
    if constexpr (PARTIALS) return TileCost{BM, BN, T::kLeastSteps < 4 ? 4 : T::kLeastSteps, T::kStepsMultiple, step, around, again, launch<BM, BN, WM, WN, WK, S, SX, kRounded>,
                                            launch<BM, BN, WM, WN, WK, S, SX, kPartials>, launch<BM, BN, WM, WN, WK, S, SX, kSilu>};
    else return TileCost{BM, BN, T::kLeastSteps, T::kStepsMultiple, step, around, again, launch<BM, BN, WM, WN, WK, S, SX, kRounded>, nullptr,
                         launch<BM, BN, WM, WN, WK, S, SX, kSilu>};
}
const TileCost kTiles[] = {
    // The two smallest hold four steps in LDS or six.  Six are the faster where a slice has as many and W comes from HBM (us, four / six: gate/up of 32 rows 12.66 / 12.30, down 8.33 / 8.05,
    // QKV of 96 rows in two slices 8.52 / 8.02; W from the memory-side cache, 512 columns of K, 3.7 / 3.8), but K of 256, and K cut into slices of four steps, would go to larger tiles without four:
    // 32 rows x 1024 x 256 3.1 / 4.1, 128 rows 3.1 / 4.8.  Slices of four steps are for few sums: with the norm behind them, us, half as many with six / so: 32 rows x 1024 x 1024 6.50 / 6.06, x 2048
    // 6.65 / 6.39, 16 rows less; but 32 rows x 2048 x 2048 7.98 / 8.15, 64 rows 8.42 / 9.39 (the first tile's 0.7).
    tile<32, 64, 2, 2, 1, 4, 4, true>(0.173f, 0.7f, 1.04f),
    tile<32, 64, 2, 2, 1, 6, 6, true>(0.165f, 0.4f, 1.1f),
    tile<64, 64, 2, 2, 2, 4, 4, true>(0.233f, 0.7f),
    tile<64, 64, 2, 2, 2, 6, 6, true>(0.223f, 0.7f, 1.1f),
    tile<128, 64, 2, 2, 2, 4, 4, true>(0.326f, 1.7f),
    tile<192, 64, 2, 2, 2, 4, 4, true>(0.408f, 2.9f),
    tile<128, 128, 2, 2, 2, 4, 4, true>(0.487f, 2.6f),
    tile<192, 128, 2, 2, 2, 4, 4, true>(0.584f, 3.5f),
    tile<128, 192, 4, 2, 1, 4, 4, true>(0.617f, 2.3f),
    tile<192, 192, 4, 2, 1, 3, 3, false>(0.741f, 5.0f),
    tile<256, 128, 4, 2, 1, 3, 3, true>(0.60f, 4.5f),        // slices of long K: 1024 x 2048 x 6144 and the norm behind it 40.0 us as two of 128 x 128 tiles, 37.9 as four
    tile<256, 192, 4, 2, 1, 3, 2, false>(0.983f, 3.7f),
    tile<256, 256, 4, 2, 1, 3, 2, false>(1.149f, 5.9f),
};

struct Plan { const TileCost* tile; int splits; double cost; };

// The cheapest tile and number of slices by the costs above, in rounds of one workgroup per CU (the small tiles' second one
// per CU is worth little: they share its intake).  Partial sums cost their writing and the next kernel's reading, 0.35 us per
// MB together (5.7 TB/s), a rounded result less than half of that per element.  Against the best of all timed choices this
// costs 0.3 % on average and 4 % at most at the decoder's widths, 0.6 % on average and 16 % at most at the others.
Plan plan_of(int64_t rows, int64_t n, int64_t k, bool rounded, bool partials, bool silu)
{
    Plan best{nullptr, 0, 0};
    const int cus = mdx::compute_units();
    const double mb = (double)rows * (double)n * 4e-6;
    for (const TileCost& t : kTiles) {
        const int64_t cols = silu ? t.bn / 2 : t.bn, tiles = ((rows + t.bm - 1) / t.bm) * ((n + cols - 1) / cols);
        for (int64_t s = 1; s <= k / (kStepK * t.least_steps) && s <= 32; ++s) {
            if (k % (kStepK * t.steps_multiple * s) != 0 || (s > 1 && !partials)) continue;
            const double steps = (double)(k / kStepK / s), rounds = (double)((tiles * s + cus - 1) / cus);
            for (int form = 0; form < 2; ++form) {                                  // 0: rounded or SiLU, 1: partial sums
                if (form == 0 ? (s > 1 || !(rounded || silu)) : (!partials || !t.partials)) continue;
                const double cost = rounds * (steps * t.step + t.around) * (rounds > 1 ? t.again : 1.f) + (form ? 0.35 * (double)s : 0.15) * mb;
                if (!best.tile || cost < best.cost) best = Plan{&t, form ? (int)s : 0, cost};
            }
        }
    }
    return best;                                                                    // splits 0: not partial sums
}

// The QKV projection with what follows it: tiles of one head, by the same costs.  Two launches / one, us per decoder layer: 160 rows
// 85.6 / 87.5, 256 94.5 / 96.4, 384 117.9 / 115.5, 512 124.1 / 121.3, 768 153.0 / 150.8, 1024 179.6 / 176.5, 1504 241.5 / 238.4.
struct HeadsPlan { int (*run)(LinearParams, hipStream_t); float cost; };
HeadsPlan heads_plan(int64_t rows, int64_t n, int64_t k)
{
    const int cus = mdx::compute_units();
    auto cost = [&](int bm, float step, float around) {
        const int64_t tiles = (rows + bm - 1) / bm * (n / mdx_qk::kHeadDim);
        return (float)((tiles + cus - 1) / cus) * ((float)(k / kStepK) * step + around);
    };
    const float c64 = cost(64, 0.338f, 1.7f), c128 = cost(128, 0.487f, 2.6f), c192 = cost(192, 0.584f, 3.5f);
    if (c64 <= c128 && c64 <= c192) return {launch<64, 128, 2, 2, 2, 4, 4, kHeads>, c64};
    if (c128 <= c192) return {launch<128, 128, 2, 2, 2, 4, 4, kHeads>, c128};
    return {launch<192, 128, 2, 2, 2, 4, 4, kHeads>, c192};
}

constexpr int64_t kSizeLimit = (int64_t)1 << 28;

bool sizes_covered(int64_t rows, int64_t n, int64_t k)
{
    return rows > 0 && rows < kSizeLimit && n > 0 && n % 8 == 0 && n < kSizeLimit && k >= 256 && k % 128 == 0 && k < kSizeLimit;
}

bool narrow(int64_t x_row_stride, int64_t w_row_stride) { return x_row_stride < kNarrowStride && w_row_stride < kNarrowStride; }

// any_stride: the two mdx_decode_linear_* calls, which have always taken rows however far apart
int check_linear(const char* what, bool any_stride, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, const void* out,
                 int64_t rows, int64_t n, int64_t k)
{
    MDX_REQUIRE(rows >= 0 && n >= 0 && k >= 0, MDX_EINVAL, "%s: negative size", what);
    MDX_REQUIRE(x && w && out, MDX_EINVAL, "%s: null pointer", what);
    MDX_REQUIRE(mdx::aligned16(x) && mdx::aligned16(w) && mdx::aligned16(out) && x_row_stride % 8 == 0 && w_row_stride % 8 == 0 &&
                x_row_stride >= k && w_row_stride >= k, MDX_EUNSUPPORTED,
                "%s: x, W and the result must be 16-byte aligned, row strides multiples of 8 elements and at least k", what);
    MDX_REQUIRE(any_stride || narrow(x_row_stride, w_row_stride), MDX_EUNSUPPORTED, "%s: row strides %lld and %lld (below %lld elements)", what,
                (long long)x_row_stride, (long long)w_row_stride, (long long)kNarrowStride);
    return MDX_OK;
}

LinearParams params_of(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int64_t rows, int64_t n, int64_t k)
{
    LinearParams A{};
    A.in = Operands{(const __bf16*)x, (const __bf16*)w, x_row_stride, w_row_stride, (int)rows, (int)n};
    A.k_split = (int)k; A.splits = 1;
    return A;
}

int run_partials(const char* what, bool any_stride, const Plan& plan, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, float* partials,
                 int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const int rc = check_linear(what, any_stride, x, x_row_stride, w, w_row_stride, partials, rows, n, k);
    if (rc != MDX_OK) return rc;
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.partials = partials;
    A.splits = plan.splits;
    if (!narrow(x_row_stride, w_row_stride)) return launch<32, 64, 2, 2, 1, 4, 4, kPartials, true>(A, static_cast<hipStream_t>(stream));
    return plan.tile->partials(A, static_cast<hipStream_t>(stream));
}

int run_rows(const char* what, bool any_stride, bool silu, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, void* y, int64_t y_row_stride,
             int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const int rc = check_linear(what, any_stride, x, x_row_stride, w, w_row_stride, y, rows, n, k);
    if (rc != MDX_OK) return rc;
    MDX_REQUIRE(y_row_stride % 4 == 0 && y_row_stride >= n, MDX_EUNSUPPORTED, "%s: row stride of y (a multiple of 4, at least n)", what);
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.y = (__bf16*)y;
    A.y_stride = y_row_stride;
    if (silu && !narrow(x_row_stride, w_row_stride)) return launch<32, 64, 2, 2, 1, 4, 4, kSilu, true>(A, static_cast<hipStream_t>(stream));
    const Plan plan = plan_of(rows, n, k, !silu, false, silu);
    return (silu ? plan.tile->silu : plan.tile->rounded)(A, static_cast<hipStream_t>(stream));
}

// Where the kernel is the better one (table at the top of this file): up to 1536 rows; with the SiLU in the epilogue, which
// saves writing and reading twice the result, up to 8192, and beyond where W is wide.  Other widths, us, here / library's product: 5120 x 5120, 1024 rows (54 GFLOP) 58.1 / 61.1, 1280 77.1 / 71.7;
// 7168 x 5120, 512 (38) 51.3 / 49.4, 1280 (94) 101 / 85; 8192 x 8192, 384 (52) 59.6 / 64.3, 768 (103) 94.4 / 97.4, 1024 (137) 141 / 116; 6144 x 4096, 1024 (52) 52.5 / 51.7, 1280 (64)
// 68.2 / 57.3: from 52 GFLOP on the library's tiles come to their rate.  Where K is long beside n they do not: 5120 x 17408, 1024 rows (183) 173 / 244, 4096 x 12288, 768 (77) 77 / 90.
// Beyond 8192 rows it is where W's halves are no narrower than K and 1024 (n x k, here / library's product and SiLU, us): 35 840 rows, 6144 x 2048 1410 / 1494, 1024 x 512
// 102 / 166, 3072 x 1024 428 / 486, 8960 x 1536 1600 / 1819, 8192 x 3072 2608 / 2676, 12288 x 4096 5205 / 5281; 16 384 rows, 17408 x 5120 4000 / 4466; but 2048 x 8192 787 / 741.
constexpr int64_t kMaxRows = 1536, kMaxSiluRows = 8192, kLeastSiluWidth = 1024;
bool silu_pays(int64_t rows, int64_t n, int64_t k) { return rows <= kMaxSiluRows || (n >= kLeastSiluWidth && n >= k); }
constexpr double kMaxWork = 52e9;
bool linear_pays(int64_t rows, int64_t n, int64_t k) { return rows <= kMaxRows && (2.0 * (double)rows * (double)n * (double)k <= kMaxWork || k >= 3 * n); }
// With the head rows finished in the epilogue (heads_plan): from where tiles of 128 columns are enough to fill most CUs; fewer rows
// are bound by what a CU takes in, and the product in narrower tiles or slices of K with a second launch is the faster.  So it is where these tiles cost more
// than the product's own plan by what the second launch takes (2.5 us by the costs above): 32 heads on 8, one launch / two, us: 2560 columns of K, 768 rows 39.2 / 43.1, 1024 (tiles
// for a round and a half) 59.7 / 46.1; 4096, 640 rows 42.2 / 46.9, 1024 77.0 / 59.6; 64 on 8, 8192, 512 rows 91 / 95, 640 143 / 123; 16 on 2, 2048, 384 rows 17.7 / 16.0, 512 17.6 / 21.1.
constexpr int64_t kMinHeadRows = 384;
constexpr double kSecondLaunch = 2.5;
bool heads_covered(int64_t rows, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int64_t k)
{
    return num_q_heads > 0 && num_kv_heads > 0 && head_dim == mdx_qk::kHeadDim && rows >= kMinHeadRows && rows <= kMaxRows &&
           sizes_covered(rows, ((int64_t)num_q_heads + 2 * (int64_t)num_kv_heads) * head_dim, k);
}
constexpr int64_t kMaxDecodeRows = 128, kMaxDecodeSiluRows = 64, kDecodeSizeLimit = (int64_t)1 << 30;

Plan decode_plan(int64_t rows, int64_t n, int64_t k)
{
    if (rows <= 0 || rows > kMaxDecodeRows || n <= 0 || n % 64 != 0 || n >= kDecodeSizeLimit || k <= 0 || k % 256 != 0 || k >= kDecodeSizeLimit) return Plan{nullptr, 0, 0};
    return plan_of(rows, n, k, false, true, false);
}

}  // namespace

extern "C" int32_t mdx_linear_splits(int64_t rows, int64_t n, int64_t k)
{
    if (!sizes_covered(rows, n, k) || !linear_pays(rows, n, k)) return -1;
    return plan_of(rows, n, k, true, true, false).splits;
}

extern "C" int mdx_linear(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                          void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(sizes_covered(rows, n, k), MDX_EUNSUPPORTED, "linear: %lld rows, n %lld (a multiple of 8), k %lld (a multiple of 128, at least 256)",
                (long long)rows, (long long)n, (long long)k);
    return run_rows("linear", false, false, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}

extern "C" int mdx_linear_partials(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                   float* partials, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    Plan plan{nullptr, 0, 0};
    if (sizes_covered(rows, n, k) && rows <= kMaxRows) plan = plan_of(rows, n, k, true, true, false);
    MDX_REQUIRE(plan.splits > 0, MDX_EUNSUPPORTED, "linear_partials: %lld rows, n %lld, k %lld are not cut along k", (long long)rows, (long long)n, (long long)k);
    return run_partials("linear_partials", false, plan, x, x_row_stride, w, w_row_stride, partials, rows, n, k, stream);
}

extern "C" int32_t mdx_linear_silu_supported(int64_t rows, int64_t n, int64_t k) { return sizes_covered(rows, n, k) && silu_pays(rows, n, k); }

extern "C" int mdx_linear_silu(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                               void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(sizes_covered(rows, n, k), MDX_EUNSUPPORTED, "linear_silu: %lld rows, n %lld (a multiple of 8), k %lld (a multiple of 128, at least 256)",
                (long long)rows, (long long)n, (long long)k);
    return run_rows("linear_silu", false, true, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}

extern "C" int32_t mdx_linear_qk_norm_rope_store_supported(int64_t rows, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int64_t k)
{
    if (!heads_covered(rows, num_q_heads, num_kv_heads, head_dim, k)) return 0;
    const int64_t n = ((int64_t)num_q_heads + 2 * (int64_t)num_kv_heads) * head_dim;
    return heads_plan(rows, n, k).cost <= plan_of(rows, n, k, true, true, false).cost + kSecondLaunch;
}

extern "C" int mdx_linear_qk_norm_rope_store(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                             const void* q_weight, const void* k_weight, float eps,
                                             const float* cos_table, const float* sin_table, int64_t max_positions, const int64_t* positions,
                                             void* q_out, int64_t q_out_row_stride, void* k_out, int64_t k_out_row_stride,
                                             void* v_out, int64_t v_out_row_stride,
                                             void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_slots,
                                             int64_t rows, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int64_t k, mdx_stream_t stream)
{
    const char* what = "linear_qk_norm_rope_store";
    MDX_REQUIRE(heads_covered(rows, num_q_heads, num_kv_heads, head_dim, k), MDX_EUNSUPPORTED,
                "%s: %lld rows (%lld to %lld), head_dim %d (only %d), k %lld (a multiple of 128, at least 256)", what, (long long)rows,
                (long long)kMinHeadRows, (long long)kMaxRows, head_dim, mdx_qk::kHeadDim, (long long)k);
    const int64_t n = ((int64_t)num_q_heads + 2 * (int64_t)num_kv_heads) * head_dim;
    const int rc = check_linear(what, false, x, x_row_stride, w, w_row_stride, q_out, rows, n, k);
    if (rc != MDX_OK) return rc;
    MDX_REQUIRE(q_weight && k_weight && cos_table && sin_table && positions, MDX_EINVAL, "%s: null pointer", what);
    MDX_REQUIRE((k_cache == nullptr) == (v_cache == nullptr), MDX_EINVAL, "%s: give both caches or neither", what);
    MDX_REQUIRE(!k_cache || slot_mapping, MDX_EINVAL, "%s: caches without slot_mapping", what);
    MDX_REQUIRE(mdx::aligned16(q_weight) && mdx::aligned16(k_weight) && mdx::aligned16(k_out) && mdx::aligned16(v_out) &&
                mdx::aligned16(k_cache) && mdx::aligned16(v_cache) && q_out_row_stride % 8 == 0 && k_out_row_stride % 8 == 0 && v_out_row_stride % 8 == 0,
                MDX_EUNSUPPORTED, "%s: tensors must be 16-byte aligned with row strides that are multiples of 8", what);
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.rows = RowParams{(const __bf16*)q_weight, (const __bf16*)k_weight, eps, cos_table, sin_table, max_positions, positions,
                       (__bf16*)q_out, q_out_row_stride, (__bf16*)k_out, k_out_row_stride, (__bf16*)v_out, v_out_row_stride,
                       (__bf16*)k_cache, (__bf16*)v_cache, slot_mapping, num_slots, num_q_heads, num_kv_heads};
    return heads_plan(rows, n, k).run(A, static_cast<hipStream_t>(stream));
}

extern "C" int32_t mdx_decode_linear_splits(int64_t rows, int64_t n, int64_t k) { return decode_plan(rows, n, k).splits; }

extern "C" int mdx_decode_linear_partials(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                          float* partials, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const Plan plan = decode_plan(rows, n, k);
    MDX_REQUIRE(plan.tile, MDX_EUNSUPPORTED, "decode_linear: %lld rows (up to %lld), n %lld (a multiple of 64), k %lld (a multiple of 256)",
                (long long)rows, (long long)kMaxDecodeRows, (long long)n, (long long)k);
    return run_partials("decode_linear", true, plan, x, x_row_stride, w, w_row_stride, partials, rows, n, k, stream);
}

extern "C" int32_t mdx_decode_linear_silu_supported(int64_t rows, int64_t n, int64_t k)
{
    return rows > 0 && rows <= kMaxDecodeSiluRows && n > 0 && n % 24 == 0 && n < kDecodeSizeLimit / 2 && k > 0 && k % 512 == 0 && k < kDecodeSizeLimit;
}

extern "C" int mdx_decode_linear_silu(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                      void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(mdx_decode_linear_silu_supported(rows, n, k), MDX_EUNSUPPORTED,
                "decode_linear_silu: %lld rows (up to %lld), n %lld (a multiple of 24), k %lld (a multiple of 512)", (long long)rows,
                (long long)kMaxDecodeSiluRows, (long long)n, (long long)k);
    return run_rows("decode_linear_silu", true, true, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}
