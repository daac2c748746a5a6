// Linear layers of the decoder, x . W^T for up to a few thousand rows of x: the QKV, output and down projections and the
// gate/up projection with the SiLU-and-multiply behind it (nanovllm/models/sdar.py:73-112, layers/linear.py,
// layers/activation.py:7-16).  The result is rounded to bf16, or left as fp32 partial sums over slices of K that the next
// kernel adds up (residual + RMSNorm; q/k norm + RoPE + store: they read every element once anyway).
//
// What bounds it.  A CU takes in at most 70 GB/s from its XCD's L2 (8 wavefronts, loads to LDS, whatever is in flight; 59
// with 4, 78 with 16), all of them 18 TB/s, so a tile of BM x BN costs (BM + BN) x 128 bytes per step of 64 elements of K
// against BM x BN x 128 operations, and only tiles of about 256 x 256 are bound by the matrix pipe (1.3 PFLOP/s of them under
// the board's power limit).  With 32 to 1500 rows the chip's 256 CUs can't all have such a tile; the plan below takes the
// largest tiles that still give every CU one, cutting K where that makes them larger.  Below 100 rows the read of W from HBM
// is the floor.  From timing builds at 2048 rows, down projection, tiles of 128 x 128, us: whole 60, loads alone 58, without
// loads 40, matrix instructions alone 34, LDS reads alone 23.
//
// The kernel:
//  * S steps of x and W rows in LDS (128 bytes of a row per step), filled by loads that pass by the registers
//    (global_load_lds); the 16-byte chunk c of row r sits at c ^ (r / 2 % 8), so that the 16 rows of a fragment read cover all
//    banks once.  One barrier per step: behind it the next step is in LDS for everybody and nobody reads this one any more.
//  * the fragments of the next half step are on their way from LDS while this one is multiplied (two register sets).
//  * small and middle tiles are shared by two groups of four wavefronts, each taking one half of every step (WK = 2): tiles
//    of (BM / 2) x (BN / 2) per wavefront need half of the LDS reads that eight tiles of half the size would, and the two
//    wavefronts of a SIMD cover each other's waits.  The sums meet in LDS at the end.
//  * W is the first operand, so that a lane ends with four consecutive columns of one row.
//
// Cold weights, us, here / the library's product (gate/up: with the SiLU kernel), QKV (4096 x 2048), output (2048 x 2048), gate/up
// (12288 x 2048) and down (2048 x 6144) projection:
//   rows    32   4.8  3.8  12.4   7.1 /  11.7  8.4  18.8 16.6      (a kernel with W straight in registers: 6.5  4.6 15.2  8.6)
//   rows   128   6.9  5.0  18.4  10.8 /  12.1  8.6  22.0 17.8      (                                      10.0  6.8 23.7 12.5)
//   rows   256   9.0  6.3  24.0  15.1 /  11.3  9.7  31.1 22.5
//   rows   512  12.5  8.6  28.7  20.7 /  15.2 11.1  35.9 27.7
//   rows  1024  19.3 12.7  46.1  33.2 /  20.9 15.1  54.4 40.6
//   rows  1536  27.2 16.8  81.0  40.8 /  26.2 18.3  94.1 46.7
//   rows  4096  56.8 33.3 167.6 101.4 /  48.8 31.6 178.6 87.4
//   rows 16384 225  110   679   296   / 187   94.5 669  268
// Touching lines of W and x ahead of their loads (as the vocabulary head does), starting the workgroups at different steps, other
// bands of tiles per XCD and six steps in LDS instead of four change nothing or cost 1 us.
#include "mdx_common.h"
#include <atomic>
#include <utility>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) char lds_char;

struct LinearParams {
    const __bf16* x; const __bf16* w;
    __bf16* y; float* partials;                    // y: [M, N]; partials: [splits, M, N]
    int64_t x_stride, w_stride, y_stride;          // elements between rows
    int M, N, K;                                   // N: columns of the result (SiLU: W has 2 N rows, gate then up)
    int m_tiles, n_tiles, splits;
};

enum Form { kRounded = 0, kPartials = 1, kSilu = 2 };

constexpr int kStepK = 64, kRowBytes = 2 * kStepK; // one step of K: 128 bytes of every row
constexpr int kBand = 8;                           // row tiles that share a column tile of W one after the other

template <typename F, int... J>
__device__ __forceinline__ void for_each(F f, std::integer_sequence<int, J...>) { (f(std::integral_constant<int, J>{}), ...); }

// This wavefront's loads up to the newest N and all of its LDS reads are done, then everybody's.
template <int N> __device__ __forceinline__ void wait_loads_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <int BM, int BN, int WM, int WN, int WK, int S, int FORM>
__global__ __launch_bounds__(64 * WM * WN * WK, WM * WN * WK / 4) void linear_kernel(const LinearParams A)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    constexpr int kWaves = WM * WN * WK;
    constexpr int TM = BM / (16 * WM), TN = BN / (16 * WN);  // a wavefront's share, in matrix tiles of 16 x 16
    constexpr int kStage = (BM + BN) * kRowBytes, kLoads = (BM + BN) / 8 / kWaves;
    static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0 && (WK == 1 || (WK == 2 && TM % 2 == 0)), "tile shape");
    static_assert((FORM != kSilu || TN % 2 == 0) && S % 2 == 0, "pairs of gate and up tiles, pairs of steps");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);

    // Consecutive workgroups go to the eight XCDs in turn; each XCD takes a run of the tiles in the order (slice of K, band of
    // row tiles, column tile, row tile): what it has in flight together shares its rows of x and of W in its L2.
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3, more = gridDim.x & 7;
    int at = xcd * per_xcd + min(xcd, more) + (int)(blockIdx.x >> 3);
    const int per_split = A.m_tiles * A.n_tiles, split = at / per_split;
    at -= split * per_split;
    const int m_first = at / (kBand * A.n_tiles) * kBand, m_band = min(kBand, A.m_tiles - m_first);
    at -= m_first * A.n_tiles;
    constexpr int kCols = FORM == kSilu ? BN / 2 : BN;      // columns of the result
    const int m0 = (m_first + at % m_band) * BM, n0 = at / m_band * kCols;
    const int k_split = A.K / A.splits, n_steps = k_split / kStepK;         // (the host's choice: an even number, at least S)

    // Load i of this wavefront fills 8 rows of the tile, x rows first, then rows of W (SiLU: 16 gate rows, the 16 up rows of
    // the same columns, and so on).  Rows beyond the last are the last one again; their products are not stored.
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
    const char* base[kLoads];                               // the first of the 8 rows, at this slice of K
    unsigned offset[kLoads];                                // this lane's row and chunk from there
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r0 = 8 * (wave + kWaves * i), r = lane >> 3, chunk = (lane & 7) ^ (((r0 + r) >> 1) & 7);
        const bool of_x = r0 < BM;                          // (known when compiled: BM is a multiple of 8 kWaves)
        const int b = r0 - BM;
        const int first = of_x ? m0 + r0 : FORM == kSilu ? n0 + (b >> 5) * 16 + (b & 15) : n0 + b, last = (of_x ? A.M : A.N) - 1;
        const int64_t stride = (of_x ? A.x_stride : A.w_stride) * 2;
        const int64_t up = FORM == kSilu && !of_x && ((b >> 4) & 1) ? A.N : 0;
        base[i] = reinterpret_cast<const char*>((of_x ? A.x : A.w) + split * k_split) + (min(first, last) + up) * stride;
        offset[i] = (unsigned)(min(first + r, last) - min(first, last)) * (unsigned)stride + chunk * 16;
    }
    int64_t k_bytes = 0;                                    // where the step to ask for next begins
    auto issue = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :: "s"(lds0 + buf * kStage + (wave + kWaves * i) * 1024), "v"(offset[i]), "s"(base[i] + k_bytes) : "memory");
        k_bytes += kRowBytes;
    };
    const char* xr = lds + (wm * (BM / WM) + l16) * kRowBytes;
    const char* wr = lds + (BM + wn * (BN / WN) + l16) * kRowBytes;
    bf16x8 fx[2][TM], fw[2][TN];
    auto read = [&](int set, int buf, int half) {            // a half of a step: 32 elements of K
        const int pos = ((half * 4 + g) ^ ((l16 >> 1) & 7)) * 16 + buf * kStage;
#pragma unroll
        for (int i = 0; i < TM; ++i) fx[set][i] = *reinterpret_cast<const bf16x8*>(xr + pos + i * 16 * kRowBytes);
#pragma unroll
        for (int i = 0; i < TN; ++i) fw[set][i] = *reinterpret_cast<const bf16x8*>(wr + pos + i * 16 * kRowBytes);
    };
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int half) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[half][j], fx[half][i], acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (int s = 0; s < S; ++s) issue(s);
    wait_loads_and_meet<(S - 1) * kLoads>();
    read(0, 0, WK == 2 ? wk : 0);
    int buf = 0;                                             // t % S
    auto next = [&](int b) { return b + 1 == S ? 0 : b + 1; };
    for (int t = 0; t < n_steps - S; t += 2) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (WK == 1) { read(1, buf, 1); multiply(0); }
            wait_loads_and_meet<(S - 2) * kLoads>();
            issue(buf);
            buf = next(buf);
            if constexpr (WK == 1) { read(0, buf, 0); multiply(1); }
            else { read(1 - h, buf, wk); multiply(h); }
        }
    }
    // the last S steps: nothing more to load
    for_each([&](auto step) {
        constexpr int J = decltype(step)::value;
        if constexpr (WK == 1) { read(1, buf, 1); multiply(0); }
        if constexpr (J + 1 < S) {
            wait_loads_and_meet<(S - 2 - J) * kLoads>();
            buf = next(buf);
            if constexpr (WK == 1) read(0, buf, 0); else read(1 - (J & 1), buf, wk);
        }
        if constexpr (WK == 1) multiply(1); else multiply(J & 1);
    }, std::make_integer_sequence<int, S>{});

    // where two wavefronts share a tile, each holds the sums over its halves of the steps, and finishes half of the rows
    constexpr int H = TM / WK;
    f32x4* sums = reinterpret_cast<f32x4*>(lds);             // [wave][H][TN][lane]
    if constexpr (WK == 2) {
        wait_loads_and_meet<0>();
        f32x4* mine = sums + wave * H * TN * 64 + lane;
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) mine[(i * TN + j) * 64] = wk ? acc[i][j] : acc[H + i][j];
        __syncthreads();
    }
    const f32x4* theirs = sums + (wave ^ (WM * WN)) * H * TN * 64 + lane;
    const int mb = m0 + wm * (BM / WM) + (WK == 2 ? wk * H * 16 : 0) + l16;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const int m = mb + i * 16;
        f32x4 sum[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (WK == 2) sum[j] = (wk ? acc[H + i][j] : acc[i][j]) + theirs[(i * TN + j) * 64];
            else sum[j] = acc[i][j];
        }
        if (m >= A.M) continue;
        if (FORM == kSilu) {
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const int n = n0 + (wn * TN + j) * 8 + 4 * g;
                bf16x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gate = (float)(__bf16)sum[j][e];      // the projection's own rounding, then SiLU's
                    out[e] = (__bf16)((float)(__bf16)(gate / (1.0f + __expf(-gate))) * (float)(__bf16)sum[j + 1][e]);
                }
                if (n < A.N) *reinterpret_cast<bf16x4*>(A.y + (int64_t)m * A.y_stride + n) = out;
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + (wn * TN + j) * 16 + 4 * g;
                if (n >= A.N) continue;
                if (FORM == kPartials) {
                    *reinterpret_cast<f32x4*>(A.partials + ((int64_t)split * A.M + m) * A.N + n) = sum[j];
                } else {
                    bf16x4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) out[e] = (__bf16)sum[j][e];
                    *reinterpret_cast<bf16x4*>(A.y + (int64_t)m * A.y_stride + n) = out;
                }
            }
        }
    }
}

template <int BM, int BN, int WM, int WN, int WK, int S, int FORM>
int launch(LinearParams A, hipStream_t stream)
{
    constexpr int kTiles = S * (BM + BN) * kRowBytes, kSums = WK == 2 ? BM * BN * 4 : 0, kLdsBytes = kTiles > kSums ? kTiles : kSums;
    static_assert(kLdsBytes <= 160 * 1024, "LDS");
    if (kLdsBytes > 65536) {
        // the kernel's LDS limit is raised once per device
        static std::atomic<bool> raised[64];
        int device = 0;
        hipError_t e = hipGetDevice(&device);
        MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "linear: no current device (%s)", hipGetErrorString(e));
        if (!raised[device].load(std::memory_order_acquire)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(linear_kernel<BM, BN, WM, WN, WK, S, FORM>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
            MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "linear: cannot reserve %d bytes of LDS (%s)", kLdsBytes, hipGetErrorString(e));
            raised[device].store(true, std::memory_order_release);
        }
    }
    constexpr int kCols = FORM == kSilu ? BN / 2 : BN;
    A.m_tiles = (A.M + BM - 1) / BM;
    A.n_tiles = (A.N + kCols - 1) / kCols;
    const int64_t grid = (int64_t)A.m_tiles * A.n_tiles * A.splits;
    MDX_REQUIRE(grid < ((int64_t)1 << 31), MDX_EUNSUPPORTED, "linear: %lld tiles", (long long)grid);
    linear_kernel<BM, BN, WM, WN, WK, S, FORM><<<(unsigned)grid, 64 * WM * WN * WK, kLdsBytes, stream>>>(A);
    return mdx::check_launch("linear");
}

// The tiles there are, and what a round of them costs: a step of K and what stands before and behind the steps, us, fitted to
// 4900 timings (four projections of the decoder, 16 to 8192 rows, every tile, 1 to 24 slices of K).
struct Tile {
    int bm, bn, stages;
    float step, around;
    int (*rounded)(LinearParams, hipStream_t);
    int (*partials)(LinearParams, hipStream_t);             // none for the tiles that only many rows fill
    int (*silu)(LinearParams, hipStream_t);
};
#define MDX_TILE(BM, BN, WM, WN, WK, S) launch<BM, BN, WM, WN, WK, S, kRounded>, launch<BM, BN, WM, WN, WK, S, kPartials>, launch<BM, BN, WM, WN, WK, S, kSilu>
#define MDX_LARGE_TILE(BM, BN, WM, WN, WK, S) launch<BM, BN, WM, WN, WK, S, kRounded>, nullptr, launch<BM, BN, WM, WN, WK, S, kSilu>
const Tile kTileTable[] = {
    {32, 64, 4, 0.150f, 0.2f, MDX_TILE(32, 64, 2, 2, 1, 4)},
    {64, 64, 4, 0.200f, 0.5f, MDX_TILE(64, 64, 2, 2, 2, 4)},
    {128, 64, 4, 0.302f, 1.3f, MDX_TILE(128, 64, 2, 2, 2, 4)},
    {192, 64, 4, 0.395f, 1.6f, MDX_TILE(192, 64, 2, 2, 2, 4)},
    {128, 128, 4, 0.470f, 1.8f, MDX_TILE(128, 128, 2, 2, 2, 4)},
    {192, 128, 4, 0.606f, 2.6f, MDX_TILE(192, 128, 2, 2, 2, 4)},
    {128, 192, 4, 0.677f, 1.5f, MDX_TILE(128, 192, 4, 2, 1, 4)},
    {256, 192, 2, 1.166f, 1.2f, MDX_LARGE_TILE(256, 192, 4, 2, 1, 2)},
    {256, 256, 2, 1.432f, 1.3f, MDX_LARGE_TILE(256, 256, 2, 4, 1, 2)},
};
#undef MDX_TILE
#undef MDX_LARGE_TILE

struct Plan { const Tile* tile; int splits; };

// The cheapest tile and number of slices by the costs above, in rounds of one workgroup per CU (the small tiles' second one
// per CU is worth little: they share its intake).  Partial sums cost their writing and the next kernel's reading, 0.35 us per
// MB together (5.7 TB/s), a rounded result a quarter of that per element.  Against the best of all timed choices this
// costs 1 % on average and 10 % at most.
Plan plan_of(int64_t rows, int64_t n, int64_t k, bool rounded, bool partials, bool silu)
{
    Plan best{nullptr, 0};
    double least = 0;
    const int cus = mdx::compute_units();
    const double mb = (double)rows * (double)n * 4e-6;
    for (const Tile& t : kTileTable) {
        const int64_t cols = silu ? t.bn / 2 : t.bn, tiles = ((rows + t.bm - 1) / t.bm) * ((n + cols - 1) / cols);
        for (int64_t s = 1; s <= k / (kStepK * t.stages) && s <= 32; ++s) {
            if (k % (2 * kStepK * s) != 0 || (s > 1 && !partials)) continue;      // whole pairs of steps
            const double steps = (double)(k / kStepK / s), rounds = (double)((tiles * s + cus - 1) / cus);
            for (int form = 0; form < 2; ++form) {                                  // 0: rounded or SiLU, 1: partial sums
                if (form == 0 ? (s > 1 || !(rounded || silu)) : (!partials || !t.partials)) continue;
                const double cost = 2.0 + rounds * (steps * t.step + t.around) + (form ? 0.35 * (double)s : 0.09) * mb;
                if (!best.tile || cost < least) { best = Plan{&t, form ? (int)s : 0}; least = cost; }
            }
        }
    }
    return best;                                                                    // splits 0: not partial sums
}

constexpr int64_t kSizeLimit = (int64_t)1 << 28;

bool sizes_covered(int64_t rows, int64_t n, int64_t k)
{
    return rows > 0 && rows < kSizeLimit && n > 0 && n % 8 == 0 && n < kSizeLimit && k >= 256 && k % 128 == 0 && k < kSizeLimit;
}

int check_linear(const char* what, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, const void* out, int64_t rows, int64_t n, int64_t k)
{
    MDX_REQUIRE(rows >= 0 && n >= 0 && k >= 0, MDX_EINVAL, "%s: negative size", what);
    MDX_REQUIRE(x && w && out, MDX_EINVAL, "%s: null pointer", what);
    MDX_REQUIRE(mdx::aligned16(x) && mdx::aligned16(w) && mdx::aligned16(out) && x_row_stride % 8 == 0 && w_row_stride % 8 == 0 &&
                x_row_stride >= k && w_row_stride >= k && x_row_stride < kSizeLimit && w_row_stride < kSizeLimit, MDX_EUNSUPPORTED,
                "%s: x, W and the result must be 16-byte aligned, row strides multiples of 8 elements and at least k", what);
    return MDX_OK;
}

LinearParams params_of(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int64_t rows, int64_t n, int64_t k)
{
    LinearParams A{};
    A.x = (const __bf16*)x; A.w = (const __bf16*)w;
    A.x_stride = x_row_stride; A.w_stride = w_row_stride;
    A.M = (int)rows; A.N = (int)n; A.K = (int)k; A.splits = 1;
    return A;
}

int run_partials(const char* what, const Plan& plan, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, float* partials,
                 int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const int rc = check_linear(what, x, x_row_stride, w, w_row_stride, partials, rows, n, k);
    if (rc != MDX_OK) return rc;
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.partials = partials;
    A.splits = plan.splits;
    return plan.tile->partials(A, static_cast<hipStream_t>(stream));
}

int run_rows(const char* what, bool silu, const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, void* y, int64_t y_row_stride,
             int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const int rc = check_linear(what, x, x_row_stride, w, w_row_stride, y, rows, n, k);
    if (rc != MDX_OK) return rc;
    MDX_REQUIRE(y_row_stride % 4 == 0 && y_row_stride >= n, MDX_EUNSUPPORTED, "%s: row stride of y (a multiple of 4, at least n)", what);
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.y = (__bf16*)y;
    A.y_stride = y_row_stride;
    const Plan plan = plan_of(rows, n, k, !silu, false, silu);
    return (silu ? plan.tile->silu : plan.tile->rounded)(A, static_cast<hipStream_t>(stream));
}

// Where the kernel is the better one (table at the top of this file): up to 1536 rows; with the SiLU in the epilogue, which
// saves writing and reading twice the result, up to 8192.
constexpr int64_t kMaxRows = 1536, kMaxSiluRows = 8192;
constexpr int64_t kMaxDecodeRows = 128, kMaxDecodeSiluRows = 64;

Plan decode_plan(int64_t rows, int64_t n, int64_t k)
{
    if (!sizes_covered(rows, n, k) || rows > kMaxDecodeRows || n % 64 != 0 || k % 256 != 0) return Plan{nullptr, 0};
    return plan_of(rows, n, k, false, true, false);
}

}  // namespace

extern "C" int32_t mdx_linear_splits(int64_t rows, int64_t n, int64_t k)
{
    if (!sizes_covered(rows, n, k) || rows > kMaxRows) return -1;
    return plan_of(rows, n, k, true, true, false).splits;
}

extern "C" int mdx_linear(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                          void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(sizes_covered(rows, n, k), MDX_EUNSUPPORTED, "linear: %lld rows, n %lld (a multiple of 8), k %lld (a multiple of 128, at least 256)",
                (long long)rows, (long long)n, (long long)k);
    return run_rows("linear", false, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}

extern "C" int mdx_linear_partials(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                   float* partials, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(mdx_linear_splits(rows, n, k) > 0, MDX_EUNSUPPORTED, "linear_partials: %lld rows, n %lld, k %lld are not cut along k",
                (long long)rows, (long long)n, (long long)k);
    return run_partials("linear_partials", plan_of(rows, n, k, true, true, false), x, x_row_stride, w, w_row_stride, partials, rows, n, k, stream);
}

extern "C" int32_t mdx_linear_silu_supported(int64_t rows, int64_t n, int64_t k) { return sizes_covered(rows, n, k) && rows <= kMaxSiluRows; }

extern "C" int mdx_linear_silu(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                               void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(sizes_covered(rows, n, k), MDX_EUNSUPPORTED, "linear_silu: %lld rows, n %lld (a multiple of 8), k %lld (a multiple of 128, at least 256)",
                (long long)rows, (long long)n, (long long)k);
    return run_rows("linear_silu", true, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}

extern "C" int32_t mdx_decode_linear_splits(int64_t rows, int64_t n, int64_t k) { return decode_plan(rows, n, k).splits; }

extern "C" int mdx_decode_linear_partials(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                          float* partials, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    const Plan plan = decode_plan(rows, n, k);
    MDX_REQUIRE(plan.tile, MDX_EUNSUPPORTED, "decode_linear: %lld rows (up to %lld), n %lld (a multiple of 64), k %lld (a multiple of 256)",
                (long long)rows, (long long)kMaxDecodeRows, (long long)n, (long long)k);
    return run_partials("decode_linear", plan, x, x_row_stride, w, w_row_stride, partials, rows, n, k, stream);
}

extern "C" int32_t mdx_decode_linear_silu_supported(int64_t rows, int64_t n, int64_t k)
{
    return sizes_covered(rows, n, k) && rows <= kMaxDecodeSiluRows && n % 24 == 0 && k % 512 == 0;
}

extern "C" int mdx_decode_linear_silu(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                      void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream)
{
    MDX_REQUIRE(mdx_decode_linear_silu_supported(rows, n, k), MDX_EUNSUPPORTED,
                "decode_linear_silu: %lld rows (up to %lld), n %lld (a multiple of 24), k %lld (a multiple of 512)", (long long)rows,
                (long long)kMaxDecodeSiluRows, (long long)n, (long long)k);
    return run_rows("decode_linear_silu", true, x, x_row_stride, w, w_row_stride, y, y_row_stride, rows, n, k, stream);
}
