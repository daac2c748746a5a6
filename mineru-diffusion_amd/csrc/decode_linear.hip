// Linear layers of a decode pass: x . W^T for up to 128 rows of x (the positions of one to four denoising blocks), as
// K-split partial sums that the next kernel adds up (QKV, output and down projections: nanovllm/models/sdar.py:73-112), or
// with the SiLU-and-multiply that follows a gate/up projection (layers/activation.py:7-16).
//
// With so few rows the product is a read of W (100 MB per decoder layer), and what matters is that the whole chip asks for
// it at once and that little stands before or behind the read:
//
//  * about one workgroup per CU: a workgroup owns 64 rows of W (48 of a gate/up projection: 24 of each half) and one slice
//    of K, the slices chosen so that tiles x slices fill the CUs.  Cutting K instead of taking narrower tiles keeps what a
//    workgroup reads of x (its slice alone) below what it reads of W; with 16 columns per workgroup and all of K each, x cost
//    more than W (32 rows: 8.9 + 7.6 + 17.0 + 17.6 us for the four layers below).  The partial sums are small, and the
//    kernels that follow (residual + RMSNorm; q/k norm + RoPE + store) read every element once anyway.
//  * fragments of W go from memory straight into the registers that the matrix instruction reads; x, which the workgroup's
//    wavefronts share, goes to LDS without passing through registers (global_load_lds), its 16-byte chunks swizzled by
//    row so that fragment reads cover all banks.  The next step's loads of both are issued before this step is multiplied.
//  * the contraction order inside a step is free, so a lane takes 32 consecutive bytes of its row of W as two fragments: the
//    four lanes of a row cover a line with two loads.
//
// QKV (4096 x 2048), output (2048 x 2048), gate/up (12288 x 2048, with SiLU) and down (2048 x 6144) projections, cold weights, us, as
// here / library product (+ SiLU kernel): 32 rows 6.5 4.6 15.2 8.6 / 11.7 8.4 18.8 16.6, 64 rows 7.8 5.2 17.9 10.0 / 12.1 8.8
// 20.3 19.4, 128 rows 10.0 6.8 23.7 12.5 / 14.8 8.4 22.3 17.8.  Beyond 128 rows the library's tiles win (256 rows: 15 10 37 20 /
// 14 10 31 23), for gate/up beyond 64.  Bound: the HBM read of W, about 4.5 TB/s in bursts this short, behind 3 us of launch.
#include "mdx_common.h"
#include <atomic>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) char lds_char;

struct LinearParams {
    const __bf16* x; const __bf16* w;
    __bf16* y; float* partials;                    // y: [M, N] (SILU); partials: [splits, M, N]
    int64_t x_stride, w_stride, y_stride;          // elements between rows
    int M, N, K;                                   // N: columns of the result (SILU: W has 2 N rows, gate then up)
    int n_tiles, splits;
};

// 64 lanes x 16 bytes from memory to 1 KB of LDS at `lds` (lane i's bytes at lds + 16 i), counted by vmcnt.
__device__ __forceinline__ void load_to_lds(unsigned lds, const void* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(lds), "v"(p) : "memory");
}

// MT: tiles of 16 rows of x.  WN: wavefronts side by side, 16 rows of W each (SILU: 8 gate and 8 up rows).  WK: wavefronts that
// share a tile of W along K.  KC: elements of K per step.
template <int MT, int WN, int WK, int KC, bool SILU>
__global__ __launch_bounds__(64 * WN * WK, 1) void decode_linear_kernel(const LinearParams A)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];            // two x tiles of [16 MT][KC], later the sums of the other WK wavefronts
    constexpr int kWaves = WN * WK, kRowBytes = KC * 2, kTileBytes = 16 * MT * kRowBytes;
    constexpr int kRowLanes = KC / 8, kRowsPerLoad = 64 / kRowLanes;        // one load to LDS: rows of x
    constexpr int kWaveK = KC / WK, kPairs = kWaveK / 64;                   // a wavefront's share of a step, in pairs of matrix steps
    constexpr int kCols = SILU ? 8 : 16;                                    // columns of the result per wavefront
    static_assert(kRowLanes <= 64 && kWaveK % 64 == 0, "step sizes");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int wn = wave % WN, wk = wave / WN;

    const int tile = blockIdx.x, split = blockIdx.y;
    const int n0 = (tile * WN + wn) * kCols;
    const int k_split = A.K / A.splits, n_steps = k_split / KC;             // (the host's choice: a multiple of KC)
    const int row = SILU ? (l16 < 8 ? n0 + l16 : A.N + n0 + l16 - 8) : n0 + l16;
    const __bf16* wp = A.w + (int64_t)row * A.w_stride + split * k_split + wk * kWaveK + g * 16;
    const __bf16* xp = A.x + split * k_split;
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;

    // x rows of step t into buffer `buf`: position p of row m holds chunk p ^ (m % 16)
    auto stage = [&](int t, int buf) {
#pragma unroll
        for (int i = wave; i < 16 * MT / kRowsPerLoad; i += kWaves) {
            const int m = i * kRowsPerLoad + lane / kRowLanes, chunk = (lane % kRowLanes) ^ (m & 15);
            load_to_lds((unsigned)__builtin_amdgcn_readfirstlane((int)(lds0 + buf * kTileBytes + i * 1024)),
                        xp + (int64_t)min(m, A.M - 1) * A.x_stride + t * KC + chunk * 8);
        }
    };
    bf16x8 wa[kPairs][2], wb[kPairs][2];
    auto fetch = [&](bf16x8 (&w)[kPairs][2], int t) {
#pragma unroll
        for (int p = 0; p < kPairs; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                w[p][h] = *reinterpret_cast<const bf16x8*>(wp + t * KC + p * 64 + h * 8);
    };
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const bf16x8 (&w)[kPairs][2], int buf) {
        const char* rows = lds + buf * kTileBytes + l16 * kRowBytes;
#pragma unroll
        for (int p = 0; p < kPairs; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int at = ((wk * kWaveK / 8 + p * 8 + g * 2 + h) ^ l16) * 16;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[p][h], *reinterpret_cast<const bf16x8*>(rows + mt * 16 * kRowBytes + at), acc[mt], 0, 0, 0);
            }
    };
    // A step's x is in LDS for everybody once each wavefront has waited for its own loads; its W, issued after them, may still be on
    // its way (the compiler waits for that register by register).
    auto arrived = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(2 * kPairs) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    stage(0, 0);
    fetch(wa, 0);
    for (int t = 0; t < n_steps; t += 2) {
        arrived();
        if (t + 1 < n_steps) { stage(t + 1, 1); fetch(wb, t + 1); }
        __builtin_amdgcn_sched_barrier(0);
        multiply(wa, 0);
        if (t + 1 >= n_steps) break;
        arrived();
        if (t + 2 < n_steps) { stage(t + 2, 0); fetch(wa, t + 2); }
        __builtin_amdgcn_sched_barrier(0);
        multiply(wb, 1);
    }

    if (WK > 1) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the x tiles have been read by everybody
        f32x4* sums = reinterpret_cast<f32x4*>(lds);                         // [WK - 1][WN][MT][lane]
        if (wk > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) sums[(((wk - 1) * WN + wn) * MT + mt) * 64 + lane] = acc[mt];
        }
        __syncthreads();
        if (wk > 0) return;
#pragma unroll
        for (int k = 0; k < WK - 1; ++k)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] += sums[((k * WN + wn) * MT + mt) * 64 + lane];
    }
    // lane (g, l16) holds the rows 4 g .. 4 g + 3 of W's tile for row l16 of each x tile
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + l16;
        if (SILU) {
            f32x4 up;                                                        // lanes of the gate rows (g < 2) take the up rows' sums
#pragma unroll
            for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(acc[mt][i], 32);
            if (g >= 2 || m >= A.M) continue;
            bf16x4 out;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float gate = (float)(__bf16)acc[mt][i];                // the projection's own rounding, then SiLU's
                out[i] = (__bf16)((float)(__bf16)(gate / (1.0f + __expf(-gate))) * (float)(__bf16)up[i]);
            }
            *reinterpret_cast<bf16x4*>(A.y + (int64_t)m * A.y_stride + n0 + 4 * g) = out;
        } else if (m < A.M) {
            *reinterpret_cast<f32x4*>(A.partials + ((int64_t)split * A.M + m) * A.N + n0 + 4 * g) = acc[mt];
        }
    }
}

constexpr int kMaxRows = 128, kMaxSiluRows = 64, kStep = 256, kSiluStep = 512;

template <int MT, int WN, int WK, int KC, bool SILU>
int launch(const LinearParams& A, hipStream_t stream)
{
    constexpr int kTiles = 2 * 16 * MT * KC * 2, kSums = (WK - 1) * WN * MT * 1024, kLdsBytes = kTiles > kSums ? kTiles : kSums;
    if (kLdsBytes > 65536) {
        // the kernel's LDS limit is raised once per device
        static std::atomic<bool> raised[64];
        int device = 0;
        hipError_t e = hipGetDevice(&device);
        MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "decode_linear: no current device (%s)", hipGetErrorString(e));
        if (!raised[device].load(std::memory_order_acquire)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(decode_linear_kernel<MT, WN, WK, KC, SILU>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
            MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "decode_linear: cannot reserve %d bytes of LDS (%s)", kLdsBytes, hipGetErrorString(e));
            raised[device].store(true, std::memory_order_release);
        }
    }
    decode_linear_kernel<MT, WN, WK, KC, SILU><<<dim3((unsigned)A.n_tiles, (unsigned)A.splits), 64 * WN * WK, kLdsBytes, stream>>>(A);
    return mdx::check_launch("decode_linear");
}

int check_linear(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, const void* out, int64_t rows, int64_t n, int64_t k)
{
    MDX_REQUIRE(rows >= 0 && n >= 0 && k >= 0, MDX_EINVAL, "decode_linear: negative size");
    MDX_REQUIRE(x && w && out, MDX_EINVAL, "decode_linear: null pointer");
    MDX_REQUIRE(mdx::aligned16(x) && mdx::aligned16(w) && mdx::aligned16(out) && x_row_stride % 8 == 0 && w_row_stride % 8 == 0 &&
                x_row_stride >= k && w_row_stride >= k, MDX_EUNSUPPORTED,
                "decode_linear: x, W and the result must be 16-byte aligned, row strides multiples of 8 elements and at least k");
    return MDX_OK;
}

LinearParams params_of(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int64_t rows, int64_t n, int64_t k)
{
    LinearParams A{};
    A.x = (const __bf16*)x; A.w = (const __bf16*)w;
    A.x_stride = x_row_stride; A.w_stride = w_row_stride;
    A.M = (int)rows; A.N = (int)n; A.K = (int)k;
    return A;
}

}  // namespace

extern "C" int32_t mdx_decode_linear_splits(int64_t rows, int64_t n, int64_t k)
{
    if (rows <= 0 || rows > kMaxRows || n <= 0 || n % 64 != 0 || n >= ((int64_t)1 << 30) || k <= 0 || k % kStep != 0 || k >= ((int64_t)1 << 30)) return 0;
    // as many slices of K as fill the CUs once, each a whole number of steps
    int64_t s = mdx::compute_units() / (n / 64);
    if (s > k / kStep) s = k / kStep;
    if (s < 1) s = 1;
    while (k / kStep % s != 0) --s;
    return (int32_t)s;
}

extern "C" int mdx_decode_linear_partials(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                          float* partials, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int splits = mdx_decode_linear_splits(rows, n, k);
    MDX_REQUIRE(splits > 0, MDX_EUNSUPPORTED, "decode_linear: %lld rows (up to %d), n %lld (a multiple of 64), k %lld (a multiple of %d)",
                (long long)rows, kMaxRows, (long long)n, (long long)k, kStep);
    const int rc = check_linear(x, x_row_stride, w, w_row_stride, partials, rows, n, k);
    if (rc != MDX_OK) return rc;
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.partials = partials;
    A.n_tiles = (int)(n / 64);
    A.splits = splits;
    return rows <= 32 ? launch<2, 4, 2, kStep, false>(A, stream) : rows <= 64 ? launch<4, 4, 2, kStep, false>(A, stream)
                                                                               : launch<8, 4, 2, kStep, false>(A, stream);
}

extern "C" int32_t mdx_decode_linear_silu_supported(int64_t rows, int64_t n, int64_t k)
{
    return rows > 0 && rows <= kMaxSiluRows && n > 0 && n % 24 == 0 && n < ((int64_t)1 << 29) && k > 0 && k % kSiluStep == 0 && k < ((int64_t)1 << 30);
}

extern "C" int mdx_decode_linear_silu(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                      void* y, int64_t y_row_stride, int64_t rows, int64_t n, int64_t k, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(mdx_decode_linear_silu_supported(rows, n, k), MDX_EUNSUPPORTED,
                "decode_linear_silu: %lld rows (up to %d), n %lld (a multiple of 24), k %lld (a multiple of %d)", (long long)rows, kMaxSiluRows,
                (long long)n, (long long)k, kSiluStep);
    const int rc = check_linear(x, x_row_stride, w, w_row_stride, y, rows, n, k);
    if (rc != MDX_OK) return rc;
    MDX_REQUIRE(y_row_stride % 4 == 0 && y_row_stride >= n, MDX_EUNSUPPORTED, "decode_linear_silu: row stride of y (a multiple of 4, at least n)");
    LinearParams A = params_of(x, x_row_stride, w, w_row_stride, rows, n, k);
    A.y = (__bf16*)y;
    A.y_stride = y_row_stride;
    A.n_tiles = (int)(n / 24);
    A.splits = 1;
    return rows <= 32 ? launch<2, 3, 2, kSiluStep, true>(A, stream) : launch<4, 3, 2, kSiluStep, true>(A, stream);
}
