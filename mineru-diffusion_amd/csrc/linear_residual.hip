// A linear layer of few rows with what stands before the next one: residual + x . W^T, and the norm of that as far as a tile can
// take it (nanovllm/layers/linear.py and layernorm.py:28-41, called at nanovllm/models/sdar.py:84,150-152).
//
// RMSNorm needs a row's sum of squares before it can scale anything, and a product that is cut along K for the sake of 256 CUs has to be
// summed before that: a launch between two products that does nothing else.  The scale of a row passes through the next product, though:
// (s w / rms) . V = ((s w) . V) / rms.  So this kernel leaves s (the new residual), z = s w, and the sums of s^2 over each tile's 16 columns;
// mdx_linear_scaled_silu (linear.hip) works on z, adds a row's sums up and scales its result.  z is rounded once where the normed row was
// rounded twice.  Through the engine, ms, three launches / these two: one request 63.4 / 61.4, two 76.4 / 75.6, one of 50 tokens in 4 pages 30.1 / 29.4.
//
// What bounds it: one trip to HBM for W, and what a CU takes in (70 GB/s, linear_tile.h).  A workgroup has 16 columns and 16 TM rows over all of K, cut into
// eight for its eight wavefronts, whose sums meet in LDS at the end.  Each wavefront has a ring of S steps of 64 columns of K in LDS, its own, so that the loop has no
// barrier.  (Fragments straight into registers are loads of 64 bytes of 16 rows each, and both halves of a line came from L2: output projection of 2048 x
// 2048 6.0 us under the profiler, here 4.5, the partial sums that this replaces 4.2; 2048 x 6144 14.0, 10.7 and 7.6.)  With up to 32 rows two workgroups of 16 share a column tile
// (2048 columns: 256 workgroups that take in 131 KB each instead of 128 with 196), next to each other on an XCD, so that W comes from HBM once.  A down projection's
// long K has no such split: with it the same way one request took 62.0 ms and two 77.3, so k ends at 4096.
#include "linear_tile.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kTileCols = 16, kStepK = 64;              // columns of a tile; of K in a step
constexpr int kMaxRows = 64, kMaxK = 4096;

struct ResidualParams {
    const __bf16* x; int64_t x_stride;                  // [M, K]
    const __bf16* w; int64_t w_stride;                  // [N, K]
    const __bf16* residual_in; int64_t in_stride;       // [M, N]
    __bf16* residual_out; int64_t out_stride;
    const __bf16* norm_weight;                          // [N]
    __bf16* z; int64_t z_stride;                        // [M, N]
    float* sums;                                        // [M, N / 16]
    int M, N, K, groups;                                // groups of 16 TM rows
};

// This wavefront's loads up to the newest N have landed.
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <int TM, int S>
__global__ __launch_bounds__(kThreads, 2) void linear_residual_kernel(const ResidualParams P)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    constexpr int kLoads = 2 * (1 + TM), kSlotBytes = kLoads * 1024;       // a step: 8 rows of 128 bytes per load, of W, then of x
    const int block = (int)blockIdx.x + mdx::fetch_arguments<sizeof(ResidualParams)>();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
    const int at = block >> 3, group = at % P.groups, tile = (block & 7) + 8 * (at / P.groups);
    const int n0 = tile * kTileCols, m0 = group * 16 * TM;
    if (n0 >= P.N) return;

    // wavefront i < TM finishes row tile i: in lane (g, l16) the columns 4 g .. + 3 of row l16
    const int n = n0 + 4 * g, m = m0 + 16 * wave + l16;
    bf16x4 residual, weight;
    if (wave < TM) {
        residual = *reinterpret_cast<const bf16x4*>(P.residual_in + (int64_t)min(m, P.M - 1) * P.in_stride + n);
        weight = *reinterpret_cast<const bf16x4*>(P.norm_weight + n);
    }

    // this wavefront's share of K, and its ring: row r of a load at r * 128, its 16-byte chunk c at c ^ (r / 2 % 8) (linear_tile.h).  Rows of x beyond the
    // last are the last one again.
    const int steps = P.K / (kWaves * kStepK);
    char* ring = lds + wave * S * kSlotBytes;
    const unsigned ring0 = (unsigned)(uintptr_t)(lds_char*)ring;
    const char* base[kLoads];
    unsigned offset[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const bool of_x = i >= 2;
        const int r0 = 8 * (of_x ? i - 2 : i), r = lane >> 3, chunk = (lane & 7) ^ (((r0 + r) >> 1) & 7);
        const int first = of_x ? min(m0 + r0, P.M - 1) : n0 + r0, mine = of_x ? min(m0 + r0 + r, P.M - 1) : first + r;
        const int64_t stride = (of_x ? P.x_stride : P.w_stride) * 2;
        base[i] = reinterpret_cast<const char*>(of_x ? P.x : P.w) + first * stride + (int64_t)wave * steps * kStepK * 2;
        offset[i] = (unsigned)(mine - first) * (unsigned)stride + chunk * 16;
    }
    auto load = [&](int slot, int step) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(ring0 + slot * kSlotBytes + i * 1024), "v"(offset[i]), "s"(base[i] + (int64_t)step * 128) : "memory");
    };
    f32x4 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 fw[2], fx[2][TM];
    auto read = [&](int slot) {
        const char* row = ring + slot * kSlotBytes + l16 * 128;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int pos = ((4 * h + g) ^ ((l16 >> 1) & 7)) * 16;
            fw[h] = *reinterpret_cast<const bf16x8*>(row + pos);
#pragma unroll
            for (int i = 0; i < TM; ++i) fx[h][i] = *reinterpret_cast<const bf16x8*>(row + (1 + i) * 2048 + pos);
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[h], fx[h][i], acc[i], 0, 0, 0);
    };
    // (fewer steps than slots: the last one once more, so that the counts below hold; it isn't multiplied)
#pragma unroll
    for (int s = 0; s < S; ++s) load(s, min(s, steps - 1));
    int slot = 0;
    for (int step = S; step < steps; ++step) {
        wait_loads<(S - 1) * kLoads>();
        read(slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                 // (the slot has been read)
        load(slot, step);
        multiply();
        slot = slot + 1 == S ? 0 : slot + 1;
    }
    mdx_tile::for_each([&](auto j) {
        constexpr int J = decltype(j)::value;
        wait_loads<(S - 1 - J) * kLoads>();
        if (J < steps) {
            read(slot);
            multiply();
            slot = slot + 1 == S ? 0 : slot + 1;
        }
    }, std::make_integer_sequence<int, S>{});

    // (all loads into this ring have landed and been read)
    auto sums_of = [&](int w, int i) { return reinterpret_cast<f32x4*>(lds + w * S * kSlotBytes) + i * 64 + lane; };
#pragma unroll
    for (int i = 0; i < TM; ++i) *sums_of(wave, i) = acc[i];
    __syncthreads();
    if (wave >= TM) return;
    f32x4 sum = *sums_of(0, wave);
#pragma unroll
    for (int k = 1; k < kWaves; ++k) sum += *sums_of(k, wave);
    bf16x4 r, z;
    float sq = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float s = (float)(__bf16)sum[e] + (float)residual[e];       // the layer's own rounding, then the sum's
        r[e] = (__bf16)s;
        z[e] = (__bf16)(s * (float)weight[e]);
        sq += s * s;
    }
    sq += __shfl_xor(sq, 16);
    sq += __shfl_xor(sq, 32);
    if (m >= P.M) return;
    *reinterpret_cast<bf16x4*>(P.residual_out + (int64_t)m * P.out_stride + n) = r;
    *reinterpret_cast<bf16x4*>(P.z + (int64_t)m * P.z_stride + n) = z;
    if (g == 0) P.sums[(int64_t)m * (P.N / kTileCols) + tile] = sq;
}

template <int TM, int S>
int launch(ResidualParams P, hipStream_t stream)
{
    constexpr int kLdsBytes = kWaves * S * 2 * (1 + TM) * 1024;
    static std::atomic<bool> raised[64];
    const int rc = mdx_tile::reserve_lds(reinterpret_cast<const void*>(linear_residual_kernel<TM, S>), kLdsBytes, raised, "linear_residual");
    if (rc != MDX_OK) return rc;
    P.groups = (P.M + 16 * TM - 1) / (16 * TM);
    const int64_t grid = (int64_t)((P.N / kTileCols + 7) / 8) * 8 * P.groups;
    linear_residual_kernel<TM, S><<<(unsigned)grid, kThreads, kLdsBytes, stream>>>(P);
    return mdx::check_launch("linear_residual");
}

}  // namespace

// (k: every wavefront has whole lines; n: a row's sums are read by eight lanes, four at a time, up to eight times)
extern "C" int32_t mdx_linear_residual_supported(int64_t rows, int64_t n, int64_t k)
{
    return rows > 0 && rows <= kMaxRows && n > 0 && n % 512 == 0 && n <= 4096 && k > 0 && k % (kWaves * kStepK) == 0 && k <= kMaxK;
}

extern "C" int mdx_linear_residual(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride,
                                   const void* residual_in, int64_t residual_in_row_stride, void* residual_out, int64_t residual_out_row_stride,
                                   const void* norm_weight, void* z, int64_t z_row_stride, float* sums,
                                   int64_t rows, int64_t n, int64_t k, mdx_stream_t stream_)
{
    const char* what = "linear_residual";
    MDX_REQUIRE(rows >= 0, MDX_EINVAL, "%s: negative size", what);
    if (rows == 0) return MDX_OK;
    MDX_REQUIRE(mdx_linear_residual_supported(rows, n, k), MDX_EUNSUPPORTED, "%s: %lld rows (up to %d), n %lld (a multiple of 512 up to 4096), k %lld (a multiple of 512 up to %d)",
                what, (long long)rows, kMaxRows, (long long)n, (long long)k, kMaxK);
    MDX_REQUIRE(x && w && residual_in && residual_out && norm_weight && z && sums, MDX_EINVAL, "%s: null pointer", what);
    MDX_REQUIRE(mdx::aligned16(x) && mdx::aligned16(w) && mdx::aligned16(residual_in) && mdx::aligned16(residual_out) && mdx::aligned16(norm_weight) && mdx::aligned16(z) &&
                x_row_stride % 8 == 0 && w_row_stride % 8 == 0 && residual_in_row_stride % 8 == 0 && residual_out_row_stride % 8 == 0 && z_row_stride % 8 == 0,
                MDX_EUNSUPPORTED, "%s: rows must be 16-byte aligned", what);
    MDX_REQUIRE(x_row_stride >= k && w_row_stride >= k && residual_in_row_stride >= n && residual_out_row_stride >= n && z_row_stride >= n, MDX_EINVAL,
                "%s: row stride smaller than the row", what);
    ResidualParams P{(const __bf16*)x, x_row_stride, (const __bf16*)w, w_row_stride, (const __bf16*)residual_in, residual_in_row_stride,
                     (__bf16*)residual_out, residual_out_row_stride, (const __bf16*)norm_weight, (__bf16*)z, z_row_stride, sums, (int)rows, (int)n, (int)k, 0};
    MDX_REQUIRE(x_row_stride < mdx_tile::kNarrowStride && w_row_stride < mdx_tile::kNarrowStride, MDX_EUNSUPPORTED, "%s: row strides of x and W", what);
    return rows <= 32 ? launch<1, 4>(P, static_cast<hipStream_t>(stream_)) : launch<2, 3>(P, static_cast<hipStream_t>(stream_));
}
