// A tile of x . W^T on the matrix pipe, in registers: what the linear layers (linear.hip) and the fused vocabulary head
// (lm_head_unmask.hip) have in common.
//
// What bounds it.  A CU takes in at most 70 GB/s from its XCD's L2 (8 wavefronts, loads to LDS, whatever is in flight; 59
// with 4, 78 with 16), all of them 18 TB/s, so a tile of BM x BN costs (BM + BN) x 128 bytes per step of 64 elements of K
// against BM x BN x 128 operations, and only tiles of about 256 x 256 are bound by the matrix pipe (1.25 PFLOP/s of them under
// the board's power limit).  From timing builds, us: 2048 x 2048 x 6144, one tile of 128 x 128 per CU: whole 60, loads alone 58,
// without loads 40, matrix instructions alone 34, LDS reads alone 23; 8192 x 2048 x 6144, one of 256 x 256: 157, 135, 132, 109, 47.
//
//  * S steps of W rows and SX of x rows in LDS (128 bytes of a row per step), filled by loads that pass by the registers
//    (global_load_lds); the 16-byte chunk c of row r sits at c ^ (r / 2 % 8), so that the 16 rows of a fragment read cover all
//    banks once.  One barrier per step: behind it the next step is in LDS for everybody and nobody reads this one any more.
//  * the fragments of the next half step are on their way from LDS while this one is multiplied (two register sets).
//  * small and middle tiles are shared by two groups of four wavefronts, each taking one half of every step (WK = 2): tiles
//    of (BM / 2) x (BN / 2) per wavefront need half of the LDS reads that eight tiles of half the size would, and the two
//    wavefronts of a SIMD cover each other's waits.  The sums meet in LDS at the end.
//  * of the largest tiles only two steps fit in LDS, and a step asked for behind one barrier has to be there at the next; but
//    x fits once more (SX = 3), so that half of a step's loads have two steps to land: 8192 rows of a gate/up projection 358
//    -> 340 us, 1024 rows 50.1 -> 48.8, the head's 500 rows 309 -> 300.
//  * W is the first operand, so that a lane ends with four consecutive columns of one row of x.
// Touching lines of W and x ahead of their loads, starting the workgroups at different steps of K, other bands of tiles per XCD,
// steps of 32 elements (half lines: slower) and six steps in LDS instead of four of the small tiles gained nothing.
#pragma once
#include "mdx_common.h"
#include <type_traits>
#include <utility>

namespace mdx_tile {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) char lds_char;

struct Operands {
    const __bf16* x; const __bf16* w;
    int64_t x_stride, w_stride;                    // elements between rows
    int M, N;                                      // rows of x and of W (pairs: of each half of W)
};

constexpr int kStepK = 64, kRowBytes = 2 * kStepK; // one step of K: 128 bytes of every row

template <typename F, int... J>
__device__ __forceinline__ void for_each(F f, std::integer_sequence<int, J...>) { (f(std::integral_constant<int, J>{}), ...); }

// This wavefront's loads up to the newest N and all of its LDS reads are done, then everybody's.
template <int N> __device__ __forceinline__ void wait_loads_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// BM rows of x by BN rows of W on WM x WN x WK wavefronts.  PAIRS: W is two matrices one after the other (gate, up), and the
// tile's rows of W are 16 rows of the first, the same 16 of the second, and so on.  WIDE: row strides of any size; else below
// kNarrowStride elements, so that a lane's place among the eight rows of a load is 32 bits beside a scalar address (7 x 2^29 bytes).
constexpr int64_t kNarrowStride = (int64_t)1 << 28;
template <int BM_, int BN_, int WM_, int WN_, int WK_, int S_, int SX_, bool PAIRS, bool WIDE = false> struct Tile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, S = S_, SX = SX_;
    static constexpr int kWaves = WM * WN * WK, kThreads = 64 * kWaves;
    static constexpr int TM = BM / (16 * WM), TN = BN / (16 * WN);     // a wavefront's share, in matrix tiles of 16 x 16
    static constexpr int kCols = PAIRS ? BN / 2 : BN;                  // columns of the result
    static constexpr int kXBytes = BM * kRowBytes, kWBytes = BN * kRowBytes, kStepsBytes = SX * kXBytes + S * kWBytes;
    static constexpr int kLeastSteps = SX, kStepsMultiple = WK;        // of 64 elements: at least, and a multiple of
    static constexpr int kXLoads = BM / 8 / kWaves, kLoads = (BM + BN) / 8 / kWaves;
    static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0, "whole loads per wavefront, of x or of W");
    static_assert(WK == 1 || (WK == 2 && TM % 2 == 0 && S % 2 == 0), "halves of a step, pairs of steps");
    static_assert(SX == S || (SX == 3 && S == 2 && WK == 1), "one more step of x, or as many");
    static_assert(!PAIRS || TN % 2 == 0, "pairs of tiles");
    typedef f32x4 Sums[TM][TN];

    int lane, wave, l16, g, wm, wn, wk;
    __device__ __forceinline__ Tile() {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        l16 = lane & 15; g = lane >> 4;
        wm = wave % WM; wn = wave / WM % WN; wk = wave / (WM * WN);
    }

    // Tile (m0, n0) over n_steps steps of K from element k0 on (n_steps: at least kLeastSteps, a multiple of kStepsMultiple).  Sum
    // (i, j) of a wavefront holds, in lane (g, l16), the rows 16 j + 4 g .. + 3 of its part of W by row 16 i + l16 of its part of
    // x; with WK = 2 over its halves of the steps.
    __device__ __forceinline__ void product(const Operands& A, int m0, int n0, int64_t k0, int n_steps, char* lds, Sums& acc) const
    {
        constexpr int kExtra = SX - S;
        // Load i of this wavefront fills 8 rows of the tile, x rows first, then rows of W.  Rows beyond the last are the last one
        // again; their products are not used.
        const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)lds;
        const char* base[kLoads];                           // the first of the 8 rows, at this slice of K
        typedef std::conditional_t<WIDE, uint64_t, unsigned> Offset;
        Offset offset[kLoads];                              // this lane's row and chunk from there
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const bool of_x = i < kXLoads;
            const int r0 = 8 * (wave + kWaves * (of_x ? i : i - kXLoads)), r = lane >> 3, chunk = (lane & 7) ^ (((r0 + r) >> 1) & 7);
            const int first = of_x ? m0 + r0 : PAIRS ? n0 + (r0 >> 5) * 16 + (r0 & 15) : n0 + r0, last = (of_x ? A.M : A.N) - 1;
            const int64_t stride = (of_x ? A.x_stride : A.w_stride) * 2;
            const int64_t second = PAIRS && !of_x && ((r0 >> 4) & 1) ? A.N : 0;
            base[i] = reinterpret_cast<const char*>((of_x ? A.x : A.w) + k0) + (min(first, last) + second) * stride;
            offset[i] = (Offset)(min(first + r, last) - min(first, last)) * (Offset)stride + chunk * 16;
        }
        int64_t x_at = 0, w_at = 0;                         // where the step to ask for next begins
        auto load = [&](int i, unsigned dst, int64_t at) {
            if constexpr (WIDE) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(dst), "v"(base[i] + at + offset[i]) : "memory");
            else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(dst), "v"(offset[i]), "s"(base[i] + at) : "memory");
        };
        auto load_x = [&](int slot) {
#pragma unroll
            for (int i = 0; i < kXLoads; ++i) load(i, lds0 + slot * kXBytes + (wave + kWaves * i) * 1024, x_at);
            x_at += kRowBytes;
        };
        auto load_w = [&](int slot) {
#pragma unroll
            for (int i = kXLoads; i < kLoads; ++i) load(i, lds0 + SX * kXBytes + slot * kWBytes + (wave + kWaves * (i - kXLoads)) * 1024, w_at);
            w_at += kRowBytes;
        };
        const char* xr = lds + (wm * (BM / WM) + l16) * kRowBytes;
        const char* wr = lds + SX * kXBytes + (wn * (BN / WN) + l16) * kRowBytes;
        bf16x8 fx[2][TM], fw[2][TN];
        int sx = 0, sw = 0;                                 // the slots of the step that is read
        auto read = [&](int set, int half) {                // 32 elements of K
            const int pos = ((half * 4 + g) ^ ((l16 >> 1) & 7)) * 16;
#pragma unroll
            for (int i = 0; i < TM; ++i) fx[set][i] = *reinterpret_cast<const bf16x8*>(xr + sx * kXBytes + pos + i * 16 * kRowBytes);
#pragma unroll
            for (int j = 0; j < TN; ++j) fw[set][j] = *reinterpret_cast<const bf16x8*>(wr + sw * kWBytes + pos + j * 16 * kRowBytes);
        };
        auto next = [&]() { sx = sx + 1 == SX ? 0 : sx + 1; sw = sw + 1 == S ? 0 : sw + 1; };
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto multiply = [&](int set) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[set][j], fx[set][i], acc[i][j], 0, 0, 0);
        };

#pragma unroll
        for (int s = 0; s < S; ++s) { load_w(s); load_x(s); }
        if (kExtra) load_x(S);
        wait_loads_and_meet<(S - 1) * kLoads + kExtra * kXLoads>();
        read(0, WK == 2 ? wk : 0);
        // Step t: its second half is read while the first is multiplied (WK = 2: each wavefront has one half, read a step ahead);
        // then step t + 1 has to be in LDS, and what t's slots held is done with: steps t + S of W and t + SX of x are asked for.
        for (int t = 0; t < n_steps - SX; t += WK) {
#pragma unroll
            for (int h = 0; h < WK; ++h) {
                if constexpr (WK == 1) { read(1, 1); multiply(0); }
                wait_loads_and_meet<(S - 2) * kLoads + kExtra * kXLoads>();
                load_w(sw);
                load_x(sx);
                next();
                if constexpr (WK == 1) { read(0, 0); multiply(1); }
                else { read(1 - h, wk); multiply(h); }
            }
        }
        // the last SX steps: nothing more to load, but W's last step where x is one ahead of it
        for_each([&](auto step) {
            constexpr int J = decltype(step)::value;
            if constexpr (WK == 1) { read(1, 1); multiply(0); }
            if constexpr (J + 1 < SX) {
                wait_loads_and_meet<kExtra ? (J == 0 ? kXLoads : 0) : (S - 2 - J) * kLoads>();
                if constexpr (kExtra && J == 0) load_w(sw);
                next();
                if constexpr (WK == 1) read(0, 0); else read(1 - (J & 1), wk);
            }
            if constexpr (WK == 1) multiply(1); else multiply(J & 1);
        }, std::make_integer_sequence<int, SX>{});
    }
};

// Workgroup -> tile.  Consecutive workgroups go to the eight XCDs in turn; each XCD takes a run of the tiles in the order (slice,
// band of row tiles, column tile, row tile): what it has in flight together shares its rows of x and of W in its L2.
constexpr int kBand = 8;                           // row tiles that share a column tile of W one after the other
struct Place { int split, m, n; };
__device__ __forceinline__ Place place_of(int block, int m_tiles, int n_tiles) {
    const int xcd = block & 7, per_xcd = gridDim.x >> 3, more = gridDim.x & 7;
    int at = xcd * per_xcd + min(xcd, more) + (block >> 3);
    const int per_split = m_tiles * n_tiles, split = at / per_split;
    at -= split * per_split;
    const int m_first = at / (kBand * n_tiles) * kBand, m_band = min(kBand, m_tiles - m_first);
    at -= m_first * n_tiles;
    return Place{split, m_first + at % m_band, at / m_band};
}

// A kernel's LDS limit is raised once per device (`raised`: the kernel's own).
inline int reserve_lds(const void* kernel, int bytes, std::atomic<bool>* raised, const char* what) {
    if (bytes <= 65536) return MDX_OK;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "%s: no current device (%s)", what, hipGetErrorString(e));
    if (!raised[device].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "%s: cannot reserve %d bytes of LDS (%s)", what, bytes, hipGetErrorString(e));
        raised[device].store(true, std::memory_order_release);
    }
    return MDX_OK;
}

}  // namespace mdx_tile
