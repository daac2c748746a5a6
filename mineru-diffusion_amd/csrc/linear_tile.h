// A tile of x . W^T on the matrix pipe, in registers: what the linear layers (linear.hip) and the fused vocabulary head
// (lm_head_unmask.hip) have in common.
//
// What bounds it.  A CU takes in up to 100 GB/s of lines that are in its XCD's L2 or the memory-side cache (1 KB per load, to LDS or registers, 128-byte rows or
// whole KB alike), so a step of 64 elements of K of a 256 x 256 tile has its 64 KB in 0.65 us, and the matrix pipe takes 0.85 us for it at 2.4 GHz, 1.1 under the
// board's power limit; a 128 x 128 tile's 0.33 us against 0.21.  W from HBM comes later, not slower: the gate/up projection of 1024 rows takes 38 us with W from HBM,
// 33 without loads (zeros, so that the clock holds).
//
//  * S steps of W rows and SX of x rows in LDS (128 bytes of a row per step), filled by loads that pass by the registers
//    (global_load_lds); the 16-byte chunk c of row r sits at c ^ (r / 2 % 8), so that the 16 rows of a fragment read cover all
//    banks once.  One barrier per step: behind it the next step is in LDS for everybody and nobody reads this one any more.
//  * the fragments of the next half step are on their way from LDS while this one is multiplied (two register sets).
//  * loads and fragment reads stand between the products, each at its place (sched_barrier; with fewer than eight products per wavefront and half step all of them before the first): as a burst behind the barrier, where the compiler leaves them, 64 loads
//    of 1 KB keep the CU's address unit busy for over 1000 cycles, and the products behind them wait to be issued, in all wavefronts at once.  In bursts / between the
//    products, with W from HBM, us: gate/up projection with its SiLU, 1024 rows 51.5 / 45.1, 2048 102 / 88, 4096 183 / 163, 35 840 1480 / 1360; 128 x 128 tiles, 1024 x 2048 x 6144
//    34.5 / 30; smaller tiles 0 to 5 % less; the head's 500 rows 304 / 277.
//  * small and middle tiles are shared by two groups of four wavefronts, each taking one half of every step (WK = 2): tiles
//    of (BM / 2) x (BN / 2) per wavefront need half of the LDS reads that eight tiles of half the size would, and the two
//    wavefronts of a SIMD cover each other's waits.  The sums meet in LDS at the end.
//  * of the largest tiles only two steps and a half fit in LDS.  W has the third (S = 3): it comes from HBM, x mostly from L2 (the head, x / W one step further ahead, us: 256 rows
//    194 / 186, 500 299 / 282, 1024 551 / 531).
//  * W is the first operand, so that a lane ends with four consecutive columns of one row of x.
// Touching lines of W ahead of their loads (a CU's loads come back in order: gate/up 45 -> 49 us), starting the workgroups at different steps of K, other bands of
// tiles per XCD, steps of 32 elements (half lines: slower), more steps in LDS for the middle tiles, a wavefront priority around the products and a barrier that does not wait for the reads (five steps in LDS)
// gained nothing; four wavefronts of 128 x 128 instead of eight of 64 x 128 are slower (35 840 rows 1356 -> 1402 us, the head's 1024 528 -> 544).
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
    static constexpr int kAhead = S > SX ? S : SX;
    static constexpr int kLeastSteps = kAhead, kStepsMultiple = WK;    // of 64 elements: at least, and a multiple of
    static constexpr int kXLoads = BM / 8 / kWaves, kWLoads = BN / 8 / kWaves, kLoads = kXLoads + kWLoads;
    static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0, "whole loads per wavefront, of x or of W");
    static_assert(WK == 1 || (WK == 2 && TM % 2 == 0 && S % 2 == 0), "halves of a step, pairs of steps");
    static_assert(SX == S || (SX == 2 && S == 3 && WK == 1), "one more step of W, or as many");
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
        // load i of the next step of x, of W (in order)
        auto load_x = [&](int slot, int i) {
            load(i, lds0 + slot * kXBytes + (wave + kWaves * i) * 1024, x_at);
            if (i == kXLoads - 1) x_at += kRowBytes;
        };
        auto load_w = [&](int slot, int i) {
            load(kXLoads + i, lds0 + SX * kXBytes + slot * kWBytes + (wave + kWaves * i) * 1024, w_at);
            if (i == kWLoads - 1) w_at += kRowBytes;
        };
        const char* xr = lds + (wm * (BM / WM) + l16) * kRowBytes;
        const char* wr = lds + SX * kXBytes + (wn * (BN / WN) + l16) * kRowBytes;
        bf16x8 fx[2][TM], fw[2][TN];
        int sx = 0, sw = 0;                                 // the slots of the step that is read
        constexpr int kReads = TM + TN;
        auto read = [&](int set, int half, int k) {         // fragment k of 32 elements of K, x first, then W
            const int pos = ((half * 4 + g) ^ ((l16 >> 1) & 7)) * 16;
            if (k < TM) fx[set][k] = *reinterpret_cast<const bf16x8*>(xr + sx * kXBytes + pos + k * 16 * kRowBytes);
            else fw[set][k - TM] = *reinterpret_cast<const bf16x8*>(wr + sw * kWBytes + pos + (k - TM) * 16 * kRowBytes);
        };
        auto next = [&]() { sx = sx + 1 == SX ? 0 : sx + 1; sw = sw + 1 == S ? 0 : sw + 1; };
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

        // The products of fragment set MUL.  Between them, pinned there: `reads` fragments for the other set, in the first three quarters (WK = 2: half), and
        // `loads` loads, all along.  (From the second product on: the first one's wait for its fragments must not find a new read in the queue.)
        constexpr int kProducts = TM * TN, kLead = kProducts >= 8 ? 1 : 0, kReadSpan = kProducts * (WK == 1 ? 6 : 4) / 8;
        auto blend = [&](auto mul, auto reads, int half, auto loads, auto&& ask) {
            constexpr int MUL = decltype(mul)::value, R = decltype(reads)::value, L = decltype(loads)::value;
            for_each([&](auto product) {
                constexpr int P = decltype(product)::value, j = P / TM, i = P % TM;
                constexpr auto at = [](int k, int n, int span) constexpr { const int p = kLead * (k * span / n + 1); return p < kProducts ? p : kProducts - 1; };
#pragma unroll
                for (int l = 0; l < L; ++l) if (at(l, L, kProducts) == P) ask(l);
#pragma unroll
                for (int r = 0; r < R; ++r) if (at(r, R, kReadSpan) == P) read(1 - MUL, half, r);
                __builtin_amdgcn_sched_barrier(0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[MUL][j], fx[MUL][i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, kProducts>{});
        };
        const std::integral_constant<int, 0> none;
        const std::integral_constant<int, kReads> all;
        const std::integral_constant<int, kLoads> step_loads;
        const std::integral_constant<int, 1> one;

        if constexpr (WK == 1) {
            // Step t: its second half is read while the first is multiplied; then step t + 1 has to be in LDS, and what t's slots held is done with: the loads
            // that take them, of W's step t + S and x's t + SX, those that are needed sooner first, go between the products of the second half.
            constexpr bool kXFirst = S > SX;
            constexpr int kNear = kXFirst ? SX : S, kFirst = kXFirst ? kXLoads : kWLoads, kSecond = kLoads - kFirst;
            auto ask = [&](int slot_x, int slot_w, int l) {
                const int i = l < kFirst ? l : l - kFirst;
                if ((l < kFirst) == kXFirst) load_x(slot_x, i); else load_w(slot_w, i);
            };
#pragma unroll
            for (int s = 0; s < kAhead; ++s)
#pragma unroll
                for (int l = s < kNear ? 0 : kFirst; l < kLoads; ++l) ask(s, s, l);
            wait_loads_and_meet<(kNear - 1) * kFirst + (kAhead - 1) * kSecond>();
#pragma unroll
            for (int r = 0; r < kReads; ++r) read(0, 0, r);
            for (int t = 0; t < n_steps - kAhead; ++t) {
                blend(none, all, 1, none, [](int) {});
                wait_loads_and_meet<(kNear - 2) * kFirst + (kAhead - 2) * kSecond>();
                const int slot_x = sx, slot_w = sw;
                next();
                blend(one, all, 0, step_loads, [&](int l) { ask(slot_x, slot_w, l); });
            }
            // the last kAhead steps: nothing more to load, but the last step of what is not as far ahead
            for_each([&](auto step) {
                constexpr int J = decltype(step)::value, kMore = J < kAhead - kNear ? kFirst : 0;
                blend(none, all, 1, none, [](int) {});
                if constexpr (J + 1 < kAhead) {
                    wait_loads_and_meet<kNear < kAhead ? (J == 0 ? kSecond : 0) : (S - 2 - J) * kLoads>();
                    const int slot_x = sx, slot_w = sw;
                    next();
                    blend(one, all, 0, std::integral_constant<int, kMore>{}, [&](int l) { ask(slot_x, slot_w, l); });
                } else {
                    blend(one, none, 0, none, [](int) {});
                }
            }, std::make_integer_sequence<int, kAhead>{});
        } else {
            // Step t: each wavefront has one half of it, read a step ahead.
            auto ask = [&](int slot, int l) { if (l < kWLoads) load_w(slot, l); else load_x(slot, l - kWLoads); };
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int l = 0; l < kLoads; ++l) ask(s, l);
            wait_loads_and_meet<(S - 1) * kLoads>();
#pragma unroll
            for (int r = 0; r < kReads; ++r) read(0, wk, r);
            for (int t = 0; t < n_steps - S; t += 2) {
                for_each([&](auto set) {
                    wait_loads_and_meet<(S - 2) * kLoads>();
                    const int slot = sw;
                    next();
                    blend(set, all, wk, step_loads, [&](int l) { ask(slot, l); });
                }, std::make_integer_sequence<int, 2>{});
            }
            for_each([&](auto step) {
                constexpr int J = decltype(step)::value;
                const std::integral_constant<int, J & 1> set;
                if constexpr (J + 1 < S) {
                    wait_loads_and_meet<(S - 2 - J) * kLoads>();
                    next();
                    blend(set, all, wk, none, [](int) {});
                } else {
                    blend(set, none, wk, none, [](int) {});
                }
            }, std::make_integer_sequence<int, S>{});
        }
    }
};

// Workgroup -> tile.  Consecutive workgroups go to the eight XCDs in turn; each XCD takes a run of the tiles in the order (slice,
// band of row tiles, column tile, row tile): what it has in flight together shares its rows of x and of W in its L2.
constexpr int kBand = 8;                           // row tiles that share a column tile of W one after the other
struct Place { int split, m, n; };
// What that takes: the grid's tiles and what they are divided by.  (With the size of the grid from the dispatch and three general divisions a workgroup asked for its first line after
// 2000 cycles, 0.9 us, so after 1300.  Us, before / now, weights from HBM: 32 rows x 4096 x 2048 6.05 / 5.9, 2048 x 2048 4.33 / 4.13, 256 rows x 2048 x 6144
// 15.5 / 15.35, 1024 rows 30.1 / 29.6, the head of 200 rows 185.8 / 184.8; one request through the engine 61.2 / 60.4 ms.)
struct Places { int m_tiles, n_tiles; unsigned per_xcd, more; mdx::Divisor per_split, m; };
inline Places places_of(int m_tiles, int n_tiles, int64_t grid) {        // grid: below 2^31
    return Places{m_tiles, n_tiles, (unsigned)(grid >> 3), (unsigned)(grid & 7), mdx::divisor((uint64_t)m_tiles * n_tiles, (uint64_t)grid), mdx::divisor(m_tiles, (uint64_t)grid)};
}
__device__ __forceinline__ Place place_of(unsigned block, const Places& P) {
    const unsigned xcd = block & 7;
    unsigned at = xcd * P.per_xcd + min(xcd, P.more) + (block >> 3);
    const unsigned split = at < P.per_split.d ? 0 : mdx::quotient(at, P.per_split);
    at -= split * P.per_split.d;
    if (P.m_tiles <= kBand) {
        const unsigned n = mdx::quotient(at, P.m);
        return Place{(int)split, (int)(at - n * P.m_tiles), (int)n};
    }
    const unsigned m_first = at / (kBand * P.n_tiles) * kBand, m_band = min((unsigned)kBand, P.m_tiles - m_first);
    at -= m_first * P.n_tiles;
    const unsigned n = mdx::quotient(at, m_band);
    return Place{(int)split, (int)(m_first + at - n * m_band), (int)n};
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
