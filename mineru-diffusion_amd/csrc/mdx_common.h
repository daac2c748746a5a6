// Shared host-side helpers of libmdx: error reporting and argument checks.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include "../../include/mdx.h"

namespace mdx {

// Thread-local message behind mdx_last_error().
char* error_buffer();

inline int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error_buffer(), 512, fmt, ap);
    va_end(ap);
    return code;
}

// Checks the launch that was just enqueued; never synchronises.
inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(MDX_ELAUNCH, "%s: %s", what, hipGetErrorString(e));
    return MDX_OK;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int kWave = 64;          // gfx950 wavefront

}  // namespace mdx

// 16-byte vector used for every wide load/store (a native vector type, so the
// nontemporal builtins accept it).
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

namespace mdx {

// Compute units of the current device, read once per device; 256 where no device can be asked (a shape query in a process
// without a GPU).
inline int compute_units() {
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cached[kMaxDevices];
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return 256;
    int n = cached[device].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) n = 256;
        cached[device].store(n, std::memory_order_relaxed);
    }
    return n;
}

}  // namespace mdx

namespace mdx {

// Sum over the 64 lanes: DPP shifts inside the rows of 16 lanes, the two row broadcasts, the total from lane 63
// (six additions, no LDS traffic: the butterfly of cross-lane LDS permutes it replaces sat in every workgroup's start).
__device__ __forceinline__ int wave_sum(int x) {
    int v = x;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ int wave_max(int x) {                         // same pattern; x >= 0
    int v = x;
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
    return __builtin_amdgcn_readlane(v, 63);
}

// The value (of 4 or 8 bytes) of the lane whose number differs in the one bit `mask`, a constant once loops are unrolled; all 64 lanes take part.  In the vector unit: a permute
// through LDS is a trip of over 100 cycles, and a reduction over a wavefront is six of them one behind the other.  Norms, the pick behind a filter, by permutes / so: one request through the
// engine 61.9 / 61.2 ms, 12 x 32 rows filtered with a top-k of 50 34.1 / 33.8 us, of 400 54.6 / 53.1, 3 x 32 rows 20.1 / 19.6.  Not everywhere: the vocabulary pass, whose reduction ends
// every workgroup, is slower so (32 rows 10.97 / 11.99 us; why is not known), and the head's epilogue too (100 rows 155.0 / 155.5).
__device__ __forceinline__ unsigned xor_lanes_word(unsigned x, int mask) {
    const bool upper = (__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)) & mask) != 0;
    switch (mask) {
    case 1: return __builtin_amdgcn_update_dpp(0, x, 0xb1, 0xf, 0xf, false);                                                             // quad_perm 1 0 3 2
    case 2: return __builtin_amdgcn_update_dpp(0, x, 0x4e, 0xf, 0xf, false);                                                             // quad_perm 2 3 0 1
    case 4: return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, false), 0x1b, 0xf, 0xf, false);     // row_half_mirror, quad_perm 3 2 1 0
    case 8: return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false);                                                            // row_ror:8
    case 16: { const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false); return upper ? r[0] : r[1]; }
    default: { const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false); return upper ? r[0] : r[1]; }
    }
}
template <typename V> __device__ __forceinline__ V xor_lanes(V v, int mask) {
    static_assert(sizeof(V) == 4 || sizeof(V) == 8, "words");
    if constexpr (sizeof(V) == 4) {
        return __builtin_bit_cast(V, xor_lanes_word(__builtin_bit_cast(unsigned, v), mask));
    } else {
        const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
        return __builtin_bit_cast(V, (unsigned long long)xor_lanes_word((unsigned)(x >> 32), mask) << 32 | xor_lanes_word((unsigned)x, mask));
    }
}

// n / d of wavefront-uniform numbers for a d that the compiler doesn't know and that is mostly a power of two (heads, groups of heads, tiles): the general
// sequence goes through a float reciprocal in the vector unit and back, in every workgroup's start.  Attention calls, us, by that sequence / so: paged, one sequence of 1337 keys 14.6 / 14.35, four of 1000-3000
// 23.0 / 22.7, 32 of 600-2400 55.9 / 55.5; prompts 3 x 40-150 7.75 / 7.6, 500 13.4 / 13.2.  (In fp32 arithmetic 20.2 / 20.4: not there.)
__device__ __forceinline__ unsigned quotient(unsigned n, unsigned d) { return (d & (d - 1)) == 0 ? n >> __builtin_ctz(d) : n / d; }

// Division of 0 .. n_max by d with one multiplication (the host's choice of the factor; where it does not suffice, 0, by the general sequence).
struct Divisor { unsigned d, factor; };
inline Divisor divisor(uint64_t d, uint64_t n_max) { return Divisor{(unsigned)d, d > 1 && n_max * d < ((uint64_t)1 << 32) ? (unsigned)((((uint64_t)1 << 32) + d - 1) / d) : 0u}; }
__device__ __forceinline__ unsigned quotient(unsigned n, Divisor by) { return by.factor ? __umulhi(n, by.factor) : by.d == 1 ? n : n / by.d; }

// A kernel's arguments come through the scalar cache, 64 bytes at a time, and the compiler asks for them where they are first used, some of them behind
// other loads.  This asks for all lines of BYTES bytes of arguments, and for the grid's size if it is given, at once.  Returns 0 in a way that the
// compiler doesn't see, to be added to something that is used early.  (Not a volatile asm: behind one, the compiler no longer takes page tables and
// lengths for constant and reads them through vector loads.)
// One sequence through attention and combine: 14.2 -> 13.8 us.  Probably a trip to memory less in every workgroup's chain; under the profiler
// one run differs from the next by as much (attention of one sequence 11.0 to 11.4 us with it, 11.3 without).
template <int BYTES>
__device__ __forceinline__ int fetch_arguments(int grid = 0)
{
    typedef __attribute__((address_space(4))) const int Word;
    Word* const a = (Word*)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int kLines = (BYTES + 63) / 64;
    static_assert(kLines >= 1 && kLines <= 4, "lines of arguments");
    int zero;
    if constexpr (kLines == 1) asm("" : "=s"(zero) : "0"(0), "s"(grid), "s"(a[0]));
    if constexpr (kLines == 2) asm("" : "=s"(zero) : "0"(0), "s"(grid), "s"(a[0]), "s"(a[16]));
    if constexpr (kLines == 3) asm("" : "=s"(zero) : "0"(0), "s"(grid), "s"(a[0]), "s"(a[16]), "s"(a[32]));
    if constexpr (kLines == 4) asm("" : "=s"(zero) : "0"(0), "s"(grid), "s"(a[0]), "s"(a[16]), "s"(a[32]), "s"(a[48]));
    return zero;
}

}  // namespace mdx

#define MDX_REQUIRE(cond, code, ...) \
    do { if (!(cond)) return ::mdx::fail(code, __VA_ARGS__); } while (0)
