// The per-block confidence unmask step: softmax confidence + first-index argmax
// over the vocabulary, then threshold / top-k selection of masked positions.
//
// The vocabulary pass is a single HBM stream over the logits (311 MB at
// [32 x 32 x 151936] bf16), so it is built for bandwidth, not MFMA: 16-byte
// coalesced loads, several in flight per lane, an online (max, sum-of-exp)
// pair per lane that is only rescaled when a 16-byte chunk raises the running
// maximum, wavefront shuffles and one LDS hop for the row reduction.  The
// argmax is found without per-element index bookkeeping: a lane notes the
// position of a new maximum only when a 16-byte chunk raises its running maximum,
// while that chunk is still in registers.
//
// Semantics follow engines/nano_dvlm/nanovllm/layers/sampler.py:11-61 and
// mineru_diffusion/modeling_mineru_diffusion.py:518-532.
#include "mdx_common.h"
#include "gumbel_noise.h"
#include "filtered_pick.h"
#include "logit_keys.h"
#include <hip/hip_fp16.h>

namespace {

using namespace mdx_noise;

constexpr int kThreads = 256;
constexpr int kUnroll = 2;               // 16-byte loads in flight per lane
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegBig = mdx_keys::kNoConfidence;   // finite stand-in for -inf: keeps (m - m) away from inf - inf
constexpr int kNoIndex = 0x7fffffff;

struct Partial {                         // one row's (or row split's) running state
    float m;                             // max of the raw logits seen
    float s;                             // sum of exp((x - m)/T)
    int idx;                             // first index holding m
    float pick;                          // with noise: best (x/T + g); else unused
    float pick_x;                        // with noise: raw logit at that index
    int pick_idx;                        // with noise: first index of the best
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max of three in one instruction.  fmaxf(fmaxf(a, b), c) costs the compiler two more instructions per
// freshly unpacked pair, to quiet signalling NaNs that logits do not hold.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Combine b into a.  c = log2(e)/T.
__device__ __forceinline__ void combine(Partial& a, const Partial& b, float c, bool noise) {
    const float M = fmaxf(a.m, b.m);
    a.s = a.s * fast_exp2((a.m - M) * c) + b.s * fast_exp2((b.m - M) * c);
    a.idx = (b.m > a.m) ? b.idx : ((b.m == a.m) ? min(a.idx, b.idx) : a.idx);
    a.m = M;
    if (noise) {
        const bool take = (b.pick > a.pick) || (b.pick == a.pick && b.pick_idx < a.pick_idx);
        if (take) { a.pick = b.pick; a.pick_x = b.pick_x; a.pick_idx = b.pick_idx; }
    }
}

__device__ __forceinline__ Partial shfl_xor(const Partial& p, int mask, bool noise) {
    Partial r;
    r.m = __shfl_xor(p.m, mask);
    r.s = __shfl_xor(p.s, mask);
    r.idx = __shfl_xor(p.idx, mask);
    if (noise) {
        r.pick = __shfl_xor(p.pick, mask);
        r.pick_x = __shfl_xor(p.pick_x, mask);
        r.pick_idx = __shfl_xor(p.pick_idx, mask);
    } else {
        r.pick = kNegBig; r.pick_x = 0.f; r.pick_idx = kNoIndex;
    }
    return r;
}

// A row's final answer.  A row without any finite logit (all -inf) has no softmax: it reports
// token 0 (where an argmax over equal values lands) with confidence 0, so no rule ever commits it.
template <bool NOISE>
__device__ __forceinline__ void finish_row(const Partial& r, float c, int64_t& x0, float& x0_p) {
    if (r.idx == kNoIndex) { x0 = 0; x0_p = 0.f; return; }
    if (NOISE) {
        x0 = r.pick_idx;
        x0_p = fast_exp2((r.pick_x - r.m) * c) / r.s;
    } else {
        x0 = r.idx;
        x0_p = fminf(1.0f / r.s, 1.0f);          // the sum holds exp2(0) up to rounding
    }
}

// --- element access by logits type: EPC = elements per 16-byte chunk ---------
template <typename T> struct Elem;
template <> struct Elem<__bf16> {
    static constexpr int EPC = 8;
    static __device__ __forceinline__ void unpack(const u32x4& u, float* x) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[2 * i] = __uint_as_float(w[i] << 16);
            x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ float one(const __bf16* p) {
        return __uint_as_float((uint32_t)(*reinterpret_cast<const uint16_t*>(p)) << 16);
    }
};
template <> struct Elem<__half> {
    static constexpr int EPC = 8;
    static __device__ __forceinline__ void unpack(const u32x4& u, float* x) {
        const __half2* h = reinterpret_cast<const __half2*>(&u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float2 f = __half22float2(h[i]);
            x[2 * i] = f.x;
            x[2 * i + 1] = f.y;
        }
    }
    static __device__ __forceinline__ float one(const __half* p) { return __half2float(*p); }
};
template <> struct Elem<float> {
    static constexpr int EPC = 4;
    static __device__ __forceinline__ void unpack(const u32x4& u, float* x) {
        x[0] = __uint_as_float(u.x); x[1] = __uint_as_float(u.y);
        x[2] = __uint_as_float(u.z); x[3] = __uint_as_float(u.w);
    }
    static __device__ __forceinline__ float one(const float* p) { return *p; }
};

// One element through the slow path (row head/tail).  With noise, l = x / T is a
// true fp32 division so the noisy argmax matches an fp32 host computation bit for bit.
template <bool NOISE>
__device__ __forceinline__ void visit(Partial& p, float x, int index, float c, float T, float g) {
    if (x > p.m) {
        p.s *= fast_exp2((p.m - x) * c);
        p.m = x;
        p.idx = index;
    } else if (x == p.m && index < p.idx) {
        p.idx = index;
    }
    p.s += fast_exp2((x - p.m) * c);
    if (NOISE) {
        const float l = x / T;
        const float v = l + g;
        if (v > p.pick || (v == p.pick && index < p.pick_idx)) { p.pick = v; p.pick_x = x; p.pick_idx = index; }
    }
}

// What the selection needs.  `arrive`: null, or an arrival counter per sequence, zero between launches, and the vocabulary pass selects
// by itself (select_when_last).  (Arrivals at one cache line take about 3 ns each, one behind the other: with the counters next to each other,
// 8 sequences of 9 splits took 26 us instead of 18.)
constexpr int kCounterWords = 64;                            // from one counter to the next
struct Selection {
    uint32_t* arrive;
    int64_t* tokens; int64_t mask_token_id; float threshold; int k;
    uint8_t* transfer; int32_t* count; int block_len, lanes;
};

// The rule for a block of up to 64 positions, by ONE wavefront: lane p owns position p, counts are ballots, and the rank among the masked positions
// comes from reading every lane's confidence in turn -- no LDS, no atomics, no barrier.
__device__ __forceinline__ void select_by_wave(const Selection& S, int b, int p, bool masked, int64_t pick, float pick_p)
{
    const bool on = p < S.block_len;
    const int64_t at = (int64_t)b * S.block_len + p;
    const float conf = masked ? pick_p : -INFINITY;
    const bool hi = conf > S.threshold;
    bool commit;
    if (__popcll(__ballot(hi)) >= S.k) {
        commit = hi;
    } else {
        // rank among masked positions: higher confidence first, lower position first on ties
        int rank = 0;
        for (int j = 0; j < S.block_len; ++j) {
            const float cj = __shfl(conf, j);
            rank += (cj > conf || (cj == conf && j < p)) ? 1 : 0;
        }
        commit = masked && rank < S.k && conf > -INFINITY;   // at most min(k, #masked) positions; a confidence of -inf is never committed
    }
    const int n_commit = __popcll(__ballot(commit));
    if (on) {
        S.transfer[at] = commit ? 1 : 0;
        if (commit) S.tokens[at] = pick;
    }
    if (p == 0) S.count[b] = n_commit;
}

// The rows that a call asks for, where it does not want all: a kernel's first argument, so that a workgroup's row is one scalar load away.
constexpr int kMaxLiveRows = 1024;
struct LiveRows { uint16_t row[kMaxLiveRows]; };
__device__ __forceinline__ int live_row(int i) {
    typedef __attribute__((address_space(4))) const uint32_t Word;
    const uint32_t two = ((Word*)__builtin_amdgcn_kernarg_segment_ptr())[i >> 1];
    return (int)(i & 1 ? two >> 16 : two & 0xffff);
}

// Between workgroups of one launch: stores that are written through to memory and loads that take no line that this XCD's L2 may still hold.
template <typename T> __device__ __forceinline__ void put_agent(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ T get_agent(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void store_agent(Partial* to, const Partial& p) {
    put_agent(&to->m, p.m); put_agent(&to->s, p.s); put_agent(&to->idx, p.idx);
    put_agent(&to->pick, p.pick); put_agent(&to->pick_x, p.pick_x); put_agent(&to->pick_idx, p.pick_idx);
}
template <bool NOISE> __device__ __forceinline__ Partial load_agent(const Partial* from) {
    return Partial{get_agent(&from->m), get_agent(&from->s), get_agent(&from->idx), NOISE ? get_agent(&from->pick) : kNegBig,
                   NOISE ? get_agent(&from->pick_x) : 0.f, NOISE ? get_agent(&from->pick_idx) : kNoIndex};
}

// A row's splits merged by a group of lanes: each takes every lanes-th, then the exchanges.  (One lane per row walking
// the splits was a chain of dependent trips to memory: 6.2 us for nine splits, a third of what 96 sampled rows take.  Two or
// three splits are walked all the same: a selection launch of 16 lanes per position takes 0.4 us longer than one of one.)
constexpr int kMergeLanes = 16;                // at most
int merge_lanes(int nsplit) { return nsplit <= 3 ? 1 : nsplit <= 8 ? 4 : kMergeLanes; }
template <bool NOISE> __device__ __forceinline__ Partial merge_lanes_of(Partial r, int lanes, float c) {
    for (int off = lanes / 2; off >= 1; off >>= 1) combine(r, shfl_xor(r, off, NOISE), c, NOISE);
    return r;
}
template <bool NOISE>
__device__ __forceinline__ Partial merge_splits(const Partial* __restrict__ partials, int nsplit, int lane, int lanes, float c) {
    Partial r;
    r.m = kNegBig; r.s = 0.f; r.idx = kNoIndex; r.pick = kNegBig; r.pick_x = 0.f; r.pick_idx = kNoIndex;
    for (int s = lane; s < nsplit; s += lanes) combine(r, partials[s], c, NOISE);
    return merge_lanes_of<NOISE>(r, lanes, c);
}

// The end of a workgroup of the vocabulary pass that selects by itself: the last one of a sequence to arrive merges its rows' splits and applies
// the rule.  No workgroup waits for another; what the last one reads of the others was in memory before they arrived.  own: in thread 0, what the workgroup has found.
// Three trips to memory (store, arrival, merge) take the GPU about as long as a second launch does, and the host 2 to 3.5 us less (one_launch_pays has where they don't).
// (A counter per row as well, and a merge per row, was a trip more: 5 sequences 16.2, 8 18.6.  Arrivals at 16 counters of a sequence first, the last of each at the sequence's own: 1 block of 32 in
// 9 splits 12.5 / 10.9, 2 13.2 / 12.2, 3 14.0 / 13.6, 5 15.1 / 15.5; two launches 9.6, 10.9, 12.3, 15.0.)
template <bool NOISE, bool LIVE>
__device__ __forceinline__ void select_when_last(const Selection& S, const Partial& own, int row, int split, float c, int nsplit, Partial* partials, int64_t* x0, float* x0_p)
{
    __shared__ bool last;
    __shared__ float conf_s[mdx::kWave];
    __shared__ int pick_s[mdx::kWave];
    const int tid = threadIdx.x, b = row / S.block_len;
    const int64_t first = (int64_t)b * S.block_len;
    uint32_t* const counter = S.arrive + (int64_t)b * kCounterWords;
    bool masked = false;
    if (tid < mdx::kWave) {
        if (tid == 0) {
            if (nsplit > 1) {
                store_agent(partials + (int64_t)row * nsplit + split, own);
            } else {
                int64_t tok; float conf;
                finish_row<NOISE>(own, c, tok, conf);
                put_agent(x0 + row, tok);
                put_agent(x0_p + row, conf);
            }
        }
        int rows = S.block_len;
        if (LIVE) {                          // (the list is in order, and a sequence has at most 64 rows)
            unsigned long long asked = 0;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int e = (int)blockIdx.x - (mdx::kWave - 1) + k * mdx::kWave + tid;
                const int other = e >= 0 && e < (int)gridDim.x ? live_row(e) - (int)first : -1;
                if (other >= 0 && other < S.block_len) asked |= 1ull << other;
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) asked |= __shfl_xor(asked, off);
            masked = (asked >> tid) & 1;
            rows = __popcll(asked);
        } else if (tid < S.block_len) {
            masked = S.tokens[first + tid] == S.mask_token_id;
        }
        if (tid == 0) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(rows * nsplit - 1);
        }
    }
    __syncthreads();
    if (!last) return;
    if (nsplit > 1) {
        // (rows that a call does not ask for: whatever is there, of positions that are in no race)
        const int lane = tid & (S.lanes - 1), step = kThreads / S.lanes;
        for (int p = tid / S.lanes; p < S.block_len; p += 2 * step) {
            Partial r[2];                    // both on their way together
#pragma unroll
            for (int k = 0; k < 2; ++k)
                if (p + k * step < S.block_len && lane < nsplit) r[k] = load_agent<NOISE>(partials + (first + p + k * step) * nsplit + lane);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int64_t at = first + p + k * step;
                if (p + k * step >= S.block_len) break;      // (whole groups)
                Partial sum;
                sum.m = kNegBig; sum.s = 0.f; sum.idx = kNoIndex; sum.pick = kNegBig; sum.pick_x = 0.f; sum.pick_idx = kNoIndex;
                if (lane < nsplit) combine(sum, r[k], c, NOISE);
                for (int sp = lane + S.lanes; sp < nsplit; sp += S.lanes) combine(sum, load_agent<NOISE>(partials + at * nsplit + sp), c, NOISE);
                sum = merge_lanes_of<NOISE>(sum, S.lanes, c);
                if (lane == 0) {
                    int64_t tok; float conf;
                    finish_row<NOISE>(sum, c, tok, conf);
                    x0[at] = tok;
                    x0_p[at] = conf;
                    pick_s[p + k * step] = (int)tok;
                    conf_s[p + k * step] = conf;
                }
            }
        }
        __syncthreads();
    }
    if (tid >= mdx::kWave) return;
    int64_t pick = 0;
    float pick_p = 0.f;
    if (masked) {
        pick = nsplit > 1 ? pick_s[tid] : get_agent(x0 + first + tid);
        pick_p = nsplit > 1 ? conf_s[tid] : get_agent(x0_p + first + tid);
    }
    select_by_wave(S, b, tid, masked, pick, pick_p);
    if (tid == 0) put_agent(counter, 0u);                    // ready for the next launch
}

// grid = (rows, nsplit).  Each workgroup reduces chunks [split*cps, (split+1)*cps)
// of one row; split 0 also takes the unaligned head and tail elements.
// NOISE: 0 = plain argmax, 1 = noise read from a tensor, 2 = noise drawn in the kernel.
// FLOOR: elements below floors[row] count as -inf (what a top-k / top-p filter would have left of the row).
// LIVE: none, or LiveRows: only those rows.
// With S.arrive the launch selects as well (never with floors: the filtered step selects in a launch of its own).
template <typename T, int NOISE, bool FLOOR, typename... LIVE>
__global__ __launch_bounds__(kThreads) void confidence_argmax_kernel(
    const LIVE... live, const T* __restrict__ logits, int64_t row_stride,
    const float* __restrict__ temperatures, int rows_per_temp,
    const NoiseSpec N, const float* __restrict__ floors,
    int64_t vocab, int nsplit,
    Partial* __restrict__ partials,          // [rows, nsplit] when nsplit > 1
    int64_t* __restrict__ x0, float* __restrict__ x0_p, const Selection S)
{
    constexpr int EPC = Elem<T>::EPC;
    // (without LIVE from an unsigned number: from a signed one the compiler forms other code, and the step of 8 sequences takes 19.8 instead of 19.3 us, the
    // sampled one 42.6 instead of 42.1)
    const uint32_t row32 = sizeof...(LIVE) > 0 ? (uint32_t)live_row(blockIdx.x) : blockIdx.x;
    const int64_t row = row32;
    const int split = blockIdx.y;
    const int tid = threadIdx.x;
    const T* rp = logits + row * row_stride;
    const float* np = NOISE == 1 ? N.noise + row * N.noise_row_stride : nullptr;
    // (rows and vocabulary are below 2^31; two divisions of 64 bits here cost a workgroup's first load 1 % of the whole step: us, 32 sequences 53.6 / 53.3, one 11.03 / 10.84)
    const float T_ = temperatures ? temperatures[mdx::quotient(row32, rows_per_temp)] : 1.0f;
    const float c = kLog2e / T_;
    const float floor = FLOOR ? floors[row] : 0.f;
    auto unpack = [&](const u32x4& u, float (&x)[Elem<T>::EPC]) {
        Elem<T>::unpack(u, x);
#pragma unroll
        for (int i = 0; FLOOR && i < Elem<T>::EPC; ++i) x[i] = x[i] >= floor ? x[i] : -INFINITY;
    };
    auto one = [&](int64_t e) {
        const float x = Elem<T>::one(rp + e);
        return !FLOOR || x >= floor ? x : -INFINITY;
    };

    // Row geometry: `lead` scalar elements up to the first 16-byte boundary,
    // `nchunk` aligned chunks, then a scalar tail.
    const uintptr_t addr = reinterpret_cast<uintptr_t>(rp);
    int64_t lead = ((16 - (addr & 15)) & 15) / sizeof(T);
    if (lead > vocab) lead = vocab;
    const int64_t nchunk = (vocab - lead) / EPC;
    const int64_t tail0 = lead + nchunk * EPC;
    const u32x4* cp = reinterpret_cast<const u32x4*>(rp + lead);

    const int64_t cps = mdx::quotient((unsigned)nchunk + nsplit - 1, nsplit);      // chunks per split
    const int64_t cbeg = split * cps;
    const int64_t cend = min(nchunk, cbeg + cps);

    Partial p;
    p.m = kNegBig; p.s = 0.f; p.idx = kNoIndex; p.pick = kNegBig; p.pick_x = 0.f; p.pick_idx = kNoIndex;
    __shared__ float lead_seen;              // mode 2: the best noisy logit any wavefront of the workgroup has published
    if (NOISE == 2) {
        if (tid == 0) lead_seen = kNegBig;
        __syncthreads();
    }

    // Softmax over 16-byte chunks (modes 0 and 2).  Per lane: running max m, h = -(m * c) rounded to fp32,
    // and s = sum of exp2(x * c + h), each exponent one FMA (x * c + h is rounded once, so the term of x == m is exp2(lo) with
    // lo = m * c + h, the rounding error of the product, known exactly).  The sum that the row
    // reduction wants, sum of exp2((x - m) * c), is s * exp2(-lo): applied once per lane after
    // the loop.  Folding m * c into the FMA without that correction would carry its rounding,
    // 2^-24 |m c|, into every term (1e-3 at logits of thousands).
    float m = kNegBig, s = 0.f, h = 0.f;
    int first_at = -1;           // element (counted from the first aligned chunk) that first held m
    auto take_values = [&](const float (&x)[EPC], int first) -> float {         // of the chunk from element `first` on; returns the largest
        float cm = x[EPC - 1];
#pragma unroll
        for (int i = 0; i + 2 < EPC; i += 2) cm = max3(cm, x[i], x[i + 1]);
        if (EPC % 2 == 0) cm = max3(cm, x[EPC - 2], x[EPC - 2]);
        if (cm > m) {
            // found here, while the chunk is in registers: reading it again at the end
            // would fetch a whole cache line per lane from HBM (10 % more traffic)
            int j = EPC - 1;
#pragma unroll
            for (int i = EPC - 2; i >= 0; --i) if (x[i] == cm) j = i;
            first_at = first + j;
            const float h_new = -(cm * c);
            s = s > 0.f ? s * fast_exp2(h_new - h) : 0.f;   // h_new <= h once a finite maximum exists
            m = cm;
            h = h_new;
        }
        float acc = fast_exp2(__builtin_fmaf(x[0], c, h));
#pragma unroll
        for (int i = 1; i < EPC; ++i) acc += fast_exp2(__builtin_fmaf(x[i], c, h));
        s += acc;
        return cm;
    };
    auto lane_softmax_done = [&]() {
        if (m > kNegBig) s *= fast_exp2(-__builtin_fmaf(m, c, h));   // to the base of m itself (a lane that saw no finite element keeps s == 0)
        p.m = m;
        p.s = s;
        if (first_at >= 0) p.idx = (int)lead + first_at;
    };

    if (NOISE == 0) {
        auto take = [&](const u32x4 u, int64_t chunk) {
            float x[EPC];
            unpack(u, x);
            take_values(x, (int)chunk * EPC);
        };
        int64_t ch = cbeg + tid;
        // Main loop: the next group's kUnroll loads are issued before this group is reduced, so a lane
        // always has loads outstanding while it computes (measured on [1024 x 151936] bf16: 53.7 -> 50.9 us
        // for the step with two loads per group; four per group, or alternating between two register
        // sets instead of handing the prefetched group over, are 3 to 5 % slower).
        constexpr int64_t kStep = (int64_t)kUnroll * kThreads;
        auto have = [&](int64_t at) { return at + kStep - kThreads < cend; };
        auto fetch = [&](u32x4 (&r)[kUnroll], int64_t at) {
#pragma unroll
            for (int k = 0; k < kUnroll; ++k) r[k] = __builtin_nontemporal_load(cp + at + (int64_t)k * kThreads);
        };
        auto reduce = [&](const u32x4 (&r)[kUnroll], int64_t at) {
#pragma unroll
            for (int k = 0; k < kUnroll; ++k) take(r[k], at + (int64_t)k * kThreads);
        };
        u32x4 u[kUnroll];
        if (have(ch)) fetch(u, ch);
        for (; have(ch); ch += kStep) {
            const bool more = have(ch + kStep);
            u32x4 w[kUnroll];
            if (more) fetch(w, ch + kStep);
            reduce(u, ch);
            if (more) {
#pragma unroll
                for (int k = 0; k < kUnroll; ++k) u[k] = w[k];
            }
        }
        for (; ch < cend; ch += kThreads) take(__builtin_nontemporal_load(cp + ch), ch);
        lane_softmax_done();
        if (split == 0) {            // unaligned head and tail, a handful of elements
            for (int64_t e = tid; e < lead; e += kThreads) visit<false>(p, one(e), (int)e, c, T_, 0.f);
            for (int64_t e = tail0 + tid; e < vocab; e += kThreads) visit<false>(p, one(e), (int)e, c, T_, 0.f);
        }
    } else {
        // With noise.  The softmax runs over 16-byte chunks as without noise; the noisy argmax is element by
        // element: l = x / T by a true division (skipped, not approximated, when T = 1: x / 1 == x), v = l + g, the
        // larger v or at equal v the lower index wins -- the arithmetic of an fp32 host computation, bit for bit.
        // The noise g of an element is read from the tensor (mode 1; 16-byte loads when the row's noise lines up
        // with its chunks) or drawn from the generator (mode 2: a chunk whose first column is a multiple of 4 --
        // every row that starts on a 16-byte boundary -- takes whole generator outputs, EPC / 4 of them; otherwise
        // every element asks for its own), so both modes draw the same tokens from the same noise.
        const RowNoise rn = NOISE == 2 ? row_noise(N, row) : RowNoise{0, 0, 0, 0, 0};
        const bool whole_groups = (lead & 3) == 0;
        const bool noise_lines_up = NOISE == 1 && (reinterpret_cast<uintptr_t>(np + lead) & 15) == 0;
        const bool unit_T = T_ == 1.0f;
        float best = kNegBig, best_x = 0.f;
        float seen = kNegBig;            // mode 2: what this wavefront knows of the workgroup's best noisy logit (same in all lanes)
        int best_idx = kNoIndex, since_look = 0;
        auto offer = [&](float x, int index, float g) {
            const float v = (unit_T ? x : x / T_) + g;
            if (v > best || (v == best && index < best_idx)) { best = v; best_x = x; best_idx = index; }
        };
        // No less than x / T, for the tests below: the reciprocal and the product are off by 2^-24 of it each.  (One instruction per
        // chunk more than the product instead of the ten of a division; with 32-bit counts in the loop, which is bound by its
        // instructions from 256 rows on: 768 rows 89.5 -> 87.3 us for the step, 1024 114 -> 111.5; 32 to 160 rows level.)
        const float inv_T = 1.0f / T_;
        const bool plain_T = inv_T > 1e-30f && inv_T < 1e30f;
        auto at_most = [&](float x) {
            const float l = plain_T ? x * inv_T : x / T_;
            return __builtin_fmaf(fabsf(l), 4.76837158203125e-07f, l);
        };
        auto noise_at = [&](int64_t e) { return NOISE == 1 ? np[e] : rn.at((int)e); };
        // The chunks after this one are on their way while it is worked on: few wavefronts share a SIMD here (96 rows:
        // three), and where the noise of a chunk is skipped there is little else to hide a trip to HBM behind.
        const u32x4* part = cp + cbeg;
        const uint32_t chunks = (uint32_t)max(cend - cbeg, (int64_t)0);
        const int e0 = (int)cbeg * EPC;                          // element, counted from the first aligned chunk, that the part begins with
        u32x4 next[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; ++k)
            if (tid + k * kThreads < chunks) next[k] = __builtin_nontemporal_load(part + tid + k * kThreads);
        for (uint32_t at = (uint32_t)tid; at < chunks; at += kThreads) {
            float x[EPC];
            unpack(next[0], x);
#pragma unroll
            for (int k = 0; k + 1 < kUnroll; ++k) next[k] = next[k + 1];
            if (at + kUnroll * kThreads < chunks) next[kUnroll - 1] = __builtin_nontemporal_load(part + at + kUnroll * kThreads);
            const float cmx = take_values(x, e0 + (int)at * EPC);
            const int c0 = (int)lead + e0 + (int)at * EPC;
            // No draw of the generator exceeds kGumbelMax, and rounding is monotonic: an element of this chunk can
            // take (or tie) the row's lead only if (largest element) / T + kGumbelMax reaches the best noisy logit
            // that anybody in the workgroup has found so far (lead_seen: published by the wavefronts as they go; an
            // old value only makes the test more cautious).  Where that holds in no lane of the wavefront the
            // chunk's noise is not drawn -- every chunk of -inf that a top-k / top-p filter left behind, and the
            // bulk of a peaked row; what is skipped could not have been picked.  (A noise tensor may hold
            // anything: mode 1 reads all of it.)
            if (NOISE == 2) {
                ++since_look;                          // the others' news at chunks 1, 2, 4, 8, 16, 24, ...: an LDS read per chunk would cost what it saves
                if ((since_look & min(since_look - 1, 7)) == 0)
                    seen = fmaxf(seen, __hip_atomic_load(&lead_seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                const bool may_lead = at_most(cmx) + kGumbelMax >= fmaxf(best, seen);
                if (__builtin_amdgcn_ballot_w64(may_lead) == 0) continue;
            }
            if (NOISE == 1) {
                float g[EPC];
                if (noise_lines_up) {
#pragma unroll
                    for (int q = 0; q < EPC / 4; ++q) {
                        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(np + c0) + q);
                        g[4 * q + 0] = __uint_as_float(w.x); g[4 * q + 1] = __uint_as_float(w.y);
                        g[4 * q + 2] = __uint_as_float(w.z); g[4 * q + 3] = __uint_as_float(w.w);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < EPC; ++i) g[i] = np[c0 + i];
                }
#pragma unroll
                for (int i = 0; i < EPC; ++i) offer(x[i], c0 + i, g[i]);
            } else if (whole_groups) {
                U4 r[EPC / 4];
#pragma unroll
                for (int q = 0; q < EPC / 4; ++q) r[q] = rn.group((uint32_t)(c0 >> 2) + q);
                // The generator's bits decide before any logarithm is taken.  An element reaches the lead only with
                // noise -ln(-ln u) >= need = lead - (largest element) / T, i.e. -ln u <= e^-need; and -ln u >= 1 - u
                // = (j + 1/2) 2^-23, where j = ~bits >> 9 counts u down from its largest value.  So only draws with
                // j <= e^-need 2^23 matter: at need = 10, one in 22 000.  need is taken 0.02 + 2^-22 |lead| lower than
                // computed, which covers the error of the hardware logarithms (2e-6) and every rounding on the way.
                const float lim = fmaxf(best, seen);
                const float need = lim - at_most(cmx) - __builtin_fmaf(fabsf(lim), 2.384185791015625e-07f, 0.02f);
                const float reach = fminf(fast_exp2(__builtin_fmaf(-kLog2e, need, 23.f)), 8388608.f);    // NaN (lead and element both infinite) -> the other operand
                uint32_t top = 0;
#pragma unroll
                for (int q = 0; q < EPC / 4; ++q) top = max(max(top, max(r[q].x, r[q].y)), max(r[q].z, r[q].w));
                const uint32_t bound = (uint32_t)reach + 1u;
                if (__builtin_amdgcn_ballot_w64((~top >> 9) <= bound) == 0) continue;
                // and element by element, since mostly one draw of the wavefront's 512 has passed: two logarithms and a
                // division instead of sixteen and eight
                auto offer_draw = [&](float x_, int index, uint32_t bits) {
                    if ((~bits >> 9) <= bound) offer(x_, index, gumbel_of(bits));
                };
#pragma unroll
                for (int q = 0; q < EPC / 4; ++q) {
                    offer_draw(x[4 * q + 0], c0 + 4 * q + 0, r[q].x);
                    offer_draw(x[4 * q + 1], c0 + 4 * q + 1, r[q].y);
                    offer_draw(x[4 * q + 2], c0 + 4 * q + 2, r[q].z);
                    offer_draw(x[4 * q + 3], c0 + 4 * q + 3, r[q].w);
                }
            } else {
#pragma unroll
                for (int i = 0; i < EPC; ++i) offer(x[i], c0 + i, rn.at(c0 + i));
            }
            if (NOISE == 2) {
                // the wavefront's best so far, to everybody (only when it has grown: few chunks of a row raise it).
                // Only with all 64 lanes still in the loop: on the row's last, partly filled trip the lanes that
                // have left are switched off, a shuffle reads 0 from them, and a 0 published above a row whose
                // noisy logits are all negative would let the others skip the real winner.  Not publishing on
                // that one trip costs nothing (an old lead_seen only makes the skip test more cautious).
                if (__builtin_amdgcn_ballot_w64(best > seen) != 0 && __builtin_amdgcn_ballot_w64(true) == ~0ull) {
                    float wb = best;
#pragma unroll
                    for (int off = 32; off >= 1; off >>= 1) wb = fmaxf(wb, __shfl_xor(wb, off));
                    seen = fmaxf(seen, wb);
                    if ((tid & (mdx::kWave - 1)) == 0) __hip_atomic_fetch_max(&lead_seen, wb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
        }
        lane_softmax_done();
        p.pick = best; p.pick_x = best_x; p.pick_idx = best_idx;
        if (split == 0) {
            for (int64_t e = tid; e < lead; e += kThreads) visit<true>(p, one(e), (int)e, c, T_, noise_at(e));
            for (int64_t e = tail0 + tid; e < vocab; e += kThreads) visit<true>(p, one(e), (int)e, c, T_, noise_at(e));
        }
    }

    // Wavefront reduction, then across the workgroup's wavefronts through LDS.
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const Partial o = shfl_xor(p, off, NOISE != 0);
        combine(p, o, c, NOISE != 0);
    }
    __shared__ Partial wave_part[kThreads / mdx::kWave];
    if ((tid & (mdx::kWave - 1)) == 0) wave_part[tid / mdx::kWave] = p;
    __syncthreads();
    Partial r = wave_part[0];
    if (tid == 0) {
#pragma unroll
        for (int w = 1; w < kThreads / mdx::kWave; ++w) combine(r, wave_part[w], c, NOISE != 0);
    }
    if constexpr (!FLOOR) {
        if (S.arrive) { select_when_last<(NOISE != 0), (sizeof...(LIVE) > 0)>(S, r, (int)row32, split, c, nsplit, partials, x0, x0_p); return; }
    }
    if (tid != 0) return;
    if (nsplit > 1) {
        partials[row * nsplit + split] = r;
    } else {
        int64_t tok; float conf;
        finish_row<(NOISE != 0)>(r, c, tok, conf);
        x0[row] = tok;
        x0_p[row] = conf;
    }
}

template <bool NOISE>
__global__ __launch_bounds__(kThreads) void confidence_finalize_kernel(
    const Partial* __restrict__ partials, int nsplit,
    const float* __restrict__ temperatures, int rows_per_temp,
    int64_t rows, int64_t* __restrict__ x0, float* __restrict__ x0_p)
{
    const int64_t row = (int64_t)blockIdx.x * (kThreads / kMergeLanes) + threadIdx.x / kMergeLanes;
    const int lane16 = threadIdx.x % kMergeLanes;
    if (row >= rows) return;                                 // (whole groups)
    const float c = kLog2e / (temperatures ? temperatures[row / rows_per_temp] : 1.0f);
    const Partial r = merge_splits<NOISE>(partials + row * nsplit, nsplit, lane16, kMergeLanes, c);
    if (lane16 != 0) return;
    int64_t tok; float conf;
    finish_row<NOISE>(r, c, tok, conf);
    x0[row] = tok;
    x0_p[row] = conf;
}

// Where a selection kernel finds the confidences: written by the vocabulary pass, or as row splits that it merges first
// (and then writes x0 / x0_p itself), which saves a launch.
enum Source { kFromRows = 0, kFromSplits = 1, kFromNoisySplits = 2 };
constexpr int kMaxBlockLen = 1024;
constexpr int kMaxSelectThreads = 1024;

// The block's confidences and picks into LDS, merged from the splits where need be; all threads of the workgroup.
template <int SOURCE>
__device__ __forceinline__ void gather_block(float* conf_s, int* pick_s, int64_t* x0, float* x0_p, const Partial* partials, int nsplit,
                                             const float* temperatures, int b, int block_len, int lanes)
{
    const int lane = threadIdx.x & (lanes - 1);
    const float c = kLog2e / (temperatures ? temperatures[b] : 1.0f);
    for (int p = threadIdx.x / lanes; p < block_len; p += blockDim.x / lanes) {
        const int64_t at = (int64_t)b * block_len + p;
        const Partial r = merge_splits<SOURCE == kFromNoisySplits>(partials + at * nsplit, nsplit, lane, lanes, c);
        if (lane == 0) {
            int64_t tok; float conf;
            finish_row<SOURCE == kFromNoisySplits>(r, c, tok, conf);
            x0[at] = tok;
            x0_p[at] = conf;
            pick_s[p] = (int)tok;
            conf_s[p] = conf;
        }
    }
    __syncthreads();
}

// One workgroup per sequence; lane p owns block position p.
template <int SOURCE>
__global__ __launch_bounds__(kMaxBlockLen) void select_transfer_kernel(
    int64_t* __restrict__ x0, float* __restrict__ x0_p, int64_t* __restrict__ tokens,
    const Partial* __restrict__ partials, int nsplit, const float* __restrict__ temperatures,
    int64_t mask_token_id, float threshold, int k,
    uint8_t* __restrict__ transfer, int32_t* __restrict__ count, int block_len, int lanes)
{
    __shared__ float conf_s[kMaxBlockLen];
    __shared__ int pick_s[SOURCE == kFromRows ? 1 : kMaxBlockLen];
    __shared__ int n_hi, n_masked, n_commit;
    const int b = blockIdx.x;
    const int p = threadIdx.x;
    const bool on = p < block_len;
    const int64_t at = (int64_t)b * block_len + p;
    if (p == 0) { n_hi = 0; n_masked = 0; n_commit = 0; }
    int64_t pick = 0;
    float pick_p = 0.f;
    if (SOURCE != kFromRows) {
        gather_block<SOURCE>(conf_s, pick_s, x0, x0_p, partials, nsplit, temperatures, b, block_len, lanes);
        if (on) { pick = pick_s[p]; pick_p = conf_s[p]; }
    } else if (on) {
        pick = x0[at];
        pick_p = x0_p[at];
    }
    __syncthreads();
    const bool masked = on && tokens[at] == mask_token_id;
    const float conf = masked ? pick_p : -INFINITY;
    const bool hi = conf > threshold;
    if (on) conf_s[p] = conf;
    if (hi) atomicAdd(&n_hi, 1);
    if (masked) atomicAdd(&n_masked, 1);
    __syncthreads();
    bool commit;
    if (n_hi >= k) {
        commit = hi;
    } else {
        // rank among masked positions: higher confidence first, lower position first on ties
        int rank = 0;
        if (masked) {
            for (int j = 0; j < block_len; ++j) {
                const float cj = conf_s[j];
                rank += (cj > conf || (cj == conf && j < p)) ? 1 : 0;
            }
        }
        commit = masked && rank < k && conf > -INFINITY;     // at most min(k, n_masked) positions; a confidence of -inf is never committed
    }
    if (on) {
        transfer[at] = commit ? 1 : 0;
        if (commit) {
            tokens[at] = pick;
            atomicAdd(&n_commit, 1);
        }
    }
    __syncthreads();
    if (p == 0) count[b] = n_commit;
}

// The same rule for blocks of up to 64 positions (the engine's blocks hold 32) with ONE wavefront per
// sequence (select_by_wave), so that the launch costs little more than its one round trip to memory.  Where the row splits have to be merged first,
// the sequence gets more lanes per position for that, and its first wavefront goes on alone.
template <int SOURCE>
__global__ __launch_bounds__(kMaxSelectThreads) void select_transfer_wave_kernel(
    int64_t* __restrict__ x0, float* __restrict__ x0_p, const Partial* __restrict__ partials, int nsplit, const float* __restrict__ temperatures,
    const Selection S)
{
    __shared__ float conf_s[SOURCE == kFromRows ? 1 : mdx::kWave];
    __shared__ int pick_s[SOURCE == kFromRows ? 1 : mdx::kWave];
    const int b = blockIdx.x;
    const int p = threadIdx.x;
    const bool on = p < S.block_len;
    const int64_t at = (int64_t)b * S.block_len + p;
    int64_t pick = 0;
    float pick_p = 0.f;
    const int64_t tok = on ? S.tokens[at] : 0;
    if (SOURCE != kFromRows) {
        gather_block<SOURCE>(conf_s, pick_s, x0, x0_p, partials, nsplit, temperatures, b, S.block_len, S.lanes);
        if (p >= mdx::kWave) return;
        if (on) { pick = pick_s[p]; pick_p = conf_s[p]; }
    } else if (on) {
        pick = x0[at];
        pick_p = x0_p[at];
    }
    select_by_wave(S, b, p, on && tok == S.mask_token_id, pick, pick_p);
}

int launch_select(int64_t* x0, float* x0_p, int64_t* tokens, const Partial* partials, int nsplit, bool noisy, const float* temperatures,
                  int64_t mask_token_id, float threshold, int k, uint8_t* transfer, int32_t* count, int bs, int block_len,
                  hipStream_t stream)
{
    const int source = partials == nullptr || nsplit <= 1 ? kFromRows : noisy ? kFromNoisySplits : kFromSplits;
    const int whole_waves = (block_len + mdx::kWave - 1) / mdx::kWave * mdx::kWave;
    // lanes to merge splits with, for as many positions at a time as a workgroup holds
    const int lanes = merge_lanes(nsplit), wanted = (block_len * lanes + mdx::kWave - 1) / mdx::kWave * mdx::kWave;
    const int merging = wanted < kMaxSelectThreads ? wanted : kMaxSelectThreads;
    const unsigned threads = source == kFromRows ? whole_waves : (merging > whole_waves ? merging : whole_waves);
    if (block_len <= mdx::kWave) {
        const Selection S{nullptr, tokens, mask_token_id, threshold, k, transfer, count, block_len, lanes};
        if (source == kFromRows)        select_transfer_wave_kernel<kFromRows><<<(unsigned)bs, threads, 0, stream>>>(x0, x0_p, partials, nsplit, temperatures, S);
        else if (source == kFromSplits) select_transfer_wave_kernel<kFromSplits><<<(unsigned)bs, threads, 0, stream>>>(x0, x0_p, partials, nsplit, temperatures, S);
        else                            select_transfer_wave_kernel<kFromNoisySplits><<<(unsigned)bs, threads, 0, stream>>>(x0, x0_p, partials, nsplit, temperatures, S);
    } else {
#define MDX_SELECT(KERNEL, SOURCE) KERNEL<SOURCE><<<(unsigned)bs, threads, 0, stream>>>( \
        x0, x0_p, tokens, partials, nsplit, temperatures, mask_token_id, threshold, k, transfer, count, block_len, lanes)
        if (source == kFromRows)        MDX_SELECT(select_transfer_kernel, kFromRows);
        else if (source == kFromSplits) MDX_SELECT(select_transfer_kernel, kFromSplits);
        else                            MDX_SELECT(select_transfer_kernel, kFromNoisySplits);
    }
#undef MDX_SELECT
    return mdx::check_launch("select_transfer");
}

// Splits per row so that small batches still fill the chip: target >= 4 workgroups per CU
// while keeping at least 32 KiB of logits per workgroup.
int pick_nsplit(int64_t rows, int64_t vocab) {
    const int64_t target = 1024;
    int64_t n = (target + rows - 1) / rows;
    const int64_t max_by_size = vocab / 16384 > 0 ? vocab / 16384 : 1;
    if (n > max_by_size) n = max_by_size;
    if (n < 1) n = 1;
    if (n > 64) n = 64;
    return (int)n;
}

// With noise from the generator a launch is bound by arithmetic, and lasts as long as the CUs with the most workgroups do:
// among the splits from half of pick_nsplit's on (never more: the workspace is sized for those) the largest that leaves the
// CUs most evenly loaded.  (96 rows: 9 splits put four workgroups on some CUs and three on others, 8 put three on each.)
// With the logarithms of the few draws that passed only, the sampled step at N(0, 3^2), us, before / after both: 32 rows
// 24.1 / 19.6, 96 rows 33.7 / 27.1, 256 rows 53.5 / 45.9, 384 rows 75.6 / 62.1, 1024 rows 139.8 / 128.2.
int pick_nsplit_sampled(int64_t rows, int64_t vocab) {
    const int most = pick_nsplit(rows, vocab);
    const int64_t cus = mdx::compute_units();
    int best = most;
    double best_load = 0;
    for (int n = most; n >= 1 && 2 * n >= most; --n) {
        const double load = (double)((rows * n + cus - 1) / cus) / n;      // the fullest CU's share of the work, up to a constant
        if (best_load == 0 || load < best_load * 0.97) { best = n; best_load = load; }
    }
    return best;
}

template <typename T, bool FLOOR>
int launch_confidence(const void* logits, int64_t row_stride, const float* temperatures, int rows_per_temp,
                      const NoiseSpec& N, const float* floors, int64_t* x0, float* x0_p,
                      int64_t rows, int64_t vocab, int nsplit, Partial* partials, bool finalize, const LiveRows* live, const Selection& S, hipStream_t stream)
{
    const dim3 grid((unsigned)rows, (unsigned)nsplit);
    const bool noisy = N.noise != nullptr || N.philox;
    if constexpr (!FLOOR) {
        if (live) {
#define MDX_CONFIDENCE(NOISE) confidence_argmax_kernel<T, NOISE, false, LiveRows><<<grid, kThreads, 0, stream>>>( \
        *live, (const T*)logits, row_stride, temperatures, rows_per_temp, N, floors, vocab, nsplit, partials, x0, x0_p, S)
            if (N.philox)     MDX_CONFIDENCE(2);
            else if (N.noise) MDX_CONFIDENCE(1);
            else              MDX_CONFIDENCE(0);
#undef MDX_CONFIDENCE
            return mdx::check_launch("confidence_argmax");
        }
    }
#define MDX_CONFIDENCE(NOISE) confidence_argmax_kernel<T, NOISE, FLOOR><<<grid, kThreads, 0, stream>>>( \
        (const T*)logits, row_stride, temperatures, rows_per_temp, N, floors, vocab, nsplit, partials, x0, x0_p, S)
    if (N.philox)     MDX_CONFIDENCE(2);
    else if (N.noise) MDX_CONFIDENCE(1);
    else              MDX_CONFIDENCE(0);
#undef MDX_CONFIDENCE
    int rc = mdx::check_launch("confidence_argmax");
    if (rc != MDX_OK || nsplit == 1 || !finalize) return rc;
    const unsigned fgrid = (unsigned)((rows + kThreads / kMergeLanes - 1) / (kThreads / kMergeLanes));
    if (noisy)
        confidence_finalize_kernel<true><<<fgrid, kThreads, 0, stream>>>(partials, nsplit, temperatures, rows_per_temp, rows, x0, x0_p);
    else
        confidence_finalize_kernel<false><<<fgrid, kThreads, 0, stream>>>(partials, nsplit, temperatures, rows_per_temp, rows, x0, x0_p);
    return mdx::check_launch("confidence_finalize");
}

// The noise tensor that the generator stands for, written out: [rows, vocab] fp32.
__global__ __launch_bounds__(kThreads) void gumbel_noise_kernel(float* __restrict__ out, int64_t out_row_stride, int64_t vocab, const NoiseSpec N)
{
    const int64_t row = blockIdx.y;
    const RowNoise rn = row_noise(N, row);
    const int64_t group = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (group * 4 >= vocab) return;
    const U4 r = rn.group((uint32_t)group);
    const uint32_t b[4] = {r.x, r.y, r.z, r.w};
    float* dst = out + row * out_row_stride + group * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (group * 4 + i < vocab) dst[i] = gumbel_of(b[i]);
}

}  // namespace

extern "C" int64_t mdx_confidence_argmax_workspace_bytes(int64_t rows, int64_t vocab) {
    if (rows <= 0 || vocab <= 0) return 0;
    const int nsplit = pick_nsplit(rows, vocab);
    return nsplit > 1 ? rows * nsplit * (int64_t)sizeof(Partial) : 0;
}

namespace {

int confidence_pass(const void* logits, int64_t row_stride, int32_t dtype,
                    const float* temperatures, int32_t rows_per_temp,
                    const NoiseSpec& N, const float* floors,
                    int64_t* x0, float* x0_p, int64_t rows, int64_t vocab,
                    void* workspace, int64_t workspace_bytes, bool finalize, int* nsplit_out, hipStream_t stream,
                    const LiveRows* live = nullptr, int n_live = 0, Selection* select = nullptr)
{
    MDX_REQUIRE(rows >= 0 && vocab >= 0, MDX_EINVAL, "confidence_argmax: negative size");
    if (nsplit_out) *nsplit_out = 1;
    if (rows == 0) return MDX_OK;
    MDX_REQUIRE(vocab > 0, MDX_EINVAL, "confidence_argmax: empty vocabulary");
    MDX_REQUIRE(logits && x0 && x0_p, MDX_EINVAL, "confidence_argmax: null pointer");
    MDX_REQUIRE(vocab < (int64_t)0x7fffffff && rows < (int64_t)0x7fffffff, MDX_EUNSUPPORTED,
                "confidence_argmax: rows %lld or vocab %lld out of range", (long long)rows, (long long)vocab);
    MDX_REQUIRE(row_stride >= vocab, MDX_EUNSUPPORTED, "confidence_argmax: row_stride %lld < vocab %lld", (long long)row_stride, (long long)vocab);
    MDX_REQUIRE(!temperatures || rows_per_temp > 0, MDX_EINVAL, "confidence_argmax: rows_per_temp must be positive");
    MDX_REQUIRE(!N.noise || N.noise_row_stride >= vocab, MDX_EINVAL, "confidence_argmax: noise_row_stride < vocab");
    const int esz = dtype == MDX_F32 ? 4 : 2;
    MDX_REQUIRE((reinterpret_cast<uintptr_t>(logits) % esz) == 0, MDX_EUNSUPPORTED, "confidence_argmax: logits not element-aligned");
    const int64_t asked = live ? n_live : rows;
    if (asked == 0) return MDX_OK;
    const int nsplit = N.philox ? pick_nsplit_sampled(asked, vocab) : pick_nsplit(asked, vocab);
    if (nsplit_out) *nsplit_out = nsplit;
    const int64_t need = nsplit > 1 ? rows * nsplit * (int64_t)sizeof(Partial) : 0;
    MDX_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), MDX_EWORKSPACE,
                "confidence_argmax: workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
    Partial* partials = static_cast<Partial*>(workspace);
    Selection S{};
    if (select) { S = *select; S.lanes = merge_lanes(nsplit); }
#define MDX_PASS(T, FLOOR) launch_confidence<T, FLOOR>(logits, row_stride, temperatures, rows_per_temp, N, floors, x0, x0_p, asked, vocab, nsplit, partials, finalize, live, S, stream)
    switch (dtype) {
        case MDX_BF16: return floors ? MDX_PASS(__bf16, true) : MDX_PASS(__bf16, false);
        case MDX_F16:  return floors ? MDX_PASS(__half, true) : MDX_PASS(__half, false);
        case MDX_F32:  return MDX_PASS(float, false);                  // (filters take 16-bit logits only)
        default: return mdx::fail(MDX_EUNSUPPORTED, "confidence_argmax: dtype %d", dtype);
    }
#undef MDX_PASS
}

}  // namespace

extern "C" int mdx_confidence_argmax(const void* logits, int64_t row_stride, int32_t dtype,
                                     const float* temperatures, int32_t rows_per_temp,
                                     const float* noise, int64_t noise_row_stride,
                                     int64_t* x0, float* x0_p, int64_t rows, int64_t vocab,
                                     void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return confidence_pass(logits, row_stride, dtype, temperatures, rows_per_temp, tensor_noise(noise, noise_row_stride), nullptr, x0, x0_p,
                           rows, vocab, workspace, workspace_bytes, true, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int mdx_confidence_argmax_gumbel(const void* logits, int64_t row_stride, int32_t dtype,
                                            const float* temperatures, int32_t rows_per_temp,
                                            uint64_t seed, uint64_t offset, const int64_t* offset_dev, const int64_t* row_ids,
                                            int64_t* x0, float* x0_p, int64_t rows, int64_t vocab,
                                            void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return confidence_pass(logits, row_stride, dtype, temperatures, rows_per_temp, generator_noise(seed, offset, offset_dev, row_ids), nullptr,
                           x0, x0_p, rows, vocab, workspace, workspace_bytes, true, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int mdx_gumbel_noise(float* noise, int64_t noise_row_stride, int64_t rows, int64_t vocab,
                                uint64_t seed, uint64_t offset, const int64_t* offset_dev, const int64_t* row_ids,
                                mdx_stream_t stream)
{
    MDX_REQUIRE(rows >= 0 && vocab >= 0, MDX_EINVAL, "gumbel_noise: negative size");
    if (rows == 0 || vocab == 0) return MDX_OK;
    MDX_REQUIRE(noise, MDX_EINVAL, "gumbel_noise: null pointer");
    MDX_REQUIRE(noise_row_stride >= vocab, MDX_EINVAL, "gumbel_noise: noise_row_stride < vocab");
    MDX_REQUIRE(vocab < (int64_t)0x7fffffff && rows <= 65535, MDX_EUNSUPPORTED,
                "gumbel_noise: rows %lld (max 65535) or vocab %lld out of range", (long long)rows, (long long)vocab);
    const dim3 grid((unsigned)(((vocab + 3) / 4 + kThreads - 1) / kThreads), (unsigned)rows);
    gumbel_noise_kernel<<<grid, kThreads, 0, static_cast<hipStream_t>(stream)>>>(noise, noise_row_stride, vocab,
                                                                                 generator_noise(seed, offset, offset_dev, row_ids));
    return mdx::check_launch("gumbel_noise");
}

extern "C" int mdx_select_transfer(const int64_t* x0, const float* x0_p, int64_t* tokens,
                                   int64_t mask_token_id, float threshold, int32_t k,
                                   uint8_t* transfer, int32_t* count,
                                   int32_t bs, int32_t block_len, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(bs >= 0 && block_len >= 0, MDX_EINVAL, "select_transfer: negative size");
    if (bs == 0 || block_len == 0) return MDX_OK;
    MDX_REQUIRE(x0 && x0_p && tokens && transfer && count, MDX_EINVAL, "select_transfer: null pointer");
    MDX_REQUIRE(block_len <= kMaxBlockLen, MDX_EUNSUPPORTED, "select_transfer: block_len %d > %d", block_len, kMaxBlockLen);
    MDX_REQUIRE(k >= 0, MDX_EINVAL, "select_transfer: k %d < 0", k);
    return launch_select(const_cast<int64_t*>(x0), const_cast<float*>(x0_p), tokens, nullptr, 1, false, nullptr, mask_token_id, threshold, k,
                         transfer, count, bs, block_len, stream);
}

namespace {

// Whether the vocabulary pass of so many rows better selects by itself.  Not where the rows are many and short: the ends of the workgroups, three trips to memory, then hold up those
// that wait for their place (blocks of 32, us on the GPU, two launches / one: 200 blocks of 1000 entries 14.6 / 16.9, of 16 000 40.2 / 41.5, 64 of 1000 sampled 13.3 / 15.1; 64 of 4000
// 9.9 / 9.9, of 151 936 100.8 / 99.1).  Nor where a counter has more arrivals than the pass itself covers (151 936 entries in 9 splits: 1 block of 32, 288 arrivals, 9.6 / 12.6, 2 10.8 / 13.1,
// 3 12.3 / 14.0; of 64, 576, 10.9 / 18.2; in 8, 256 arrivals, 4 blocks of 32 12.4 / 12.2); draws take longer than their arrivals (1 block of 32 18.5 / 17.8, of 64 21.7 / 20.6).
// Elsewhere: 8 blocks of 32 18.5 / 18.2, 16 30.0 / 29.3, 32 51.8 / 51.4; 64 000 entries 1 block 9.2 / 9.5, and with the host's part, which the step of few rows waits for, 11.4 / 9.3.
constexpr int kMostArrivals = 256, kFewRows = 1024, kManyRows = 2048, kShortRow = 4096;
bool one_launch_pays(int64_t rows, int32_t block_len, int64_t vocab, bool seeded)
{
    if (rows < 1 || rows > kManyRows || (rows > kFewRows && vocab < kShortRow)) return false;
    return seeded || (int64_t)block_len * pick_nsplit(rows, vocab) <= kMostArrivals;
}

}  // namespace

extern "C" int32_t mdx_unmask_step_single_launch_pays(int32_t bs, int32_t block_len, int64_t vocab, int32_t seeded)
{
    return bs > 0 && block_len > 0 && block_len <= mdx::kWave && vocab > 0 && one_launch_pays((int64_t)bs * block_len, block_len, vocab, seeded != 0);
}

extern "C" int64_t mdx_unmask_step_counter_bytes(int32_t bs, int32_t block_len)
{
    if (bs <= 0 || block_len <= 0) return 0;
    return (int64_t)bs * kCounterWords * (int64_t)sizeof(uint32_t);
}

namespace {

int unmask_step_impl(const void* logits, int64_t row_stride, int32_t dtype,
                     const float* temperatures, const NoiseSpec& N,
                     int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                     int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count,
                     int32_t bs, int32_t block_len, int64_t vocab, void* workspace, int64_t workspace_bytes,
                     void* counters, int64_t counter_bytes, hipStream_t stream, const LiveRows* live = nullptr, int n_live = 0)
{
    MDX_REQUIRE(bs >= 0 && block_len >= 0, MDX_EINVAL, "unmask_step: negative size");
    MDX_REQUIRE(k >= 0, MDX_EINVAL, "unmask_step: k %d < 0", k);
    MDX_REQUIRE(block_len <= kMaxBlockLen, MDX_EUNSUPPORTED, "unmask_step: block_len %d > %d", block_len, kMaxBlockLen);
    if (bs == 0 || block_len == 0) return MDX_OK;
    MDX_REQUIRE(tokens && transfer && count, MDX_EINVAL, "unmask_step: null pointer");
    // With counters the last workgroup of a sequence selects; otherwise the selection kernel merges the row splits itself (one launch fewer).
    const bool noisy = N.noise != nullptr || N.philox;
    const bool single = counters && ((uintptr_t)counters & 3) == 0 && counter_bytes >= mdx_unmask_step_counter_bytes(bs, block_len) && block_len <= mdx::kWave && vocab > 0;
    uint32_t* const arrive = static_cast<uint32_t*>(counters);
    Selection S{arrive, tokens, mask_token_id, threshold, k, transfer, count, block_len, 1};
    int nsplit = 1;
    int rc = confidence_pass(logits, row_stride, dtype, temperatures, block_len, N, nullptr, x0, x0_p, (int64_t)bs * block_len, vocab,
                             workspace, workspace_bytes, false, &nsplit, stream, live, n_live, single ? &S : nullptr);
    if (rc != MDX_OK || single) return rc;
    // (rows that were not asked for: whatever was there, of positions that are not masked and so in no race)
    return launch_select(x0, x0_p, tokens, nsplit > 1 ? static_cast<const Partial*>(workspace) : nullptr, nsplit, noisy, temperatures,
                         mask_token_id, threshold, k, transfer, count, bs, block_len, stream);
}

// What a filtered step keeps in the caller's workspace: the row floors and the vocabulary pass's splits, or the candidates.
int64_t filtered_workspace(int64_t rows, int64_t vocab, int top_k) {
    const int64_t lists = mdx::filtered_pick_workspace_bytes(rows, vocab, top_k);
    return lists > 0 ? lists : (rows * 4 + 15) / 16 * 16 + mdx_confidence_argmax_workspace_bytes(rows, vocab);
}

}  // namespace

extern "C" int64_t mdx_unmask_step_filtered_workspace_bytes(int64_t rows, int64_t vocab, int32_t top_k)
{
    return rows <= 0 || vocab <= 0 ? 0 : filtered_workspace(rows, vocab, top_k);
}

extern "C" int mdx_unmask_step_filtered(const void* logits, int64_t row_stride, int32_t dtype,
                                        const float* temperatures, int32_t top_k, float top_p,
                                        const float* noise, int64_t noise_row_stride,
                                        int32_t seeded, uint64_t seed, uint64_t offset, const int64_t* offset_dev,
                                        int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                                        int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count,
                                        int32_t bs, int32_t block_len, int64_t vocab,
                                        void* workspace, int64_t workspace_bytes, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MDX_REQUIRE(bs >= 0 && block_len >= 0, MDX_EINVAL, "unmask_step: negative size");
    MDX_REQUIRE(k >= 0, MDX_EINVAL, "unmask_step: k %d < 0", k);
    MDX_REQUIRE(block_len <= kMaxBlockLen, MDX_EUNSUPPORTED, "unmask_step: block_len %d > %d", block_len, kMaxBlockLen);
    const int64_t rows = (int64_t)bs * block_len;
    int rc = mdx::check_filter(logits, row_stride, dtype, top_k, top_p, rows, vocab);
    if (rc != MDX_OK || rows == 0) return rc;
    MDX_REQUIRE(tokens && transfer && count && x0 && x0_p, MDX_EINVAL, "unmask_step: null pointer");
    MDX_REQUIRE(!(noise && seeded), MDX_EINVAL, "unmask_step: either a noise tensor or a seed");
    MDX_REQUIRE(!noise || noise_row_stride >= vocab, MDX_EINVAL, "unmask_step: noise_row_stride < vocab");
    const int64_t need = filtered_workspace(rows, vocab, top_k);
    MDX_REQUIRE(workspace && workspace_bytes >= need && mdx::aligned16(workspace), MDX_EWORKSPACE,
                "unmask_step: workspace of %lld bytes needed (16-byte aligned), %lld given", (long long)need, (long long)workspace_bytes);
    const NoiseSpec N = seeded ? generator_noise(seed, offset, offset_dev, nullptr) : tensor_noise(noise, noise_row_stride);
    if (mdx::filtered_pick_workspace_bytes(rows, vocab, top_k) > 0) {
        rc = mdx::filtered_pick(logits, row_stride, dtype, temperatures, block_len, top_k, top_p, N, x0, x0_p, rows, vocab, workspace, stream);
        if (rc != MDX_OK) return rc;
        return launch_select(x0, x0_p, tokens, nullptr, 1, false, nullptr, mask_token_id, threshold, k, transfer, count, bs, block_len, stream);
    }
    float* floors = static_cast<float*>(workspace);
    rc = mdx::filter_floors(logits, row_stride, dtype, temperatures, block_len, top_k, top_p, floors, rows, vocab, stream);
    if (rc != MDX_OK) return rc;
    const int64_t at = (rows * 4 + 15) / 16 * 16;
    void* splits = static_cast<char*>(workspace) + at;
    int nsplit = 1;
    rc = confidence_pass(logits, row_stride, dtype, temperatures, block_len, N, floors, x0, x0_p, rows, vocab, splits, workspace_bytes - at,
                         false, &nsplit, stream);
    if (rc != MDX_OK) return rc;
    return launch_select(x0, x0_p, tokens, nsplit > 1 ? static_cast<const Partial*>(splits) : nullptr, nsplit, N.noise || N.philox, temperatures,
                         mask_token_id, threshold, k, transfer, count, bs, block_len, stream);
}

extern "C" int mdx_unmask_step(const void* logits, int64_t row_stride, int32_t dtype,
                               const float* temperatures, const float* noise, int64_t noise_row_stride,
                               int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                               int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count,
                               int32_t bs, int32_t block_len, int64_t vocab,
                               void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return unmask_step_impl(logits, row_stride, dtype, temperatures, tensor_noise(noise, noise_row_stride), tokens, mask_token_id,
                            threshold, k, x0, x0_p, transfer, count, bs, block_len, vocab, workspace, workspace_bytes, nullptr, 0,
                            static_cast<hipStream_t>(stream));
}

extern "C" int mdx_unmask_step_gumbel(const void* logits, int64_t row_stride, int32_t dtype,
                                      const float* temperatures,
                                      uint64_t seed, uint64_t offset, const int64_t* offset_dev, const int64_t* row_ids,
                                      int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                                      int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count,
                                      int32_t bs, int32_t block_len, int64_t vocab,
                                      void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return unmask_step_impl(logits, row_stride, dtype, temperatures, generator_noise(seed, offset, offset_dev, row_ids), tokens,
                            mask_token_id, threshold, k, x0, x0_p, transfer, count, bs, block_len, vocab, workspace, workspace_bytes, nullptr, 0,
                            static_cast<hipStream_t>(stream));
}

extern "C" int mdx_unmask_step_single_launch(const void* logits, int64_t row_stride, int32_t dtype,
                                             const float* temperatures, const float* noise, int64_t noise_row_stride,
                                             int32_t seeded, uint64_t seed, uint64_t offset, const int64_t* offset_dev,
                                             int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                                             int64_t* x0, float* x0_p, uint8_t* transfer, int32_t* count,
                                             int32_t bs, int32_t block_len, int64_t vocab,
                                             void* workspace, int64_t workspace_bytes, void* counters, int64_t counter_bytes, mdx_stream_t stream)
{
    MDX_REQUIRE(!(noise && seeded), MDX_EINVAL, "unmask_step: either a noise tensor or a seed");
    const NoiseSpec N = seeded ? generator_noise(seed, offset, offset_dev, nullptr) : tensor_noise(noise, noise_row_stride);
    return unmask_step_impl(logits, row_stride, dtype, temperatures, N, tokens, mask_token_id, threshold, k, x0, x0_p, transfer, count, bs, block_len,
                            vocab, workspace, workspace_bytes, counters, counter_bytes, static_cast<hipStream_t>(stream));
}

constexpr int kSingleLaunchRows = 128;

// What the step keeps in the caller's workspace: x0, x0_p, and the splits of as many rows as there are, by the most splits that fewer rows are cut into.
namespace {
int64_t confidences_bytes(int64_t rows) { return (rows * 12 + 15) / 16 * 16; }
}

extern "C" int64_t mdx_unmask_step_host_blocks_workspace_bytes(int64_t rows, int64_t vocab)
{
    return rows <= 0 || vocab <= 0 ? 0 : confidences_bytes(rows) + rows * pick_nsplit(1, vocab) * (int64_t)sizeof(Partial);
}

extern "C" int64_t mdx_unmask_step_host_blocks_counter_bytes(int32_t bs, int32_t block_len)
{
    return (int64_t)bs * block_len < kSingleLaunchRows || (int64_t)bs * block_len > kManyRows ? 0 : mdx_unmask_step_counter_bytes(bs, block_len);
}

extern "C" int mdx_unmask_step_host_blocks_single_launch(const void* logits, int64_t row_stride, int32_t dtype,
                                                         const float* temperatures, const float* noise, int64_t noise_row_stride,
                                                         int32_t seeded, uint64_t seed, uint64_t offset, const int64_t* offset_dev,
                                                         int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                                                         uint8_t* transfer, int32_t* count, int32_t bs, int32_t block_len, int64_t vocab,
                                                         void* workspace, int64_t workspace_bytes, void* counters, int64_t counter_bytes,
                                                         mdx_stream_t stream)
{
    MDX_REQUIRE(bs >= 0 && block_len >= 0, MDX_EINVAL, "unmask_step: negative size");
    if (bs == 0 || block_len == 0) return MDX_OK;
    const int64_t rows = (int64_t)bs * block_len, need = mdx_unmask_step_host_blocks_workspace_bytes(rows, vocab);
    MDX_REQUIRE(tokens, MDX_EINVAL, "unmask_step: null pointer");
    MDX_REQUIRE(!(noise && seeded), MDX_EINVAL, "unmask_step: either a noise tensor or a seed");
    MDX_REQUIRE(workspace && workspace_bytes >= need && mdx::aligned16(workspace), MDX_EWORKSPACE,
                "unmask_step: workspace of %lld bytes needed (16-byte aligned), %lld given", (long long)need, (long long)workspace_bytes);
    // The masked positions are known here, and no other row's confidence reaches a result: a row is 304 KB of reads and 150 000 draws.  The sampler's
    // call, us, all rows / masked rows (three quarters): sampled, 1 sequence 36.3 / 34.6, 3 43.4 / 40.0, 8 63.1 / 57.9, 24 118.4 / 106.2; plain, 3 30.4 / 28.2, 24 73.9 / 65.4.
    LiveRows live;
    int n_live = 0, with_rows = 0;                           // masked rows, and the sequences that have any
    if (rows <= kMaxLiveRows) {
        for (int32_t b = 0; b < bs; ++b) {
            const int before = n_live;
            for (int64_t i = (int64_t)b * block_len; i < (int64_t)(b + 1) * block_len; ++i)
                if (tokens[i] == mask_token_id) live.row[n_live++] = (uint16_t)i;
            with_rows += n_live > before;
        }
        // Nobody would select for the sequences without any; and a caller that waits for the result does not see what a launch costs the host, so that few
        // rows are as quick in two (us, two launches / one: 32 rows 24.5 / 26, 96 40.8 / 41.0, 192 36.1 / 35.4, 576 63.1 / 62.7).
        if (with_rows < bs || n_live < kSingleLaunchRows) counters = nullptr;
    }
    if (!one_launch_pays(rows <= kMaxLiveRows ? n_live : rows, block_len, vocab, seeded != 0)) counters = nullptr;
    const NoiseSpec N = seeded ? generator_noise(seed, offset, offset_dev, nullptr) : tensor_noise(noise, noise_row_stride);
    int64_t* x0 = static_cast<int64_t*>(workspace);
    char* splits = static_cast<char*>(workspace) + confidences_bytes(rows);
    return unmask_step_impl(logits, row_stride, dtype, temperatures, N, tokens, mask_token_id, threshold, k, x0, reinterpret_cast<float*>(x0 + rows), transfer, count,
                            bs, block_len, vocab, splits, workspace_bytes - confidences_bytes(rows), counters, counter_bytes, static_cast<hipStream_t>(stream),
                            rows <= kMaxLiveRows && n_live < rows ? &live : nullptr, n_live);
}

extern "C" int mdx_unmask_step_host_blocks(const void* logits, int64_t row_stride, int32_t dtype,
                                           const float* temperatures, const float* noise, int64_t noise_row_stride,
                                           int32_t seeded, uint64_t seed, uint64_t offset, const int64_t* offset_dev,
                                           int64_t* tokens, int64_t mask_token_id, float threshold, int32_t k,
                                           uint8_t* transfer, int32_t* count, int32_t bs, int32_t block_len, int64_t vocab,
                                           void* workspace, int64_t workspace_bytes, mdx_stream_t stream)
{
    return mdx_unmask_step_host_blocks_single_launch(logits, row_stride, dtype, temperatures, noise, noise_row_stride, seeded, seed, offset, offset_dev,
                                                     tokens, mask_token_id, threshold, k, transfer, count, bs, block_len, vocab, workspace, workspace_bytes,
                                                     nullptr, 0, stream);
}
