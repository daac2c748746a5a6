// The unmask step's confidence and pick behind a top-k (and top-p) filter, from one pass over the logits.
//
// A top-k keeps a handful of a row's elements, and everything that follows -- the k-th largest value, the cumulative
// probability, the softmax, the noise and the pick -- needs those alone.  So the filtered copy of the logits that
// modeling_mineru_diffusion.py:585-615 samples from is never written:
//
//   1. topk_candidates_kernel (rows x splits): a workgroup loads its part of the row once, into registers (all loads in
//      flight together), and takes the k-th largest of its threads' largest elements as a threshold: k elements reach it,
//      so it is at most the k-th largest of the part, and few more do (a thread holds a second one rarely).  What reaches
//      it goes to the part's candidate list.  Bound by the one read of the logits.
//   2. filtered_pick_kernel (a workgroup per row): the candidates of the row's parts in the registers of one wavefront;
//      the k-th largest key and the top-p cut-off by bisection over the 16 bits of a key, a ballot or a sum per bit (what the top-k
//      keeps, if up to 64, moved to one element per lane in between); then the softmax over what is kept and the noisy argmax, with noise drawn for the kept elements only.
//
// 384 rows of 151 936, top-k 50, top-p 0.9, sampled: 157 us of filter, 36 of vocabulary pass and 5 of merge before, in
// three passes over the logits or more.  A row whose ties at the threshold outrun its list (constant rows) is done over by the four
// wavefronts of its second workgroup, pass by pass.
#include "logit_keys.h"
#include "filtered_pick.h"
#include <type_traits>

namespace {

using namespace mdx_keys;
using namespace mdx_noise;

typedef short s16x2 __attribute__((ext_vector_type(2)));

constexpr int kChunksPerThread = 10;     // 16-byte chunks of the row that a thread holds in registers
constexpr int kMaxCandidates = 2048;     // of a row: what the second kernel holds
constexpr int kPickThreads = 256;

// Bits -> signed order (an involution: the sign bit stays); -0 becomes -1, just below 0.
__device__ __forceinline__ s16x2 ordered(uint32_t w) {
    const s16x2 b = __builtin_bit_cast(s16x2, w);
    return b ^ ((b >> 15) & s16x2{0x7fff, 0x7fff});
}

// The largest key (of 16 bits) that at least `want` of the wavefront's n x 64 keys reach; 0 if fewer keys than that are nonzero.  Bit by bit, below those that all nonzero keys have in
// common: what a top-k lists lies within a factor of two or four, 8 or 9 bits of bf16.  (Us, all 16 bits / so: 12 sequences, top-k 50 32.5 / 31.6, three 18.7 / 18.0, one 15.7 /
// 14.7, top-k 400 53.3 / 52.1; fp16 keys spread wider, top-k 400 of six 42.4 / 42.6.  Two bits at a time, three counts beside each other: 32.5 / 33.2.)
template <int N> __device__ __forceinline__ uint32_t kth_key(const uint32_t (&key)[N], int want) {
    uint32_t hi = 0, lo = 0xffff;
    int n = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        hi = max(hi, key[i]);
        lo = min(lo, key[i] ? key[i] : 0xffffu);
        n += __popcll(__ballot(key[i] != 0));
    }
    if (n < want) return 0;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) { hi = max(hi, mdx::xor_lanes(hi, off)); lo = min(lo, mdx::xor_lanes(lo, off)); }
    hi = __builtin_amdgcn_readfirstlane(hi);
    lo = __builtin_amdgcn_readfirstlane(lo);
    const int bits = hi == lo ? 0 : 32 - __builtin_clz(hi ^ lo);             // below them all keys are alike
    uint32_t t = hi >> bits << bits;
    for (int bit = bits - 1; bit >= 0; --bit) {
        const uint32_t trial = t | (1u << bit);
        int reached = 0;
#pragma unroll
        for (int i = 0; i < N; ++i) reached += __popcll(__ballot(key[i] >= trial));
        if (reached >= want) t = trial;
    }
    return t;
}

// lists: [rows, nsplit, cap] of (key, column); counts: [rows, nsplit], larger than cap where the list overflowed.
// Held to 64 registers, eight wavefronts per SIMD: four workgroups of 512 threads per CU, two of 1024.  It takes 65 otherwise, and
// then only three, or one, read their rows while the others search and scan.  Whole step of 384 rows, top-k 50 and top-p 0.9: 35.0 ->
// 33.9 us; top-k 400: 68.2 -> 55.6; 1024 rows, top-k 50: 67.5 -> 65.8; 32 rows, which the chip holds at once, 17.6 and 17.5.
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS, 8) void topk_candidates_kernel(
    const uint16_t* __restrict__ logits, int64_t row_stride, int vocab, int top_k, int nsplit, int cap,
    uint2* __restrict__ lists, int* __restrict__ counts)
{
    __shared__ uint16_t largest[THREADS];
    __shared__ int n_found, threshold;
    const int tid = threadIdx.x, split = blockIdx.y;
    const int64_t r = blockIdx.x;
    const RowView row = row_view(logits + r * row_stride, vocab);
    const int per_split = mdx::quotient(row.nchunk + nsplit - 1, nsplit);               // <= THREADS * kChunksPerThread (the host's split)
    const int cbeg = split * per_split, cend = min(row.nchunk, cbeg + per_split);
    constexpr uint32_t kNothing = Bits16<T>::kNegInf | (Bits16<T>::kNegInf << 16);

    u32x4 held[kChunksPerThread];
#pragma unroll
    for (int i = 0; i < kChunksPerThread; ++i) {
        const int ch = cbeg + tid + i * THREADS;
        held[i] = ch < cend ? __builtin_nontemporal_load(row.chunks + ch) : u32x4{kNothing, kNothing, kNothing, kNothing};
    }
    if (tid == 0) n_found = 0;
    s16x2 most = s16x2{-32768, -32768};
#pragma unroll
    for (int i = 0; i < kChunksPerThread; ++i) {
        const uint32_t w[4] = {held[i].x, held[i].y, held[i].z, held[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) most = __builtin_elementwise_max(most, ordered(w[j]));
    }
    largest[tid] = (uint16_t)((int)max(most.x, most.y) + 32768);
    __syncthreads();
    const int neg_inf = (int)(int16_t)(Bits16<T>::kNegInf ^ 0x7fffu) + 32768;                  // its place in the order: never a candidate
    if (tid < 64) {
        uint32_t key[THREADS / 64];
#pragma unroll
        for (int i = 0; i < THREADS / 64; ++i) key[i] = largest[tid + 64 * i];
        const int t = max((int)kth_key(key, top_k), neg_inf + 1);
        if (tid == 0) threshold = (t == 32768 ? 32767 : t) - 32768;                            // (+0 and -0 are one value)
    }
    __syncthreads();
    const int t = threshold;
    uint2* list = lists + (r * nsplit + split) * cap;
    auto offer = [&](int s, int column) {
        if (s < t) return;
        const int at = atomicAdd(&n_found, 1);
        if (at < cap) list[at] = uint2{(uint32_t)((s == -1 ? 0 : s) + 32768), (uint32_t)column};
    };
#pragma unroll
    for (int i = 0; i < kChunksPerThread; ++i) {
        const uint32_t w[4] = {held[i].x, held[i].y, held[i].z, held[i].w};
        s16x2 s[4];
        s16x2 cm = s16x2{-32768, -32768};
#pragma unroll
        for (int j = 0; j < 4; ++j) { s[j] = ordered(w[j]); cm = __builtin_elementwise_max(cm, s[j]); }
        if (max((int)cm.x, (int)cm.y) < t) continue;
        const int column = row.lead + 8 * (cbeg + tid + i * THREADS);
#pragma unroll
        for (int j = 0; j < 4; ++j) { offer(s[j].x, column + 2 * j); offer(s[j].y, column + 2 * j + 1); }
    }
    if (split == 0) {                     // unaligned head and tail, a handful of elements: candidates whatever the threshold
        auto edge = [&](int e) {
            const int s = (int)(int16_t)row.p[e], o = s ^ ((s >> 15) & 0x7fff);
            if (o + 32768 <= neg_inf) return;
            const int at = atomicAdd(&n_found, 1);
            if (at < cap) list[at] = uint2{(uint32_t)((o == -1 ? 0 : o) + 32768), (uint32_t)e};
        };
        if (tid < row.lead) edge(tid);
        if (tid < vocab - row.tail0) edge(row.tail0 + tid);
    }
    __syncthreads();
    if (tid == 0) counts[r * nsplit + split] = n_found;
}

struct Pick { float v, x; int column; };                                     // best noisy logit, the logit itself, its first column
__device__ __forceinline__ void better(Pick& a, float v, float x, int column) {
    if (v > a.v || (v == a.v && column < a.column)) { a.v = v; a.x = x; a.column = column; }
}
__device__ __forceinline__ Pick wave_best(Pick p) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float v = mdx::xor_lanes(p.v, off), x = mdx::xor_lanes(p.x, off);
        const int column = mdx::xor_lanes(p.column, off);
        better(p, v, x, column);
    }
    return p;
}

// What is drawn on top of an element: nothing (0), a tensor's value (1), the generator's (2); v = x / T + g by a true division
// (skipped, not approximated, when T = 1), as in the unfiltered pass.
template <int NOISE> struct Drawn {
    const float* np; RowNoise rn; float T; bool unit_T;
    __device__ __forceinline__ float operator()(float x, int column) const {
        if (NOISE == 0) return x;
        return (unit_T ? x : x / T) + (NOISE == 1 ? np[column] : rn.at(column));
    }
};

// A wavefront's words in falling order over the lanes (a bitonic network in the vector unit).
__device__ __forceinline__ uint32_t sorted_down(uint32_t word) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1)
#pragma unroll
        for (int stride = size / 2; stride >= 1; stride >>= 1) {
            const uint32_t other = mdx::xor_lanes(word, stride);
            const bool larger = ((lane & stride) == 0) == ((lane & size) == 0);
            word = larger ? max(word, other) : min(word, other);
        }
    return word;
}
// The sum over the lanes up to this one.
__device__ __forceinline__ Mass running_total(Mass v) {
    auto add = [&](auto control, auto rows) {
        constexpr int C = decltype(control)::value, R = decltype(rows)::value;
        const uint32_t lo = __builtin_amdgcn_update_dpp(0, (uint32_t)v, C, R, 0xf, false), hi = __builtin_amdgcn_update_dpp(0, (uint32_t)(v >> 32), C, R, 0xf, false);
        v += ((Mass)hi << 32) | lo;
    };
    add(std::integral_constant<int, 0x111>(), std::integral_constant<int, 0xf>());        // row_shr:1, 2, 4, 8
    add(std::integral_constant<int, 0x112>(), std::integral_constant<int, 0xf>());
    add(std::integral_constant<int, 0x114>(), std::integral_constant<int, 0xf>());
    add(std::integral_constant<int, 0x118>(), std::integral_constant<int, 0xf>());
    add(std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xa>());        // row_bcast:15 into rows 1 and 3
    add(std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xc>());        // row_bcast:31 into rows 2 and 3
    return v;
}

// One wavefront: token and confidence from the elements that the top-k has kept, N per lane (key 0: none).
template <typename T, int NOISE, int N>
__device__ __forceinline__ void pick_from_kept(uint32_t (&key)[N], const int (&column)[N], float top_p, float c, const Drawn<NOISE>& drawn, int64_t& x0, float& x0_p)
{
    uint32_t mk = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) mk = max(mk, key[i]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mk = max(mk, (uint32_t)mdx::xor_lanes((int)mk, off));
    if (mk == 0) { x0 = 0; x0_p = 0.f; return; }                            // no finite logit
    const float m = value_of_key<T>(mk);
    // The kept elements come in no order, so their masses are summed in fixed point: the same logits give the same cut-off and
    // the same confidence, whichever wavefront listed its candidates first.  (384 rows, top-k 50, top-p 0.9: 35.0 -> 35.3 us.)
    const bool fixed = has_masses(m, c);
    Mass mass[N], total = 0;
    float plain = 0.f;                                                       // (no fixed point for what is not at most 1: all but always NaN)
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float term = key[i] ? __builtin_amdgcn_exp2f((value_of_key<T>(key[i]) - m) * c) : 0.f;
        mass[i] = mass_of(term);
        total += mass[i];
        plain += term;
    }
    total = wave_total(total);
    if (top_p < 1.0f && fixed) {
        const Mass target = share_of(total, top_p);
        uint32_t floor_key = 0;
        if (N == 1) {
            // (with the mass at and above each lane's key summed lane by lane, 64 times three words: 12 sequences, top-k 50 33.4 us, so 32.5, one 16.3 / 15.5)
            // in falling order of the keys, the key at which the mass so far first exceeds the target (of equal keys any will do: the mass down to
            // the last of them exceeds it then)
            const uint32_t word = sorted_down((key[0] << 6) | (uint32_t)(threadIdx.x & 63));
            const Mass so_far = running_total(__shfl(mass[0], (int)(word & 63)));
            const unsigned long long enough = __ballot(so_far > target);
            floor_key = enough ? (uint32_t)__builtin_amdgcn_readlane((int)word, __ffsll((long long)enough) - 1) >> 6 : 0;
        }
        for (int bit = 15; N > 1 && bit >= 0; --bit) {
            const uint32_t trial = floor_key | (1u << bit);
            if (trial > mk) continue;
            Mass a = 0;
#pragma unroll
            for (int i = 0; i < N; ++i) a += key[i] >= trial ? mass[i] : 0ull;
            if (wave_total(a) > target) floor_key = trial;
        }
        total = 0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (key[i] < floor_key) { key[i] = 0; mass[i] = 0; }
            total += mass[i];
        }
        total = wave_total(total);
    }
    const float Z = fixed ? (float)total * (1.0f / kMassScale) : wave_total(plain);
    Pick best{-INFINITY, 0.f, 0x7fffffff};
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (__ballot(key[i] != 0) == 0) continue;
        if (key[i]) { const float x = value_of_key<T>(key[i]); better(best, drawn(x, column[i]), x, column[i]); }
    }
    best = wave_best(best);
    if (best.column == 0x7fffffff || !(best.x > kNoConfidence)) { x0 = 0; x0_p = 0.f; return; }      // nothing but NaN, or the type's lowest values
    x0 = best.column;
    x0_p = NOISE == 0 ? fminf(1.0f / Z, 1.0f) : __builtin_amdgcn_exp2f((best.x - m) * c) / Z;
}

// The same from n candidates, of which the top-k keeps its own: moved together, to one per lane mostly, they take one draw of the
// generator per 64, where N registers with a few kept elements each take N.  (384 rows, top-k 50 and top-p 0.9 of about 210
// candidates, whole step: 38.5 -> 34.4 us, with the early lists and the lane-by-lane mass; 32 rows 21.2 -> 17.2; 384 rows, top-k 400: 73.3 -> 67.9; 0.3 and
// 0.8 more since the masses are 64-bit.)
constexpr int kManyKept = 8;
template <typename T, int NOISE, int N>
__device__ void pick_from_candidates(uint2* cand, int n, int lane, int top_k, float top_p, float c, const Drawn<NOISE>& drawn, int64_t& x0, float& x0_p)
{
    uint32_t key[N];
    int column[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int at = lane + 64 * i;
        const uint2 e = at < n ? cand[at] : uint2{0, 0};
        key[i] = e.x;                                                        // 0: none (the key of a negative NaN)
        column[i] = (int)e.y;
    }
    const uint32_t kth = kth_key(key, top_k);
    int kept = 0;
    unsigned long long stays[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        key[i] = key[i] >= kth ? key[i] : 0;
        stays[i] = __ballot(key[i] != 0);
        kept += __popcll(stays[i]);
    }
    if (kept > (N > kManyKept ? 64 * kManyKept : 64)) { pick_from_kept<T, NOISE, N>(key, column, top_p, c, drawn, x0, x0_p); return; }
    __builtin_amdgcn_wave_barrier();                                         // (one wavefront: its reads above are through before it writes)
    int before = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (key[i]) cand[before + __popcll(stays[i] & ((1ull << lane) - 1ull))] = uint2{key[i], (uint32_t)column[i]};
        before += __popcll(stays[i]);
    }
    __builtin_amdgcn_wave_barrier();
    auto pick = [&](auto count) {
        constexpr int M = decltype(count)::value;
        uint32_t k[M];
        int col[M];
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const uint2 e = lane + 64 * i < kept ? cand[lane + 64 * i] : uint2{0, 0};
            k[i] = e.x;
            col[i] = (int)e.y;
        }
        pick_from_kept<T, NOISE, M>(k, col, top_p, c, drawn, x0, x0_p);
    };
    if (kept <= 64) pick(std::integral_constant<int, 1>());
    else if constexpr (N > kManyKept) pick(std::integral_constant<int, kManyKept>());
}

template <typename T, int NOISE>
__global__ __launch_bounds__(kPickThreads) void filtered_pick_kernel(
    const uint16_t* __restrict__ logits, int64_t row_stride, int vocab, const float* __restrict__ temperatures, int rows_per_temp,
    int top_k, float top_p, const NoiseSpec N, int nsplit, int cap, const uint2* __restrict__ lists, const int* __restrict__ counts,
    int64_t* __restrict__ x0, float* __restrict__ x0_p)
{
    __shared__ uint2 cand[kMaxCandidates];
    const int64_t r = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const float T_ = temperatures ? temperatures[mdx::quotient((unsigned)r, rows_per_temp)] : 1.0f;
    const float c = kLog2e / T_;
    Drawn<NOISE> drawn;
    drawn.np = NOISE == 1 ? N.noise + r * N.noise_row_stride : nullptr;
    if (NOISE == 2) drawn.rn = row_noise(N, r);
    drawn.T = T_;
    drawn.unit_T = T_ == 1.0f;

    // The first lists are on their way before their lengths are known (what lies beyond is not taken): one trip to memory
    // instead of two per list.
    constexpr int kAhead = 4;
    uint2 early[kAhead];
    int m_early[kAhead];
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        m_early[s] = s < nsplit ? counts[r * nsplit + s] : 0;
        if (s < nsplit && tid < cap) early[s] = lists[(r * nsplit + s) * cap + tid];
    }
    int n = 0;
    bool whole = true;                                                       // every list holds all of its part's candidates
    auto take = [&](int s, int m, int from) {
        whole = whole && m <= cap;
        const uint2* list = lists + (r * nsplit + s) * cap;
        if (whole) for (int i = from + tid; i < m; i += kPickThreads) cand[n + i] = list[i];      // (nsplit * cap <= kMaxCandidates)
        n += m;
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        if (s >= nsplit) break;
        if (whole && m_early[s] <= cap && tid < m_early[s]) cand[n + tid] = early[s];
        take(s, m_early[s], kPickThreads);
    }
    for (int s = kAhead; s < nsplit; ++s) take(s, counts[r * nsplit + s], 0);
    if (whole) {
        __syncthreads();
        if (tid >= 64) return;
        int64_t token;
        float conf;
        if (n <= 256)      pick_from_candidates<T, NOISE, 4>(cand, n, lane, top_k, top_p, c, drawn, token, conf);
        else if (n <= 512) pick_from_candidates<T, NOISE, 8>(cand, n, lane, top_k, top_p, c, drawn, token, conf);
        else               pick_from_candidates<T, NOISE, kMaxCandidates / 64>(cand, n, lane, top_k, top_p, c, drawn, token, conf);
        if (lane == 0) { x0[r] = token; x0_p[r] = conf; }
        return;
    }

    // ---- too many ties for a list: the row itself, pass by pass ----
    __shared__ float fslot[kPickThreads / 64];
    __shared__ int islot[kPickThreads / 64];
    __shared__ Mass mslot[kPickThreads / 64];
    __shared__ Pick bests[kPickThreads / 64];
    const RowView row = row_view(logits + r * row_stride, vocab);
    const uint32_t floor_key = floor_by_bisection<T, kPickThreads>(row, tid, top_k, top_p, c, mslot, islot);
    Pick best{-INFINITY, 0.f, 0x7fffffff};
    float m = -INFINITY, Z = 0.f;
    auto kept = [&](uint32_t b) { return b != Bits16<T>::kNegInf && key_of(b) >= floor_key; };
    scan_row<kPickThreads>(row, tid, [&](uint32_t b, int) { if (kept(b)) m = fmaxf(m, Bits16<T>::value(b)); });
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, mdx::xor_lanes(m, off));
    __syncthreads();
    if (lane == 0) fslot[tid >> 6] = m;
    __syncthreads();
    for (int w = 0; w < kPickThreads / 64; ++w) m = fmaxf(m, fslot[w]);
    scan_row<kPickThreads>(row, tid, [&](uint32_t b, int column) {
        if (!kept(b)) return;
        const float x = Bits16<T>::value(b);
        Z += __builtin_amdgcn_exp2f((x - m) * c);
        better(best, drawn(x, column), x, column);
    });
    Z = block_total<kPickThreads>(Z, fslot, tid);
    best = wave_best(best);
    if (lane == 0) bests[tid >> 6] = best;
    __syncthreads();
    if (tid != 0) return;
    for (int w = 1; w < kPickThreads / 64; ++w) better(best, bests[w].v, bests[w].x, bests[w].column);
    const bool any = best.column != 0x7fffffff && best.x > kNoConfidence;
    x0[r] = any ? best.column : 0;
    x0_p[r] = !any ? 0.f : NOISE == 0 ? fminf(1.0f / Z, 1.0f) : __builtin_amdgcn_exp2f((best.x - m) * c) / Z;
}

// Threads per part, parts per row and list length for a top-k; threads = 0 where this form does not apply.
struct Plan { int threads, nsplit, cap; };
Plan plan_of(int64_t vocab, int top_k) {
    // The threshold is the k-th largest of `threads` values; of them about threads x ln(threads / (threads - k)) elements
    // reach it.  Half as many as threads keeps that below 0.7 threads, and half again as much room is far beyond its spread.
    for (int threads : {512, 1024}) {
        if (top_k <= 0 || top_k >= vocab || top_k > threads / 2) continue;
        const int64_t per_part = (int64_t)threads * kChunksPerThread;
        const int64_t nsplit = (vocab / 8 + per_part - 1) / per_part > 0 ? (vocab / 8 + per_part - 1) / per_part : 1;
        const int64_t cap = kMaxCandidates / nsplit;
        const double expected = threads * log((double)threads / (threads - top_k));
        if (1.4 * expected + 48 <= (double)cap) return Plan{threads, (int)nsplit, (int)cap};
    }
    return Plan{0, 0, 0};
}

template <typename T>
int launch(const Plan& plan, const void* logits, int64_t row_stride, const float* temperatures, int rows_per_temp, int top_k, float top_p,
           const NoiseSpec& N, int64_t* x0, float* x0_p, int64_t rows, int64_t vocab, void* workspace, hipStream_t stream)
{
    uint2* lists = static_cast<uint2*>(workspace);
    int* counts = reinterpret_cast<int*>(lists + rows * plan.nsplit * plan.cap);
    const uint16_t* l = static_cast<const uint16_t*>(logits);
    const dim3 grid((unsigned)rows, (unsigned)plan.nsplit);
    if (plan.threads == 512) topk_candidates_kernel<T, 512><<<grid, 512, 0, stream>>>(l, row_stride, (int)vocab, top_k, plan.nsplit, plan.cap, lists, counts);
    else                     topk_candidates_kernel<T, 1024><<<grid, 1024, 0, stream>>>(l, row_stride, (int)vocab, top_k, plan.nsplit, plan.cap, lists, counts);
    const int rc = mdx::check_launch("topk_candidates");
    if (rc != MDX_OK) return rc;
#define MDX_PICK(NOISE) filtered_pick_kernel<T, NOISE><<<(unsigned)rows, kPickThreads, 0, stream>>>( \
        l, row_stride, (int)vocab, temperatures, rows_per_temp, top_k, top_p, N, plan.nsplit, plan.cap, lists, counts, x0, x0_p)
    if (N.philox)     MDX_PICK(2);
    else if (N.noise) MDX_PICK(1);
    else              MDX_PICK(0);
#undef MDX_PICK
    return mdx::check_launch("filtered_pick");
}

}  // namespace

namespace mdx {

int64_t filtered_pick_workspace_bytes(int64_t rows, int64_t vocab, int top_k)
{
    const Plan plan = plan_of(vocab, top_k);
    return plan.threads ? rows * plan.nsplit * (plan.cap * (int64_t)sizeof(uint2) + (int64_t)sizeof(int)) : 0;
}

int filtered_pick(const void* logits, int64_t row_stride, int32_t dtype, const float* temperatures, int rows_per_temp,
                  int top_k, float top_p, const NoiseSpec& N, int64_t* x0, float* x0_p, int64_t rows, int64_t vocab,
                  void* workspace, hipStream_t stream)
{
    const Plan plan = plan_of(vocab, top_k);
    return dtype == MDX_BF16
        ? launch<__bf16>(plan, logits, row_stride, temperatures, rows_per_temp, top_k, top_p, N, x0, x0_p, rows, vocab, workspace, stream)
        : launch<__half>(plan, logits, row_stride, temperatures, rows_per_temp, top_k, top_p, N, x0, x0_p, rows, vocab, workspace, stream);
}

}  // namespace mdx
