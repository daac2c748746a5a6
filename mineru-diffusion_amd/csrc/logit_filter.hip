// Top-k / top-p filtering of a row of logits before sampling: the HF variant's top_k_logits and
// top_p_logits (mineru_diffusion/modeling_mineru_diffusion.py:585-600, applied in that order by
// sample_with_temperature_topk_topp, :608-611).  The reference sorts every row; here a row is never
// sorted.  Both filters keep exactly the elements at or above one VALUE of the row:
//
//   top-k   the k-th largest value (elements equal to it are all kept, as `logits < min_values` keeps them)
//   top-p   the value of the element at which the cumulative probability, taken from the largest
//           element down, first exceeds p (softmax over what top-k kept, at temperature T)
//
// and a 16-bit logit has only 65 536 possible values, so that value is found by COUNTING: one pass over the row adds each
// element to the counter of its own value (16-bit counters, two to a word: 128 KB of LDS, one workgroup per CU), and the
// rest is done on the counters.  A probability mass is a count times the softmax term of the value, so an element costs
// one LDS atomic and no exponential.  What bounds it: the LDS atomics, one per element.  (The form this replaced counted
// the high byte of a value and then the low byte within the crossing bin, with 16 copies of every counter and a second,
// 64-bit atomic per element for the masses, and read the row up to five times: 1024 rows of 151 936, top-k 50 with top-p 0.9
// 344 us, top-p alone 314; this one 232 with both.)
//
// Where the reference's sort leaves the order of equal values open, all elements equal to the crossing
// value are kept.  The masses are 64-bit fixed-point sums of fp32 softmax terms; against a computation in higher
// precision, a target that falls within fp32 rounding of a cumulative probability can resolve either way.
#include "logit_keys.h"
#include "filtered_pick.h"
#include <atomic>

namespace {

using namespace mdx_keys;

constexpr int kFilterThreads = 1024;
constexpr int kWaves = kFilterThreads / 64;
constexpr int kWords = 32768;                        // counters of the keys 2 w (low half) and 2 w + 1 (high half)
constexpr int kWordsPerThread = kWords / kFilterThreads;
constexpr int kHistBytes = kWords * 4;

struct Scratch {
    Mass mslot[kWaves];
    int islot[kWaves];
    uint32_t floor_key;
};

// Inclusive prefix over the workgroup's threads (wavefront scans, then the totals of the wavefronts before).
template <typename V> __device__ __forceinline__ V block_prefix(V v, V* slot, int tid, V* total) {
    const int lane = tid & 63, wave = tid >> 6;
    V x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) { const V o = __shfl_up(x, off); if (lane >= off) x += o; }
    __syncthreads();
    if (lane == 63) slot[wave] = x;
    __syncthreads();
    V before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) { if (w < wave) before += slot[w]; all += slot[w]; }
    *total = all;
    return before + x;
}

// The row's cut-off key from the counters; 0 = everything is kept.
template <typename T>
__device__ uint32_t floor_from_counts(const RowView& row, uint32_t* hist, Scratch& sh, int tid, int top_k, float top_p, float c) {
    const bool with_k = top_k > 0 && top_k < row.vocab;
    for (int i = tid; i < kWords / 4; i += kFilterThreads) reinterpret_cast<u32x4*>(hist)[i] = u32x4{0, 0, 0, 0};
    if (tid == 0) sh.floor_key = 0;
    __syncthreads();
    // -inf, which often fills most of a row, is counted in a register
    constexpr uint32_t kInfKey = Bits16<T>::kNegInf ^ 0xffffu;       // (odd: the high half of its word)
    int n_inf = 0;
    scan_row<kFilterThreads>(row, tid, [&](uint32_t b, int) {
        if (b == Bits16<T>::kNegInf) { ++n_inf; return; }
        const uint32_t key = key_of(b);
        atomicAdd(&hist[key >> 1], (key & 1u) ? 0x10000u : 1u);
    });
    n_inf = block_total<kFilterThreads>(n_inf, sh.islot, tid);

    // Thread t looks after 64 consecutive keys, thread 0 after the largest.  (Every lane starts at another word: lanes are 32 words apart.)
    const int base = kWords - kWordsPerThread * (tid + 1), lane = tid & 63;
    int cnt = 0, top = -1;
    for (int j = 0; j < kWordsPerThread; ++j) {
        const int at = base + ((j + lane) & (kWordsPerThread - 1));
        const uint32_t w = hist[at];
        cnt += (int)((w & 0xffffu) + (w >> 16));
        if (w) top = max(top, 2 * at + (w >> 16 ? 1 : 0));
    }
    if (base <= (int)(kInfKey >> 1) && (int)(kInfKey >> 1) < base + kWordsPerThread) cnt += n_inf;
    int total;
    const int upto = block_prefix(cnt, sh.islot, tid, &total);
    // a counter that ran over has lost 65536, or carried 1 into its neighbour for them: the total shows it
    if (total != row.vocab) return floor_by_bisection<T, kFilterThreads>(row, tid, top_k, top_p, c, sh.mslot, sh.islot);

    uint32_t floor_key = 0;
    if (with_k) {
        if (upto >= top_k && upto - cnt < top_k) {                   // exactly one thread: the k-th largest is among its keys
            int n = upto - cnt;
            uint32_t key = 0;
            for (int at = base + kWordsPerThread - 1; at >= base && !key; --at) {
                n += (int)(hist[at] >> 16) + (at == (int)(kInfKey >> 1) ? n_inf : 0);
                if (n >= top_k) { key = 2 * at + 1; break; }
                n += (int)(hist[at] & 0xffffu);
                if (n >= top_k) key = 2 * at;
            }
            sh.floor_key = key;
        }
        __syncthreads();
        floor_key = sh.floor_key;
    }
    if (top_p >= 1.0f) return floor_key;

#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) top = max(top, mdx::xor_lanes(top, off));
    __syncthreads();
    if (lane == 0) sh.islot[tid >> 6] = top;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) top = max(top, sh.islot[w]);
    // a row whose largest element is not finite has no softmax to take a share of: left as it is
    if (top < 0) return floor_key;
    const float m = value_of_key<T>((uint32_t)top);
    if (!has_masses(m, c)) return floor_key;

    auto mass_at = [&](uint32_t key, uint32_t n) {
        return n && key >= floor_key ? n * mass_of(__builtin_amdgcn_exp2f((value_of_key<T>(key) - m) * c)) : 0ull;
    };
    Mass mass = 0;
    if (2 * (base + kWordsPerThread) > (int)floor_key && 2 * base <= top)
        for (int j = 0; j < kWordsPerThread; ++j) {
            const int at = base + ((j + lane) & (kWordsPerThread - 1));
            const uint32_t w = hist[at];
            if (w) mass += mass_at(2 * at, w & 0xffffu) + mass_at(2 * at + 1, w >> 16);
        }
    Mass total_mass;
    const Mass mass_upto = block_prefix(mass, sh.mslot, tid, &total_mass), target = share_of(total_mass, top_p);
    if (mass_upto > target && mass_upto - mass <= target) {          // exactly one thread (the share is less than the whole)
        Mass a = mass_upto - mass;
        uint32_t key = 0;
        for (int at = base + kWordsPerThread - 1; at >= base && !key; --at) {
            const uint32_t w = hist[at];
            a += mass_at(2 * at + 1, w >> 16);
            if (a > target) { key = 2 * at + 1; break; }
            a += mass_at(2 * at, w & 0xffffu);
            if (a > target) key = 2 * at;
        }
        sh.floor_key = key;
    }
    __syncthreads();
    return sh.floor_key;
}

// WRITE: the filtered row goes to `out`; otherwise the smallest value kept goes to floors[row].
template <typename T, bool WRITE>
__global__ __launch_bounds__(kFilterThreads) void logit_filter_kernel(
    const uint16_t* logits, int64_t row_stride,          // may be `out` itself
    const float* __restrict__ temperatures, int rows_per_temp,
    int top_k, float top_p, uint16_t* out, int64_t out_row_stride, float* __restrict__ floors, int vocab)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t hist[];
    __shared__ Scratch sh;
    const int64_t r = blockIdx.x;
    const int tid = threadIdx.x;
    const RowView row = row_view(logits + r * row_stride, vocab);
    const float c = kLog2e / (temperatures ? temperatures[mdx::quotient((unsigned)r, rows_per_temp)] : 1.0f);
    const uint32_t floor_key = floor_from_counts<T>(row, hist, sh, tid, top_k, top_p, c);
    if (!WRITE) {
        // (a cut-off below -inf is a NaN's; one above +inf drops every number, as it should)
        if (tid == 0) floors[r] = floor_key > (Bits16<T>::kNegInf ^ 0xffffu) ? value_of_key<T>(floor_key) : -INFINITY;
        return;
    }
    uint16_t* op = out + r * out_row_stride;
    auto keep = [&](uint32_t b) { return key_of(b) >= floor_key ? b : Bits16<T>::kNegInf; };
    if (((reinterpret_cast<uintptr_t>(op) ^ reinterpret_cast<uintptr_t>(row.p)) & 15) == 0) {
        u32x4* oc = reinterpret_cast<u32x4*>(op + row.lead);
        for (int e = tid; e < row.lead; e += kFilterThreads) op[e] = (uint16_t)keep(row.p[e]);
        for (int ch = tid; ch < row.nchunk; ch += kFilterThreads) {
            const u32x4 u = row.chunks[ch];
            uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = keep(w[i] & 0xffffu) | (keep(w[i] >> 16) << 16);
            u32x4 o; o.x = w[0]; o.y = w[1]; o.z = w[2]; o.w = w[3];
            oc[ch] = o;
        }
        for (int e = row.tail0 + tid; e < vocab; e += kFilterThreads) op[e] = (uint16_t)keep(row.p[e]);
    } else {
        for (int e = tid; e < vocab; e += kFilterThreads) op[e] = (uint16_t)keep(row.p[e]);
    }
}

template <typename T, bool WRITE>
int launch(const void* logits, int64_t row_stride, const float* temperatures, int rows_per_temp, int top_k, float top_p,
           void* out, int64_t out_row_stride, float* floors, int64_t rows, int64_t vocab, hipStream_t stream)
{
    // the kernel's LDS limit is raised once per device
    static std::atomic<bool> raised[64];
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    MDX_REQUIRE(e == hipSuccess && device >= 0 && device < 64, MDX_ELAUNCH, "filter_logits: no current device (%s)", hipGetErrorString(e));
    if (!raised[device].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(logit_filter_kernel<T, WRITE>), hipFuncAttributeMaxDynamicSharedMemorySize, kHistBytes);
        MDX_REQUIRE(e == hipSuccess, MDX_ELAUNCH, "filter_logits: cannot reserve %d bytes of LDS (%s)", kHistBytes, hipGetErrorString(e));
        raised[device].store(true, std::memory_order_release);
    }
    logit_filter_kernel<T, WRITE><<<(unsigned)rows, kFilterThreads, kHistBytes, stream>>>(
        static_cast<const uint16_t*>(logits), row_stride, temperatures, rows_per_temp, top_k, top_p,
        static_cast<uint16_t*>(out), out_row_stride, floors, (int)vocab);
    return mdx::check_launch("filter_logits");
}

}  // namespace

namespace mdx {

int check_filter(const void* logits, int64_t row_stride, int32_t dtype, int32_t top_k, float top_p, int64_t rows, int64_t vocab)
{
    MDX_REQUIRE(rows >= 0 && vocab >= 0, MDX_EINVAL, "filter_logits: negative size");
    MDX_REQUIRE(top_k >= 0, MDX_EINVAL, "filter_logits: top_k %d < 0", top_k);
    MDX_REQUIRE(top_p >= 0.f, MDX_EINVAL, "filter_logits: top_p %g < 0 (or not a number)", (double)top_p);
    if (rows == 0) return MDX_OK;
    MDX_REQUIRE(vocab > 0, MDX_EINVAL, "filter_logits: empty vocabulary");
    MDX_REQUIRE(logits, MDX_EINVAL, "filter_logits: null pointer");
    MDX_REQUIRE(dtype == MDX_BF16 || dtype == MDX_F16, MDX_EUNSUPPORTED, "filter_logits: dtype %d (16-bit logits only)", dtype);
    MDX_REQUIRE(vocab <= (int64_t)1 << 23 && rows < (int64_t)0x7fffffff, MDX_EUNSUPPORTED,
                "filter_logits: rows %lld or vocab %lld out of range (vocab at most 8388608)", (long long)rows, (long long)vocab);
    MDX_REQUIRE(row_stride >= vocab, MDX_EUNSUPPORTED, "filter_logits: row stride smaller than the vocabulary");
    MDX_REQUIRE((reinterpret_cast<uintptr_t>(logits) % 2) == 0, MDX_EUNSUPPORTED, "filter_logits: logits not element-aligned");
    return MDX_OK;
}

int filter_floors(const void* logits, int64_t row_stride, int32_t dtype, const float* temperatures, int rows_per_temp,
                  int top_k, float top_p, float* floors, int64_t rows, int64_t vocab, hipStream_t stream)
{
    return dtype == MDX_BF16
        ? launch<__bf16, false>(logits, row_stride, temperatures, rows_per_temp, top_k, top_p, nullptr, 0, floors, rows, vocab, stream)
        : launch<__half, false>(logits, row_stride, temperatures, rows_per_temp, top_k, top_p, nullptr, 0, floors, rows, vocab, stream);
}

}  // namespace mdx

extern "C" int mdx_filter_logits(const void* logits, int64_t row_stride, int32_t dtype,
                                 const float* temperatures, int32_t rows_per_temp,
                                 int32_t top_k, float top_p,
                                 void* out, int64_t out_row_stride,
                                 int64_t rows, int64_t vocab, mdx_stream_t stream_)
{
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int rc = mdx::check_filter(logits, row_stride, dtype, top_k, top_p, rows, vocab);
    if (rc != MDX_OK || rows == 0) return rc;
    MDX_REQUIRE(out, MDX_EINVAL, "filter_logits: null pointer");
    MDX_REQUIRE(out_row_stride >= vocab, MDX_EUNSUPPORTED, "filter_logits: row stride smaller than the vocabulary");
    MDX_REQUIRE(!temperatures || rows_per_temp > 0, MDX_EINVAL, "filter_logits: rows_per_temp must be positive");
    MDX_REQUIRE((reinterpret_cast<uintptr_t>(out) % 2) == 0, MDX_EUNSUPPORTED, "filter_logits: logits not element-aligned");
    return dtype == MDX_BF16
        ? launch<__bf16, true>(logits, row_stride, temperatures, rows_per_temp, top_k, top_p, out, out_row_stride, nullptr, rows, vocab, stream)
        : launch<__half, true>(logits, row_stride, temperatures, rows_per_temp, top_k, top_p, out, out_row_stride, nullptr, rows, vocab, stream);
}
