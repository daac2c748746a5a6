// Tile arithmetic shared by the two fp32-arithmetic attention kernels (staircase_attn_f32.hip, paged_attn_f32.hip):
// the forms of the attention calls for fp32 tensors and for heads that the 16-bit kernels do not take (wider than
// 128 columns, or not a multiple of 16).  Built for exactness, not for speed: both products run on the fp32 matrix
// instruction (v_mfma_f32_32x32x2_f32), the probabilities are never rounded, 16-bit inputs are widened on their way
// into LDS.
//
// Products are transposed (S^T = K Q^T, O^T = V^T P^T), as in the 16-bit kernels, so that a query is a column of the
// matrix instruction and lives in the lane pair (r, r + 32): the softmax over keys is arithmetic inside a lane plus
// one exchange with the other half-wavefront.  A wavefront owns 32 queries of one head; K and V tiles of 32 keys sit
// in LDS as fp32.
#pragma once
#include "mdx_common.h"
#include <type_traits>

namespace mdx_attn_f32 {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileKeys = 32;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kMinusBig = -1.0e30f;

// Four consecutive elements as floats (the pointer is 16-byte aligned for fp32, 8-byte for 16-bit elements).
__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load4(const __bf16* p) {
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    return f32x4{__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                 __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
}
__device__ __forceinline__ f32x4 load4(const _Float16* p) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 raw = *reinterpret_cast<const h4*>(p);
    return f32x4{(float)raw[0], (float)raw[1], (float)raw[2], (float)raw[3]};
}
__device__ __forceinline__ void store4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void store4(__bf16* p, f32x4 v) {
    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<b4*>(p) = b4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}
__device__ __forceinline__ void store4(_Float16* p, f32x4 v) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<h4*>(p) = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}

// Row of the 32 x 32 result that accumulator register i of a lane in half-wavefront H holds.
__device__ __forceinline__ int row_of_reg(int i, int H) { return 8 * (i >> 2) + 4 * H + (i & 3); }

// D: 128 or 256, the head width that registers and LDS are laid out for (narrower heads are padded with zeros;
// products over the padding are skipped).
template <int D> struct Lds {
    // floats; rows stay 16-byte aligned and consecutive rows shift by 4 banks: the 16-byte reads of 8 consecutive keys
    // (K fragments: four columns of a key per read) cover all banks once, and so do the two keys of a V k-step
    static constexpr int kPitchK = D + 4;
    static constexpr int kPitchV = D + 4;
    static constexpr int kFloats = kTileKeys * (kPitchK + kPitchV);
    static constexpr int kBytes = kFloats * (int)sizeof(float);
    static __device__ __forceinline__ float* k_tile(float* lds) { return lds; }
    static __device__ __forceinline__ float* v_tile(float* lds) { return lds + kTileKeys * kPitchK; }
};

// Each half-wavefront contracts over a half of the head's columns: H over the columns from H * half_width(width) on.
__device__ __forceinline__ int half_width(int width) { return (width + 7) / 8 * 4; }

// One query's row of Q^T for lane (H, r): its half of the columns (row may be null: zeros, as beyond the head's width).
template <typename T, int D>
__device__ __forceinline__ void load_q(float (&q)[D / 2], const T* row, int H, int width) {
    const int half = half_width(width);
#pragma unroll
    for (int m = 0; m < D / 8; ++m) {
        const int col = H * half + 4 * m;
        f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row && 4 * m < half && col < width) x = load4(row + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) q[4 * m + e] = x[e];
    }
}

// A tile's K and V rows on their way to LDS: (part of) a thread's share of them, as loaded (16-bit elements are widened when they
// are written).  Fetching a batch of up to kBatch rows before writing any keeps their loads in flight together; loading and
// writing row by row had cost a trip to memory per row.
constexpr int kBatch = 4;
template <typename T> struct Raw4;
template <> struct Raw4<float> { typedef f32x4 type; };
template <> struct Raw4<__bf16> { typedef uint2 type; };
template <> struct Raw4<_Float16> { typedef uint2 type; };

template <typename T, int D, int THREADS> struct TileRegs {
    static constexpr int kAll = kTileKeys * (D / 4) / THREADS, kPasses = kAll < kBatch ? kAll : kBatch, kBatches = kAll / kPasses;
    typename Raw4<T>::type k[kPasses], v[kPasses];
    // row_ptr(row): element offset of that row of the tile, the same for K and V's bases; any row may be asked for.
    template <typename KRow, typename VRow>
    __device__ __forceinline__ void fetch(int batch, int tid, int width, KRow k_row, VRow v_row) {
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int u = tid + THREADS * (batch * kPasses + p), row = u / (D / 4), col = min(4 * (u % (D / 4)), width - 4);
            k[p] = *reinterpret_cast<const typename Raw4<T>::type*>(k_row(row) + col);
            v[p] = *reinterpret_cast<const typename Raw4<T>::type*>(v_row(row) + col);
        }
    }
    // real(row): whether the row holds a key (else, and beyond the head's width: zeros)
    template <typename Real>
    __device__ __forceinline__ void write(int batch, float* lds, int tid, int width, Real real) const {
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int u = tid + THREADS * (batch * kPasses + p), row = u / (D / 4), c4 = u % (D / 4);
            f32x4 kx = load4(reinterpret_cast<const T*>(&k[p])), vx = load4(reinterpret_cast<const T*>(&v[p]));
            if (!real(row) || 4 * c4 >= width) { kx = f32x4{0.f, 0.f, 0.f, 0.f}; vx = kx; }
            *reinterpret_cast<f32x4*>(Lds<D>::k_tile(lds) + row * Lds<D>::kPitchK + 4 * c4) = kx;
            *reinterpret_cast<f32x4*>(Lds<D>::v_tile(lds) + row * Lds<D>::kPitchV + 4 * c4) = vx;
        }
    }
};

// TILES tiles of 32 queries on their way to LDS, where rows lie like those of a K tile, and from there to the lanes as load_q has them
// (a lane's own row, 16 bytes at a time, touches every line eight times).
template <typename T, int D, int TILES, int THREADS> struct QueryRegs {
    static constexpr int kPasses = TILES * 32 * (D / 4) / THREADS, kBytes = TILES * 32 * Lds<D>::kPitchK * (int)sizeof(float);
    f32x4 x[kPasses];
    // row_ptr(row): that row, or null (zeros, as beyond the head's width)
    template <typename Row> __device__ __forceinline__ void fetch(int tid, int width, Row row_ptr) {
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int u = tid + THREADS * p, col = 4 * (u % (D / 4));
            const T* row = row_ptr(u / (D / 4));
            x[p] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (row && col < width) x[p] = load4(row + col);
        }
    }
    __device__ __forceinline__ void write(float* lds, int tid) const {
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int u = tid + THREADS * p;
            *reinterpret_cast<f32x4*>(lds + u / (D / 4) * Lds<D>::kPitchK + 4 * (u % (D / 4))) = x[p];
        }
    }
    static __device__ __forceinline__ void read(float (&q)[D / 2], const float* lds, int tile, int H, int r, int width) {
        const int half = half_width(width);
        const float* row = lds + (tile * 32 + r) * Lds<D>::kPitchK + H * half;
#pragma unroll
        for (int m = 0; m < D / 8; ++m) {
            const f32x4 v = 4 * m < half ? *reinterpret_cast<const f32x4*>(row + 4 * m) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) q[4 * m + e] = v[e];
        }
    }
};

// Running softmax state of a wavefront's 32 queries: l is this half-wavefront's share of the row sum.
template <int D> struct State {
    float m, l;
    f32x16 o[D / 32];
    __device__ __forceinline__ void init() {
        m = kMinusBig; l = 0.f;
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    }
};

// One tile of 32 keys against the wavefront's 32 queries.  visible(key in tile) says whether this lane's query sees it.
template <int D, typename Visible>
__device__ __forceinline__ void tile_step(const float* lds, const float (&q)[D / 2], State<D>& st, float c, int width, int lane, Visible visible)
{
    const int H = lane >> 5, r = lane & 31;
    // ---- S^T = K Q^T: rows = keys, columns = queries; k-step j covers the columns j and half + j (the order of a contraction is
    //      free), so that a lane's 16-byte read of key r feeds four k-steps.  (With the columns 2 j and 2 j + 1 half of every read
    //      of K and of Q was the other half-wavefront's: us, before / after, paged 1 x 1056 keys 23.9 / 21.3, 2 x 900-2000 36.8 / 32.9,
    //      4 x 1000-3000 62.0 / 55.2; prompts of 60 tokens 16.8 / 13.7, 300 32.5 / 27.9, 1024 107 / 91, 4000 722 / 687) ----
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    const int half = half_width(width);
    const float* krow = Lds<D>::k_tile(const_cast<float*>(lds)) + r * Lds<D>::kPitchK + H * half;
#pragma unroll
    for (int m = 0; m < D / 8; ++m) {
        if (4 * m >= half) continue;
        const f32x4 kx = *reinterpret_cast<const f32x4*>(krow + 4 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[e], q[4 * m + e], s, 0, 0, 0);
    }

    // ---- online softmax over the keys, base 2 ----
    float mx = kMinusBig;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        s[i] = visible(row_of_reg(i, H)) ? s[i] * c : -INFINITY;
        mx = fmaxf(mx, s[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(st.m, mx);
    const float alpha = __builtin_amdgcn_exp2f(st.m - m_new);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        s[i] = __builtin_amdgcn_exp2f(s[i] - m_new);
        sum += s[i];
    }
    st.l = st.l * alpha + sum;
    st.m = m_new;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) st.o[dt][i] *= alpha;

    // ---- O^T += V^T P^T: rows = d, columns = queries; k-step (g, e) covers the keys 8 g + e and 8 g + 4 + e,
    //      which are the keys of this lane's register 4 g + e in the two half-wavefronts ----
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
        if (dt * 32 >= width) continue;
        const float* vcol = Lds<D>::v_tile(const_cast<float*>(lds)) + dt * 32 + r;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            st.o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vcol[row_of_reg(i, H) * Lds<D>::kPitchV], s[i], st.o[dt], 0, 0, 0);
    }
}

// Folds, through LDS, the states of the KW wavefronts (wave, wave + 1, ... of a multiple of KW) that shared a query tile's keys, and
// hands out the columns: emit(d, O's columns d .. d + 3 of this lane's query, not yet divided by l); each wavefront gets every
// KW-th column tile.  m and l come back whole before the first emit.  Called by all wavefronts; the region must hold their states.
template <int D, int KW, typename Emit>
__device__ __forceinline__ void fold_states(float* lds, State<D>& st, int wave, int lane, int width, Emit emit) {
    constexpr int kMl = (D / 32) * 16 * 64, kStateFloats = kMl + 2 * 64;       // O as [d tile][register quad][lane][4], then m, l
    const int H = lane >> 5, kw = wave % KW;
    st.l += __shfl_xor(st.l, 32);                                              // a state is now (m, l, O) per query
    const float* states = lds + (wave - kw) * kStateFloats;
    auto quad = [&](int dt, int g) { return f32x4{st.o[dt][4 * g], st.o[dt][4 * g + 1], st.o[dt][4 * g + 2], st.o[dt][4 * g + 3]}; };
    // MINE: this wavefront's kw.  What it hands out itself stays in its registers.  (All of every state through LDS, four bytes at a time: 3600 cycles of a workgroup's
    // 24 900 of one sequence of 1056 keys.)
    auto fold = [&](auto mine) {
        constexpr int MINE = decltype(mine)::value;
        float w[KW];
        if (KW > 1) {
            __syncthreads();                                                   // the last tiles have been read by everybody
            float* dst = lds + wave * kStateFloats;
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    if (dt % KW != MINE) *reinterpret_cast<f32x4*>(dst + ((dt * 4 + g) * 64 + lane) * 4) = quad(dt, g);
            dst[kMl + lane] = st.m;
            dst[kMl + 64 + lane] = st.l;
            __syncthreads();
            float M = kMinusBig, l_all = 0.f;
#pragma unroll
            for (int s = 0; s < KW; ++s) { w[s] = states[s * kStateFloats + kMl + lane]; M = fmaxf(M, w[s]); }
#pragma unroll
            for (int s = 0; s < KW; ++s) {
                w[s] = __builtin_amdgcn_exp2f(w[s] - M);
                l_all += states[s * kStateFloats + kMl + 64 + lane] * w[s];
            }
            st.m = M;
            st.l = l_all;
        }
#pragma unroll
        for (int dt = MINE; dt < D / 32; dt += KW) {
            if (dt * 32 >= width) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
                if (KW == 1) acc = quad(dt, g);
#pragma unroll
                for (int s = 0; KW > 1 && s < KW; ++s)
                    acc += (s == MINE ? quad(dt, g) : *reinterpret_cast<const f32x4*>(states + s * kStateFloats + ((dt * 4 + g) * 64 + lane) * 4)) * w[s];
                const int d = dt * 32 + 8 * g + 4 * H;
                if (d < width) emit(d, acc);
            }
        }
    };
    // (the same throughout a wavefront; each meets the same barriers, whichever branch it takes)
    const int slice = __builtin_amdgcn_readfirstlane(kw);
    if (KW == 1 || slice == 0) fold(std::integral_constant<int, 0>());
    else if (slice == 1) fold(std::integral_constant<int, 1 % KW>());
    else if (slice == 2) fold(std::integral_constant<int, 2 % KW>());
    else fold(std::integral_constant<int, 3 % KW>());
}
template <int D> constexpr int kStateBytes = ((D / 32) * 16 * 64 + 2 * 64) * (int)sizeof(float);

}  // namespace mdx_attn_f32
