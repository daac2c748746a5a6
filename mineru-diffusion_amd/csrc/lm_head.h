// What the two forms of the fused vocabulary projection share (lm_head_unmask.hip, lm_head_rows.hip).
#pragma once
#include "mdx_common.h"

namespace mdx_head {

constexpr float kLog2e = 1.4426950408889634f;

struct Record { float m, s; int idx, pad; };   // max logit, sum of exp2((x - m) c), first index of the max

struct LmHeadParams {
    const __bf16* x; const __bf16* w;
    int64_t x_stride, w_stride;                // elements between rows
    const float* temperatures; int rows_per_temp; const int64_t* row_ids;
    int rows, vocab, hidden;
    int n_row_tiles, n_vocab_tiles, n_slices;
    Record* records;                           // [rows, n_slices]
    int64_t* x0; float* x0_p;
};

__device__ __forceinline__ float row_scale(const LmHeadParams& P, int row) {
    if (!P.temperatures || row >= P.rows) return kLog2e;
    const int64_t id = P.row_ids ? P.row_ids[row] : row;
    const int per = P.rows_per_temp;                // mostly 1 or a block's length: a shift, where a division of 64 bits per row stood in every tile's start
    return kLog2e / P.temperatures[(per & (per - 1)) == 0 ? id >> __builtin_ctz(per) : id / per];
}

// The form for few rows: whether it covers the shape, and its launch (records only; n_slices is set to their number per row).
bool few_rows_covered(int64_t rows, int64_t vocab, int64_t hidden);
int launch_few_rows(LmHeadParams& P, hipStream_t stream);

}  // namespace mdx_head
