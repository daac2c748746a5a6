// The pieces of the top-k / top-p filter that the filtered unmask step is made of (logit_filter.hip, filtered_pick.hip).
#pragma once
#include "gumbel_noise.h"

namespace mdx {

// Checks what every form of the filter asks of its arguments.
int check_filter(const void* logits, int64_t row_stride, int32_t dtype, int32_t top_k, float top_p, int64_t rows, int64_t vocab);

// floors[row] = the smallest value of the row that the filter keeps (-inf: everything).
int filter_floors(const void* logits, int64_t row_stride, int32_t dtype, const float* temperatures, int rows_per_temp,
                  int top_k, float top_p, float* floors, int64_t rows, int64_t vocab, hipStream_t stream);

// Filter, confidence and pick of a row from the few candidates that its top-k can hold: one pass over the logits.  The
// workspace query returns 0 where this form does not apply (no top-k, or one too large).
int64_t filtered_pick_workspace_bytes(int64_t rows, int64_t vocab, int top_k);
int filtered_pick(const void* logits, int64_t row_stride, int32_t dtype, const float* temperatures, int rows_per_temp,
                  int top_k, float top_p, const mdx_noise::NoiseSpec& N, int64_t* x0, float* x0_p, int64_t rows, int64_t vocab,
                  void* workspace, hipStream_t stream);

}  // namespace mdx
