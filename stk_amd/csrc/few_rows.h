// Routed products on block rows with few tokens each (few_rows.hip) and the scatter of their sums (routing.hip).
#pragma once
#include "common.h"

namespace stk {

struct SddArgs;

// Whether `slots` routed rows over `block_rows` block rows of 128 are few enough for the kernels of few_rows.hip.  The tiles
// here grow with the rows in use (32, 64, 128) and each reads its panel of weights for one block row only; the wide tiles cost
// the same from 1 to 128 rows.  stk_sdd_gather, us, wide against these (64 experts, 1024 x 4096, bf16):
//   even routing       2 rows per block row 114 / 100, 8 rows 115 / 107, 32 rows 118 / 115, 47 rows 121 / 116, 64 rows 123 / 127
//   K-major weights    2 rows 125 / 100, 32 rows 138 / 119, 47 rows 139 / 120
//   Zipf (s = 1.2)     4 rows 77 / 60, 16 rows 120 / 112, 41 rows 143 / 136, 50 rows 151 / 150
//   half on one expert 15 rows 141 / 112, 39 rows 145 / 130
//   layout of fixed capacity (block rows without a token beside those with twice the mean, which the wide tiles compute and
//   these only clear)  14 rows 139 / 109, 35 rows 152 / 126, 43 rows 159 / 131
// 8 experts top-2: 20 / 15 from 2 to 16 rows, 48 rows 20 / 17.
constexpr int64_t kFewRows = 48;
inline bool few_rows(int64_t slots, int64_t block_rows) { return slots <= kFewRows * block_rows; }
// The same for the second product.  Where the wide tiles of stk_dsd, one block row
// and 256 columns each, come near to one per compute unit they stream as fast (64 experts, 1024 columns, top-1, even: 8 rows
// 93 / 90, 16 rows 94 / 92, 32 rows 93 / 99, 47 rows 96 / 103); with half as many or fewer these win as far as those of the first
// product (16 experts, 2048 columns, 8192 deep: 2 rows 120 / 85, 16 rows 128 / 92, 38 rows 128 / 94; 8 experts,
// 1024 columns, top-2: 64 / 24 at 2 rows, 65 / 30 at 48).
inline bool few_rows_dsd(int64_t slots, int64_t block_rows, int64_t n) {
  return slots <= 16 * block_rows || (few_rows(slots, block_rows) && block_rows * ((n + 255) / 256) <= compute_units() / 2);
}

// stk_sdd_gather on such block rows; k a positive multiple of 64.
void sdd_few(const SddArgs& g, bool bk, bool bf16, hipStream_t stream);

// out[t] = sum over k of (weights[s]) * row(s), s = t * top_k + k, where row(s) = sums[s] rounded to the value type; slots whose
// slot_rows[s] is not in [0, rows) are left out.
int scatter_sums(const float* sums, int64_t slots, int64_t n, const int32_t* slot_rows, int64_t rows, const float* weights, int top_k, int64_t tokens,
                 void* out, int64_t out_stride, int dtype, hipStream_t stream);

}  // namespace stk
