// Routed products on block rows with few tokens each (few_rows.hip) and the scatter of their sums (routing.hip).
#pragma once
#include "common.h"

namespace stk {

struct SddArgs;

// Whether `slots` routed rows over `block_rows` block rows of 128 are few enough for the kernels of few_rows.hip.  The tiles
// here grow with the rows in use (32, 64, 128) and each reads its panel of weights for one block row only; the wide tiles cost
// the same from 1 to 128 rows.  stk_sdd_gather, us, wide against these (64 experts, 1024 x 4096, bf16): 4 rows per block row
// 119 / 107, 16 rows 115 / 107, 32 rows 118 / 113, 48 rows 119 / 116, 64 rows 121 / 134; 8 experts top-2: 18 / 13 from 4 to 32
// rows, 48 rows 19 / 16.
constexpr int64_t kFewRows = 48;
inline bool few_rows(int64_t slots, int64_t block_rows) { return slots <= kFewRows * block_rows; }
// The same for the second product, which also writes and reads its sums in fp32.  Where the wide tiles of stk_dsd, one block row
// and 256 columns each, come near to one per compute unit they stream as fast (64 experts, 1024 columns, top-1: 16 rows
// 94 / 96, 24 rows 94 / 101, 32 rows 95 / 107); with half as many or fewer these win as far as those of the first product
// (16 experts, 2048 columns, 8192 deep: 4 rows 123 / 92, 16 rows 123 / 97, 32 rows 123 / 104, 48 rows 124 / 113; 8 experts,
// 1024 columns, top-2: 65 / 19 at 4 rows, 65 / 26 at 48).
inline bool few_rows_dsd(int64_t slots, int64_t block_rows, int64_t n) {
  return slots <= 16 * block_rows || (few_rows(slots, block_rows) && block_rows * ((n + 255) / 256) <= compute_units() / 2);
}

// stk_sdd_gather on such block rows; k a positive multiple of 64.
void sdd_few(const SddArgs& g, bool bk, bool bf16, hipStream_t stream);

// out[t] = sum over k of (weights[s]) * row(s), s = t * top_k + k, where row(s) = the sum of sums[.][s] over the slices, added up
// in their order and rounded to the value type; slots whose slot_rows[s] is not in [0, rows) are left out.
int scatter_sums(const float* sums, int slices, int64_t slots, int64_t n, const int32_t* slot_rows, int64_t rows, const float* weights, int top_k,
                 int64_t tokens, void* out, int64_t out_stride, int dtype, hipStream_t stream);

}  // namespace stk
