// The two products of a routed layer whose block rows hold few tokens each (a decoding step, a small batch over many
// experts): stk_sdd_gather and stk_dsd_scatter_few.  With a few token rows in a block of 128 a product is one pass over
// the experts' weights, and what bounds it is how many bytes of them are in flight.  The tiles here therefore compute only
// the 32, 64 or 128 rows that reach to the last token of a block row, one 128-wide panel of weights per workgroup of four
// wavefronts (each 32 columns of it), with three 16 KB stages of weights in flight and two workgroups per compute unit:
// one's start and stores lie under the other's stream, and the many short tiles leave no long last round.  64 tokens top-2
// over 64 experts (1024 x 4096, bf16, 466 MB of weights a product): the wide tiles take 110 us for the first product and 104
// for the second with its scatter, these 94 (with the 59 MB of its result 5.6 TB/s) and 86 (5.4 TB/s); 300 tokens over 16
// experts (2048 x 8192) 101 and 123 us, these 101 and 98; 16 tokens 27 and 67 us, these 23 and 26.
// Without the non-temporal hint on the weights: 109 and 100 us; workgroups in plain order:
// 95 and 95, in eight contiguous shares 95 and 86 (and 70 instead of 46 us where four experts share the block rows unevenly).
#include "few_rows.h"
#include "sdd_tile.h"

namespace stk {

constexpr int kFewKT = 64;
constexpr int kFewThreads = 256;
constexpr int kFewLds = 80 * 1024;   // two workgroups share the 160 KB of a compute unit

// Rows that end with the last row of a block row that holds a token, 0 .. 128.
__device__ __forceinline__ int rows_in_use(const int32_t* row_slots, int slots, int block_row, int lane) {
  const int32_t* s = row_slots + (int64_t)block_row * 128;
  const uint64_t lo = __ballot((unsigned)s[lane] < (unsigned)slots), hi = __ballot((unsigned)s[64 + lane] < (unsigned)slots);
  return hi ? 128 - __builtin_clzll(hi) : lo ? 64 - __builtin_clzll(lo) : 0;
}

// acc += A x B for 32 IM rows and 128 columns; wavefront w owns the columns 32 w .. 32 w + 31.  offa: the lanes' offsets of
// the A transfers; next(a, b) sets the origins of the next K-tile, in increasing order.
template <int IM, bool BK, bool BF16, class Next>
__device__ __forceinline__ void few_rows_loop(f32x16_t (&acc)[IM], int ntiles, const uint32_t (&offa)[IM], int64_t ldb, char* smem, Next&& next) {
  using OpA = Operand<32 * IM, true, kFewKT, kFewThreads>;
  using OpB = Operand<128, BK, kFewKT, kFewThreads>;
  constexpr int kStage = OpA::kBytes + OpB::kBytes, S = IM == 1 ? 4 : IM == 2 ? 3 : 2, kLoads = IM + OpB::kSlicesPerWave;
  static_assert(OpA::kSlicesPerWave == IM && S * kStage <= kFewLds, "the stages fit");
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)((STK_LDS char*)smem);
  uint32_t offb[OpB::kSlicesPerWave];
  OpB::dma_offsets(offb, wave, lane, ldb);
  auto issue = [&](int t) {
    const elem_t *a, *b;
    next(a, b);
    const gptr_t ga = uniform_global(a), gb = uniform_global(b);
    const uint32_t stage = lds0 + (uint32_t)(t % S) * kStage;
#pragma unroll
    for (int i = 0; i < OpB::kSlicesPerWave; i++) dma16<!BK>(gb, offb[i], stage + OpA::kBytes + (i * 4 + wave) * 1024);
#pragma unroll
    for (int i = 0; i < IM; i++) dma16(ga, offa[i], stage + (i * 4 + wave) * 1024);
  };
  for (int t = 0; t < S - 1 && t < ntiles; t++) issue(t);
  for (int t = 0; t < ntiles; t++) {
    // K-tile t has landed; up to S - 2 younger ones stay in flight
    const int younger = ntiles - 1 - t;
    if (S >= 4 && younger >= 2) wait_vmcnt<2 * kLoads>();
    else if (S >= 3 && younger >= 1) wait_vmcnt<1 * kLoads>();
    else wait_vmcnt<0>();
    // every wavefront's part of it is visible, and every wavefront has read K-tile t - 1, whose stage is refilled now
    __syncthreads();
    if (t + S - 1 < ntiles) issue(t + S - 1);
    const char* stage = smem + (t % S) * kStage;
#pragma unroll
    for (int ks = 0; ks < kFewKT / 16; ks++) {
      const u32x4 b = OpB::frag(stage + OpA::kBytes, 32 * wave, ks, lane);
#pragma unroll
      for (int i = 0; i < IM; i++) acc[i] = mfma_32x32x16<BF16>(b, OpA::frag(stage, 32 * i, ks, lane), acc[i]);
    }
  }
}

// One block of the sampled product: its rows in use from the gathered tokens, zeros below.  The value of an element is that
// of the wide tiles bit for bit (the same MFMAs in the same order along k).
template <int IM, bool BK, bool BF16>
__device__ __forceinline__ void sdd_few_block(const SddArgs& g, int p, int r, int c, char* smem) {
  using OpA = Operand<32 * IM, true, kFewKT, kFewThreads>;
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  uint32_t offa[IM];
  OpA::dma_offsets_gathered(offa, wave, lane, g.lda, [&](int row) {
    const int from = gathered_row(g, r * 128 + row);
    return from < 0 ? 0 : from;
  });
  f32x16_t acc[IM] = {};
  const elem_t *a = g.lhs, *b = g.rhs + (int64_t)c * 128 * (BK ? g.ldb : 1);
  const int64_t b_step = BK ? kFewKT : kFewKT * g.ldb;
  few_rows_loop<IM, BK, BF16>(acc, g.k / kFewKT, offa, g.ldb, smem, [&](const elem_t*& ta, const elem_t*& tb) {
    ta = a, tb = b;
    a += kFewKT, b += b_step;
  });
  elem_t* out = g.out + (int64_t)p * 128 * 128;
#pragma unroll
  for (int i = 0; i < IM; i++) {
    const int row = 32 * i + (lane & 31);
    if (gathered_row(g, r * 128 + row) < 0) acc[i] = f32x16_t{};
    else activate_all(acc[i], g.activation);
    elem_t* dst = out + row * 128 + 32 * wave + 4 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; q++)
      *reinterpret_cast<u32x2*>(dst + 8 * q) = u32x2{pack2<BF16>(acc[i][4 * q], acc[i][4 * q + 1]), pack2<BF16>(acc[i][4 * q + 2], acc[i][4 * q + 3])};
  }
}

template <bool BK, bool BF16>
__global__ __launch_bounds__(kFewThreads, 2) void sdd_few_kernel(SddArgs g) {
  extern __shared__ __align__(16) char smem[];
  const int p = xcd_grouped<8>(blockIdx.x, g.nnz);
  const int r = uniform(load_index(g.row_indices, p, g.idx32)), c = uniform(load_index(g.column_indices, p, g.idx32));
  const int rows = uniform(rows_in_use(g.row_slots, g.slots, r, threadIdx.x & 63));
  int stored = 128;
  if (rows == 0) stored = 0;
  else if (rows <= 32) sdd_few_block<1, BK, BF16>(g, p, r, c, smem), stored = 32;
  else if (rows <= 64) sdd_few_block<2, BK, BF16>(g, p, r, c, smem), stored = 64;
  else sdd_few_block<4, BK, BF16>(g, p, r, c, smem);
  u32x4* out = reinterpret_cast<u32x4*>(g.out + (int64_t)p * 128 * 128);
  for (int i = stored * 16 + threadIdx.x; i < 128 * 16; i += kFewThreads) out[i] = u32x4{0u, 0u, 0u, 0u};
}

template <bool BK, bool BF16>
static void launch_sdd_few(const SddArgs& g, hipStream_t stream) {
  static const int once = (set_lds_limit(&sdd_few_kernel<BK, BF16>, kFewLds), 0);
  (void)once;
  hipLaunchKernelGGL((sdd_few_kernel<BK, BF16>), dim3(g.nnz), dim3(kFewThreads), kFewLds, stream, g);
}

void sdd_few(const SddArgs& g, bool bk, bool bf16, hipStream_t stream) {
  if (bk) bf16 ? launch_sdd_few<true, true>(g, stream) : launch_sdd_few<true, false>(g, stream);
  else bf16 ? launch_sdd_few<false, true>(g, stream) : launch_sdd_few<false, false>(g, stream);
}

struct DsdFewArgs {
  const elem_t* data;
  const int32_t* offsets;
  const void* column_indices;
  const elem_t* rhs;
  int64_t ldb;
  int n, tiles, slices, block_rows, idx32;
  const int32_t* row_slots;
  int slots;
  float* sums;   // [slices][slots][n]
};

// 128 columns of a block row times one slice of its blocks; the fp32 sums of row r go to line row_slots[r] of the slice's sums.
template <int IM, bool BK, bool BF16>
__device__ __forceinline__ void dsd_few_tile(const DsdFewArgs& g, int r, int n0, int slice, char* smem) {
  using OpA = Operand<32 * IM, true, kFewKT, kFewThreads>;
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int line = const_ints(g.offsets)[r], blocks = const_ints(g.offsets)[r + 1] - line;
  const int first = line + (int)((int64_t)blocks * slice / g.slices), last = line + (int)((int64_t)blocks * (slice + 1) / g.slices);
  uint32_t offa[IM];
  OpA::dma_offsets(offa, wave, lane, 128);
  f32x16_t acc[IM] = {};
  int t = 0, columns = 0;   // lane l holds the block column of entry first + t / 2 / 64 * 64 + l
  few_rows_loop<IM, BK, BF16>(acc, 2 * (last - first), offa, g.ldb, smem, [&](const elem_t*& a, const elem_t*& b) {
    const int e = t >> 1, half = (t & 1) * kFewKT;
    if ((t & 127) == 0) columns = first + e + lane < last ? load_index(g.column_indices, first + e + lane, g.idx32) : 0;
    const int64_t k = (int64_t)__builtin_amdgcn_readlane(columns, e & 63) * 128 + half;
    a = g.data + (int64_t)(first + e) * 128 * 128 + half;
    b = g.rhs + (BK ? (int64_t)n0 * g.ldb + k : k * g.ldb + n0);
    t++;
  });
#pragma unroll
  for (int i = 0; i < IM; i++) {
    const int slot = g.row_slots[(int64_t)r * 128 + 32 * i + (lane & 31)];
    if ((unsigned)slot >= (unsigned)g.slots) continue;
    float* dst = g.sums + ((int64_t)slice * g.slots + slot) * g.n + n0 + 32 * wave + 4 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; q++) *reinterpret_cast<float4*>(dst + 8 * q) = float4{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
  }
}

template <bool BK, bool BF16>
__global__ __launch_bounds__(kFewThreads, 2) void dsd_few_kernel(DsdFewArgs g) {
  extern __shared__ __align__(16) char smem[];
  const int bid = xcd_grouped<8>(blockIdx.x, gridDim.x);
  const int tile = bid % g.tiles, rest = bid / g.tiles, slice = rest % g.slices, r = rest / g.slices;
  const int n0 = edge_start(tile, 128, g.n);
  const int rows = uniform(rows_in_use(g.row_slots, g.slots, r, threadIdx.x & 63));
  if (rows == 0) return;
  if (rows <= 32) dsd_few_tile<1, BK, BF16>(g, r, n0, slice, smem);
  else if (rows <= 64) dsd_few_tile<2, BK, BF16>(g, r, n0, slice, smem);
  else dsd_few_tile<4, BK, BF16>(g, r, n0, slice, smem);
}

template <bool BK, bool BF16>
static void launch_dsd_few(const DsdFewArgs& g, hipStream_t stream) {
  static const int once = (set_lds_limit(&dsd_few_kernel<BK, BF16>, kFewLds), 0);
  (void)once;
  hipLaunchKernelGGL((dsd_few_kernel<BK, BF16>), dim3(g.block_rows * g.tiles * g.slices), dim3(kFewThreads), kFewLds, stream, g);
}

// Slices along k: workgroups for two rounds of two per compute unit, slices of four blocks or more.
static int few_slices(int64_t block_rows, int64_t n, int64_t nnz) {
  const int64_t tiles = block_rows * ((n + 127) / 128), want = 4 * (int64_t)compute_units(), blocks = nnz / block_rows;
  const int64_t s = tiles > 0 ? (want + tiles - 1) / tiles : 1, most = blocks / 4 < 8 ? blocks / 4 : 8;
  return (int)(s < most ? s : most > 1 ? most : 1);
}

}  // namespace stk

extern "C" int64_t stk_dsd_scatter_few_bytes(int64_t m, int64_t n, int64_t nnz, int64_t slots) {
  using namespace stk;
  if (m <= 0 || m % 128 || n < 128 || n % 64 || nnz <= 0 || slots <= 0 || !few_rows_dsd(slots, m / 128, n)) return 0;
  return (int64_t)sizeof(float) * few_slices(m / 128, n, nnz) * slots * n;
}

extern "C" int stk_dsd_scatter_few(int64_t m, int64_t k, int64_t n, const void* data, const int32_t* offsets, const void* column_indices,
                                   const void* rhs, int64_t rhs_stride_k, int64_t rhs_stride_n, const int32_t* row_slots,
                                   const int32_t* slot_rows, const float* weights, int top_k, int64_t num_tokens, void* out,
                                   int64_t out_stride_m, int64_t nnz, int blocking, int dtype, int index_dtype, void* workspace,
                                   int64_t workspace_bytes, stk_stream_t stream) {
  using namespace stk;
  const char* who = "stk_dsd_scatter_few";
  if (blocking != 128) return fail(STK_ERR_UNSUPPORTED, "%s: blocking %d (128 only)", who, blocking);
  if (dtype != STK_F16 && dtype != STK_BF16) return fail(STK_ERR_UNSUPPORTED, "%s: dtype %d", who, dtype);
  if (index_dtype != STK_I16 && index_dtype != STK_I32) return fail(STK_ERR_UNSUPPORTED, "%s: index dtype %d", who, index_dtype);
  if (m < 0 || k < 0 || n < 0 || nnz < 0 || num_tokens < 0 || top_k < 1 || num_tokens > INT32_MAX / top_k)
    return fail(STK_ERR_DIMS, "%s: sizes", who);
  if (m % 128 || k % 128)
    return fail(STK_ERR_DIMS, "incompatible dimensions: sparse [%lld, %lld] x dense [%lld, %lld] with blocking %d", (long long)m, (long long)k, (long long)k,
                (long long)n, blocking);
  const int64_t slots = num_tokens * top_k, need = stk_dsd_scatter_few_bytes(m, n, nnz, slots);
  if (need == 0) return fail(STK_ERR_UNSUPPORTED, "%s: needs few slots per block row and 128 columns or more, a multiple of 64", who);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return fail(STK_ERR_WORKSPACE, "%s: needs %lld bytes, 16-byte aligned", who, (long long)need);
  if (!data || !offsets || !column_indices || !rhs || !row_slots || !slot_rows || !out) return fail(STK_ERR_DIMS, "%s: missing pointer", who);
  const bool bk = rhs_stride_n != 1;
  if (bk && rhs_stride_k != 1) return fail(STK_ERR_UNSUPPORTED, "%s: rhs needs a unit stride", who);
  const int64_t ldb = bk ? rhs_stride_n : rhs_stride_k;
  if (ldb % 8 || ldb >= (1 << 24) || out_stride_m % 8 || !aligned16(rhs) || !aligned16(out) || !aligned16(data))
    return fail(STK_ERR_UNSUPPORTED, "%s: operands need 16-byte aligned bases and leading dimensions divisible by 8, below 2^24", who);
  const int tiles = (int)((n + 127) / 128), slices = few_slices(m / 128, n, nnz);
  if (m / 128 * tiles * slices > INT32_MAX) return fail(STK_ERR_UNSUPPORTED, "%s: size exceeds 32-bit range", who);
  const DsdFewArgs g{static_cast<const elem_t*>(data), offsets, column_indices, static_cast<const elem_t*>(rhs), ldb, (int)n, tiles, slices, (int)(m / 128),
                     index_dtype == STK_I32, row_slots, (int)slots, static_cast<float*>(workspace)};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool bf16 = dtype == STK_BF16;
  if (bk) bf16 ? launch_dsd_few<true, true>(g, s) : launch_dsd_few<true, false>(g, s);
  else bf16 ? launch_dsd_few<false, true>(g, s) : launch_dsd_few<false, false>(g, s);
  const int rc = check_launch(who);
  if (rc != STK_OK) return rc;
  return scatter_sums(g.sums, slices, slots, n, slot_rows, m, weights, top_k, num_tokens, out, out_stride_m, dtype, s);
}
