// The two products of a routed layer whose block rows hold few tokens each (a decoding step, a small batch over many
// experts): stk_sdd_gather and stk_dsd_scatter_few.  With a few token rows in a block of 128 a product is one pass over
// the experts' weights, and what bounds it is how many bytes of them are in flight.  The tiles here therefore compute only
// the 32, 64 or 128 rows that reach to the last token of a block row, one panel of 128 columns of weights per workgroup of four
// wavefronts, with a ring of 80 KB and two workgroups per compute unit: one's start and stores lie under the other's stream, and
// the many short tiles leave no long last round.  On 32 rows that is three 16 KB stages of weights in flight per workgroup, on
// 64 two, on 128 one (four of 32-deep K-tiles instead: 118 -> 140 us for the second product of 4096 tokens over 64 experts).
// 128 tokens over 58 of 64 experts (1024 x 4096, bf16, 487 MB of weights a product): the wide tiles take 114 us for the first
// product and 104 for the second with its scatter, these 100 (with the 61 MB of its result 5.5 TB/s) and 82 (5.9 TB/s); 300 tokens
// top-2 over 16 experts (2048 x 8192) 105 and 128 us, these 104 and 94; 16 tokens top-2 over 8 experts (1024 x 4096) 20 and
// 65 us, these 15 and 24.  Row-major weights are loaded non-temporally (without the hint the first product takes 15 us more), K-major
// ones are not.  With the workgroups in plain order the second product takes 9 us more; in eight contiguous shares of the list
// as long, but 70 instead of 46 us where four experts share the block rows unevenly.
#include "dsd_tile.h"
#include "few_rows.h"
#include "sdd_tile.h"

namespace stk {

constexpr int kFewThreads = 256;
constexpr int kFewKT = 64;
constexpr int kFewLds = 80 * 1024;   // two workgroups share the 160 KB of a compute unit

// Rows that end with the last row of a block row that holds a token, 0 .. 128.
__device__ __forceinline__ int rows_in_use(const int32_t* row_slots, int slots, int block_row, int lane) {
  const int32_t* s = row_slots + (int64_t)block_row * 128;
  const uint64_t lo = __ballot((unsigned)s[lane] < (unsigned)slots), hi = __ballot((unsigned)s[64 + lane] < (unsigned)slots);
  return hi ? 128 - __builtin_clzll(hi) : lo ? 64 - __builtin_clzll(lo) : 0;
}

// At most `younger` of the K-tiles behind this one are still in flight: this one has landed.
template <int MOST, int LOADS>
__device__ __forceinline__ void wait_younger(int younger) {
  if constexpr (MOST > 0) {
    if (younger < MOST) return wait_younger<MOST - 1, LOADS>(younger);
  }
  wait_vmcnt<MOST * LOADS>();
}

// Four wavefronts on a tile of 32 IM rows and TN columns, TN / 32 of them side by side, the others below with their share of
// the rows (with 32 rows of 64 columns two of them only load).  On 64 columns four more do the loading: issuing the transfers
// takes as long as multiplying, and a workgroup that has a compute unit to itself would do one behind the other (second product of
// 4 experts of 256 x 8192 41 -> 34 us, 16 of 256 x 4096 24 -> 20, 8 of 1024 x 4096 the same).
template <int IM, int TN, bool BK>
struct FewTile {
  using OpA = Operand<32 * IM, true, kFewKT, kFewThreads>;
  using OpB = Operand<TN, BK, kFewKT, kFewThreads>;
  static constexpr int kAcross = TN / 32, kDown = 4 / kAcross, kMine = IM < kDown ? 1 : IM / kDown;   // row strips of 32 a wavefront
  static constexpr int kStage = OpA::kBytes + OpB::kBytes, kStages = kFewLds / kStage, kLoads = IM + OpB::kSlicesPerWave;
  static_assert(OpA::kSlicesPerWave == IM && kStages >= 2 && (kStages - 2) * kLoads < 64, "the ring");
  static constexpr bool kLoaders = TN == 64;
  static constexpr int kThreads = kLoaders ? 512 : 256;
  int lane, wave, column, strip;   // of this wavefront: its number among the four, first column, first strip
  bool loads, multiplies;
  __device__ __forceinline__ FewTile() {
    lane = threadIdx.x & 63;
    const int all = uniform(threadIdx.x >> 6);
    wave = all & 3, loads = !kLoaders || all >= 4;
    column = 32 * (wave % kAcross), strip = wave / kAcross * kMine, multiplies = all < 4 && strip < IM;
  }
};

// acc += A x B over ntiles K-tiles.  offa: the lanes' offsets of the A transfers; next(a, b) sets the origins of the next
// K-tile, in increasing order; done(t) is called behind the sums of K-tile t.
template <class Tile, bool BK, bool BF16, class Next, class Done>
__device__ __forceinline__ void few_rows_loop(const Tile& w, f32x16_t (&acc)[Tile::kMine], int ntiles, const uint32_t (&offa)[Tile::OpA::kSlicesPerWave],
                                              int64_t ldb, char* smem, Next&& next, Done&& done) {
  using OpA = typename Tile::OpA;
  using OpB = typename Tile::OpB;
  constexpr int S = Tile::kStages;
  const uint32_t lds0 = (uint32_t)(uintptr_t)((STK_LDS char*)smem);
  uint32_t offb[OpB::kSlicesPerWave];
  OpB::dma_offsets(offb, w.wave, w.lane, ldb);
  int fill = 0, use = 0;   // stages of the ring
  auto issue = [&]() {
    const elem_t *a, *b;
    next(a, b);
    const gptr_t ga = uniform_global(a), gb = uniform_global(b);
    const uint32_t stage = lds0 + (uint32_t)fill * Tile::kStage;
    fill = fill + 1 == S ? 0 : fill + 1;
#pragma unroll
    for (int i = 0; i < OpB::kSlicesPerWave; i++) dma16<!BK>(gb, offb[i], stage + OpA::kBytes + (i * 4 + w.wave) * 1024);
#pragma unroll
    for (int i = 0; i < OpA::kSlicesPerWave; i++) dma16(ga, offa[i], stage + (i * 4 + w.wave) * 1024);
  };
  if (w.loads)
    for (int t = 0; t < S - 1 && t < ntiles; t++) issue();
  for (int t = 0; t < ntiles; t++) {
    // K-tile t has landed; up to S - 2 younger ones stay in flight
    if (w.loads) wait_younger<S - 2, Tile::kLoads>(ntiles - 1 - t);
    // every wavefront's part of it is visible, and every wavefront has read K-tile t - 1, whose stage is refilled now
    __syncthreads();
    if (w.loads && t + S - 1 < ntiles) issue();
    const char* stage = smem + use * Tile::kStage;
    use = use + 1 == S ? 0 : use + 1;
    if (w.multiplies) {
#pragma unroll
      for (int ks = 0; ks < kFewKT / 16; ks++) {
        const u32x4 b = OpB::frag(stage + OpA::kBytes, w.column, ks, w.lane);
#pragma unroll
        for (int i = 0; i < Tile::kMine; i++) acc[i] = mfma_32x32x16<BF16>(b, OpA::frag(stage, 32 * (w.strip + i), ks, w.lane), acc[i]);
      }
    }
    done(t);
  }
}

// One block of the sampled product: its rows in use from the gathered tokens, zeros below.  The value of an element is that
// of the wide tiles bit for bit (the same MFMAs in the same order along k).
template <int IM, bool BK, bool BF16>
__device__ __forceinline__ void sdd_few_block(const SddArgs& g, int p, int r, int c, char* smem) {
  using Tile = FewTile<IM, 128, BK>;
  const Tile w;
  uint32_t offa[Tile::OpA::kSlicesPerWave];
  Tile::OpA::dma_offsets_gathered(offa, w.wave, w.lane, g.lda, [&](int row) {
    const int from = gathered_row(g, r * 128 + row);
    return from < 0 ? 0 : from;
  });
  f32x16_t acc[IM] = {};
  const elem_t *a = g.lhs, *b = g.rhs + (int64_t)c * 128 * (BK ? g.ldb : 1);
  const int64_t b_step = BK ? kFewKT : kFewKT * g.ldb;
  auto next = [&](const elem_t*& ta, const elem_t*& tb) {
    ta = a, tb = b;
    a += kFewKT, b += b_step;
  };
  few_rows_loop<Tile, BK, BF16>(w, acc, g.k / kFewKT, offa, g.ldb, smem, next, [](int) {});
  elem_t* out = g.out + (int64_t)p * 128 * 128;
#pragma unroll
  for (int i = 0; i < IM; i++) {
    const int row = 32 * i + (w.lane & 31);
    if (gathered_row(g, r * 128 + row) < 0) acc[i] = f32x16_t{};
    else activate_all(acc[i], g.activation);
    elem_t* dst = out + row * 128 + w.column + 4 * (w.lane >> 5);
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
  int n, tiles, block_rows, idx32;
  const int32_t* row_slots;
  int slots;
  float* sums;        // [slots][n]
  PlanLists plan;     // of the block rows, and the last round of the stk_dsd whose sums these are
  int units, capacity;   // capacity 0: it cuts none of its tiles
};

// The sums here are those of stk_dsd bit for bit.  They follow k in the same order, and where stk_dsd cuts the tile that the
// columns from n0 on of block row r are in, they are cut at the same blocks and the parts added up in the same order: how
// many parts these are.  The tiles of the last round are at most one per compute unit, four for every lane.
__device__ __forceinline__ int slices_of_tile(const DsdFewArgs& g, int r, int n0, int lane) {
  if (g.capacity == 0) return 1;
  const TailRound round = tail_round(g.plan, g.n, g.units, g.capacity);
  if (round.slices == 1) return 1;
  bool cut = false;
  for (int item = round.whole + lane; item < round.tiles; item += 64) {
    const LineTile t = tail_round_tile(g.plan, g.n, round, item);
    cut |= t.line <= r && r < t.line + t.lines && t.column == n0 / (t.lines == 3 ? kTailTile / 2 : kTailTile);
  }
  return __ballot(cut) ? round.slices : 1;
}

// TN columns of a block row; the fp32 sums of row r go to line row_slots[r] of the sums.
template <int IM, int TN, bool BK, bool BF16>
__device__ __forceinline__ void dsd_few_tile(const DsdFewArgs& g, int r, int rows, int n0, char* smem) {
  using Tile = FewTile<IM, TN, BK>;
  const Tile w;
  const int first = const_ints(g.offsets)[r], blocks = const_ints(g.offsets)[r + 1] - first;
  int slices = slices_of_tile(g, r, n0, w.lane);
  if (slices > blocks) slices = blocks > 1 ? blocks : 1;
  uint32_t offa[Tile::OpA::kSlicesPerWave];
  // (rows behind the last one in use: the lines of the first one again; 16 experts of 2048 x 8192 91 -> 85 us)
  Tile::OpA::dma_offsets_gathered(offa, w.wave, w.lane, 128, [&](int row) { return row < rows ? row : 0; });
  constexpr int kMine = Tile::kMine, kPer = 128 / kFewKT;   // pieces of a block
  f32x16_t acc[kMine] = {}, sum[kMine] = {};
  int t = 0, columns = 0;   // lane l holds the block column of entry t / kPer / 64 * 64 + l
  auto next = [&](const elem_t*& a, const elem_t*& b) {
    const int e = t / kPer, part = t % kPer * kFewKT;
    if (t % (64 * kPer) == 0) {
      columns = e + w.lane < blocks ? load_index(g.column_indices, first + e + w.lane, g.idx32) : 0;
      // (awaited here: a wait at the lane read below, in every K-tile, would empty the ring)
      asm volatile("" : "+v"(columns));
    }
    const int64_t k = (int64_t)__builtin_amdgcn_readlane(columns, e & 63) * 128 + part;
    a = g.data + (int64_t)(first + e) * 128 * 128 + part;
    b = g.rhs + (BK ? (int64_t)n0 * g.ldb + k : k * g.ldb + n0);
    t++;
  };
  int slice = 0, end = kPer * (blocks / slices);
  auto done = [&](int i) {
    if (i + 1 != end) return;
#pragma unroll
    for (int j = 0; j < kMine; j++) {
      if (slice == 0) sum[j] = acc[j];
      else sum[j] += acc[j];
      acc[j] = f32x16_t{};
    }
    slice++;
    end = kPer * ((slice + 1) * blocks / slices);
  };
  few_rows_loop<Tile, BK, BF16>(w, acc, kPer * blocks, offa, g.ldb, smem, next, done);
  if (!w.multiplies) return;
#pragma unroll
  for (int i = 0; i < kMine; i++) {
    const int slot = g.row_slots[(int64_t)r * 128 + 32 * (w.strip + i) + (w.lane & 31)];
    if ((unsigned)slot >= (unsigned)g.slots) continue;
    float* dst = g.sums + (int64_t)slot * g.n + n0 + w.column + 4 * (w.lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; q++) *reinterpret_cast<float4*>(dst + 8 * q) = float4{sum[i][4 * q], sum[i][4 * q + 1], sum[i][4 * q + 2], sum[i][4 * q + 3]};
  }
}

template <int TN, bool BK, bool BF16>
__global__ __launch_bounds__((FewTile<1, TN, BK>::kThreads), (FewTile<1, TN, BK>::kThreads / 128)) void dsd_few_kernel(DsdFewArgs g) {
  extern __shared__ __align__(16) char smem[];
  const int bid = xcd_grouped<8>(blockIdx.x, gridDim.x), r = bid / g.tiles, n0 = bid % g.tiles * TN;
  const int rows = uniform(rows_in_use(g.row_slots, g.slots, r, threadIdx.x & 63));
  if (rows == 0) return;
  if (rows <= 32) dsd_few_tile<1, TN, BK, BF16>(g, r, rows, n0, smem);
  else if (rows <= 64) dsd_few_tile<2, TN, BK, BF16>(g, r, rows, n0, smem);
  else dsd_few_tile<4, TN, BK, BF16>(g, r, rows, n0, smem);
}

template <int TN, bool BK, bool BF16>
static void launch_dsd_few(const DsdFewArgs& g, hipStream_t stream) {
  static const int once = (set_lds_limit(&dsd_few_kernel<TN, BK, BF16>, kFewLds), 0);
  (void)once;
  hipLaunchKernelGGL((dsd_few_kernel<TN, BK, BF16>), dim3(g.block_rows * g.tiles), dim3(FewTile<1, TN, BK>::kThreads), kFewLds, stream, g);
}
template <int TN>
static void launch_dsd_few(const DsdFewArgs& g, bool bk, bool bf16, hipStream_t stream) {
  if (bk) bf16 ? launch_dsd_few<TN, true, true>(g, stream) : launch_dsd_few<TN, true, false>(g, stream);
  else bf16 ? launch_dsd_few<TN, false, true>(g, stream) : launch_dsd_few<TN, false, false>(g, stream);
}

// Columns of a tile: 128, or 64 where that would leave more than a quarter of the compute units without one.  With 64, half of
// what a workgroup moves per K-tile is the token rows, which wider tiles share.  us with 128 / 64 columns, and where the work
// allows it two steps: 64 tiles of 128 (8 experts, 1024 columns, 4096 deep) 31 / 24, two steps 65; 128 tiles (16 experts)
// 34 / 30, 68; 216 (27 of 32 experts) 41 / 50, 76; 240 (15 experts, 2048 columns, 8192 deep) 85 / 100, 120.  32 columns are as
// slow as 64 or slower everywhere.  The sums of a tile cannot be split over k between workgroups without another order, and a
// compute unit by itself takes in 40 - 60 GB/s: with up to eight slices 8 experts of 1024 x 4096 took 20 us, 8 of
// 512 x 8192 23, now 40 (two steps 117), 4 of 256 x 8192 21, now 34 (112).
static int few_columns(int64_t block_rows, int64_t n) { return n % 128 == 0 && block_rows * (n / 128) >= compute_units() * 3 / 4 ? 128 : 64; }

}  // namespace stk

extern "C" int64_t stk_dsd_scatter_few_bytes(int64_t m, int64_t n, int64_t nnz, int64_t slots) {
  using namespace stk;
  if (m <= 0 || m % 128 || n < 128 || n % 64 || nnz <= 0 || slots <= 0 || !few_rows_dsd(slots, m / 128, n)) return 0;
  return (int64_t)sizeof(float) * slots * n;
}

extern "C" int stk_dsd_scatter_few(int64_t m, int64_t k, int64_t n, const void* data, const int32_t* offsets, const void* column_indices,
                                   const void* rhs, int64_t rhs_stride_k, int64_t rhs_stride_n, const int32_t* row_slots,
                                   const int32_t* slot_rows, const float* weights, int top_k, int64_t num_tokens, void* out,
                                   int64_t out_stride_m, int64_t nnz, int blocking, int dtype, int index_dtype, void* workspace,
                                   int64_t workspace_bytes, stk_stream_t stream) {
  return stk_dsd_scatter_few_as_cut(m, k, n, data, offsets, column_indices, rhs, rhs_stride_k, rhs_stride_n, row_slots, slot_rows, weights, top_k,
                                    num_tokens, out, out_stride_m, nnz, blocking, dtype, index_dtype, workspace, workspace_bytes, nullptr, 0, stream);
}

extern "C" int stk_dsd_scatter_few_as_cut(int64_t m, int64_t k, int64_t n, const void* data, const int32_t* offsets, const void* column_indices,
                                          const void* rhs, int64_t rhs_stride_k, int64_t rhs_stride_n, const int32_t* row_slots,
                                          const int32_t* slot_rows, const float* weights, int top_k, int64_t num_tokens, void* out,
                                          int64_t out_stride_m, int64_t nnz, int blocking, int dtype, int index_dtype, void* workspace,
                                          int64_t workspace_bytes, const uint8_t* plan, int64_t dsd_workspace_bytes, stk_stream_t stream) {
  using namespace stk;
  const char* who = "stk_dsd_scatter_few";
  if (blocking != 128) return fail(STK_ERR_UNSUPPORTED, "%s: blocking %d (128 only)", who, blocking);
  if (top_k < 1 || num_tokens < 0 || num_tokens > INT32_MAX / top_k) return fail(STK_ERR_DIMS, "%s: %lld tokens, top_k %d", who, (long long)num_tokens, top_k);
  DsdProblem problem;
  const int rc = dsd_problem(who, m, k, n, data, offsets, column_indices, nullptr, nullptr, nullptr, 0, rhs, rhs_stride_k, rhs_stride_n, out,
                             out_stride_m, nnz, blocking, dtype, index_dtype, plan, &problem);
  if (rc != STK_OK) return rc;
  const int64_t slots = num_tokens * top_k, need = stk_dsd_scatter_few_bytes(m, n, nnz, slots);
  if (need == 0) return fail(STK_ERR_UNSUPPORTED, "%s: needs few slots per block row and 128 columns or more, a multiple of 64", who);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return fail(STK_ERR_WORKSPACE, "%s: needs %lld bytes, 16-byte aligned", who, (long long)need);
  if (!rhs || !row_slots || !slot_rows || !out) return fail(STK_ERR_DIMS, "%s: missing pointer", who);
  const DsdArgs& p = problem.g;
  const int columns = few_columns(p.block_rows, n);
  const DsdFewArgs g{p.data, p.walk_offsets, p.walk_columns, p.rhs, p.ldb, p.n, p.n / columns, p.block_rows, p.idx32, row_slots, (int)slots,
                     static_cast<float*>(workspace), problem.lists, compute_units(), plan ? tail_capacity(false, p.block_rows, n, nnz, dsd_workspace_bytes) : 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool bf16 = dtype == STK_BF16;
  if (columns == 128) launch_dsd_few<128>(g, problem.bk, bf16, s);
  else launch_dsd_few<64>(g, problem.bk, bf16, s);
  const int launched = check_launch(who);
  if (launched != STK_OK) return launched;
  return scatter_sums(g.sums, slots, n, slot_rows, m, weights, top_k, num_tokens, out, out_stride_m, dtype, s);
}

extern "C" int stk_dsd_cuts(int64_t m, int64_t n, int64_t nnz, int64_t workspace_bytes) {
  using namespace stk;
  return m > 0 && m % 128 == 0 && n > 0 && tail_capacity(false, m / 128, n, nnz, workspace_bytes) > 0;
}
