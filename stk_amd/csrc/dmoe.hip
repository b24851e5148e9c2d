// Topology of a dropless mixture-of-experts layer, and its fusion plan, in one launch.
//
// Block-diagonal pattern: expert e owns the block rows [first_e, first_e + R_e) given by the padded bins and the `width`
// block columns starting at e * width.  Everything is a closed form of (block row, expert):
//   block p = i * width + j          row_indices[p] = i, column_indices[p] = e(i) * width + j
//   offsets[i] = i * width
//   column c = e * width + j         offsets_t[c] = first_e * width + j * R_e
//   entry r of that column           column_indices_t = first_e + r, block_offsets_t = (first_e + r) * width + j
// which is also what a stable sort by column of the (row, column) pairs gives.
//
// So is the fusion plan (plan.hip says what it holds): the rows of an expert repeat each other, and so do its columns
// if it has rows, and no line repeats a line of another expert.  The groups that a run of n identical lines is cut into
// depend on n alone, so every list of the plan is the experts' shares one behind the other - the lists of columns with
// the experts in order of descending R_e - and its entries can be written by any thread once the shares have been
// added up.  Every workgroup adds them up for itself (a few hundred values from LDS); stk_build_plan, which has to find
// the runs by comparing the lines, takes two launches and a single workgroup per direction for what follows from them.
// 20096 rows over 64 experts of 32 block columns: 16.7 us for both, against 4 us for the topology and 31 us for the
// two launches of stk_build_plan; it is latency, not bandwidth, on either side.
#include "common.h"
#include "plan_sim.h"
#include "wave_scan.h"

namespace stk {

__device__ __forceinline__ int uniform_int(int v) { return __builtin_amdgcn_readfirstlane(v); }

constexpr int kPlanExperts = 1024;   // experts whose shares fit the LDS of a workgroup
constexpr int kSortedLines = 4096;   // longer lists keep the experts in ascending order, as in stk_build_plan

struct DmoeArgs {
  const int32_t* bins;
  int experts, blocking, block_rows, width;
  int32_t* offsets;
  void* row_indices;
  void* column_indices;
  int32_t* offsets_t;
  void* column_indices_t;
  int32_t* block_offsets_t;
  // the plan: the tiles of stk_sdd, and what lies behind them (null: no plan)
  int32_t* sdd;
  uint8_t* plan;
  int64_t max_sdd_tiles;
  int compute_units;
};

// First block row of expert e; the rows past the last bin belong to the last expert, bins that claim more rows than there
// are, or less than none, stay inside the arrays.
__device__ __forceinline__ int first_row_of(const DmoeArgs& g, int e) {
  if (e == 0) return 0;
  if (e == g.experts) return g.block_rows;
  const int r = g.bins[e - 1] / g.blocking;
  return r < 0 ? 0 : r < g.block_rows ? r : g.block_rows;
}

// Groups of a run of n identical lines, by the plan list that holds their first lines.  FOURS: the plan of 64-blocks.
struct RunGroups {
  int count[kPlanLists];
};
template <bool FOURS>
__device__ __forceinline__ RunGroups groups_of_run(int n, bool heavy) {
  RunGroups g{{0, 0, 0, 0, 0}};
  if (n <= 0) return g;
  if constexpr (!FOURS) {
    const bool three = (n & 1) && n >= 3;
    g.count[kPairs] = n / 2;
    g.count[kSingles] = n & 1;
    g.count[kTallPairs] = three ? (n - 3) / 2 : n / 2;
    g.count[kTallTriples] = three;
    g.count[kTallSingles] = n == 1;
  } else if (heavy) {
    g.count[kTallPairs] = n / 2;
    g.count[kTallSingles] = n & 1;
  } else {
    const int q = n / 4, r = n & 3;
    const bool five = r == 1 && q >= 1;   // the last five lines: a three and a pair
    g.count[kPairs] = five ? q - 1 : q;
    g.count[kTallTriples] = five || r == 3;
    g.count[kTallPairs] = five || r == 2;
    g.count[kTallSingles] = n == 1;
  }
  return g;
}
// First line, counted from the start of the run, of group `i` of list `kind`.
template <bool FOURS>
__device__ __forceinline__ int line_of_group(int n, bool heavy, int kind, int i) {
  if constexpr (!FOURS) {
    if (kind == kTallTriples) return n - 3;
    if (kind == kSingles) return n - 1;
    return kind == kTallSingles ? 0 : 2 * i;
  } else {
    if (heavy) return kind == kTallSingles ? n - 1 : 2 * i;
    const int q = n / 4, r = n & 3;
    const bool five = r == 1 && q >= 1;
    if (kind == kTallTriples) return five ? 4 * (q - 1) : 4 * q;
    if (kind == kTallPairs) return five ? 4 * (q - 1) + 3 : 4 * q;
    return 4 * i;   // (a lone line is its run's only one)
  }
}

// The shares of the experts in the ten lists of the plan and in the tile list of stk_sdd.  n and heavy of a direction are
// those of an expert's run: R_e rows of `width` blocks, or `width` columns of R_e blocks.
template <bool FOURS>
struct DmoePlan {
  const DmoeArgs& g;
  const int* first;   // [experts + 1], LDS
  __device__ __forceinline__ int rows_of(int e) const {
    const int n = first[e + 1] - first[e];
    return n > 0 ? n : 0;
  }
  __device__ __forceinline__ bool heavy(int blocks) const {
    const int64_t nnz = (int64_t)g.block_rows * g.width, share = nnz * 4 / (g.compute_units > 0 ? g.compute_units : 1);
    return FOURS && 4 * (int64_t)blocks > (share > 1 ? share : 1);
  }
  // how many groups of list `kind` expert e has in the direction
  __device__ __forceinline__ int share(bool cols, int kind, int e) const {
    const int rows = rows_of(e);
    if (!cols) return groups_of_run<FOURS>(rows, heavy(g.width)).count[kind];
    if (rows == 0) return (kind == kTallSingles || (!FOURS && kind == kSingles)) ? g.width : 0;   // empty columns: lone lines
    return groups_of_run<FOURS>(g.width, heavy(rows)).count[kind];
  }
  __device__ __forceinline__ int line(bool cols, int kind, int e, int i) const {
    const int rows = rows_of(e);
    if (!cols) return first[e] + line_of_group<FOURS>(rows, heavy(g.width), kind, i);
    return e * g.width + (rows == 0 ? i : line_of_group<FOURS>(g.width, heavy(rows), kind, i));
  }
  // Tiles of stk_sdd: an expert's groups of rows from the top, every group in tiles of up to `wide` blocks
  // (pairs and fours: 2 or 4; groups of three with 128-blocks: 1)
  static constexpr int kWide = FOURS ? 4 : 2, kWideOfThree = FOURS ? 4 : 1;
  __device__ __forceinline__ int sdd_tiles(int e) const {
    const RunGroups r = groups_of_run<FOURS>(rows_of(e), false);
    const int wide = (g.width + kWide - 1) / kWide, three = (g.width + kWideOfThree - 1) / kWideOfThree;
    return (FOURS ? r.count[kPairs] : 0) * wide + r.count[kTallPairs] * wide + r.count[kTallTriples] * three + r.count[kTallSingles] * wide;
  }
  __device__ __forceinline__ void sdd_tile(int e, int t, int32_t* at) const {
    const int n = rows_of(e);
    const RunGroups r = groups_of_run<FOURS>(n, false);
    const int wide = (g.width + kWide - 1) / kWide;
    const int whole = r.count[FOURS ? kPairs : kTallPairs];   // groups of the largest height, in front
    int rows = kWide, row, step = kWide;
    if (t < whole * wide) {
      row = t / wide * kWide;
      t %= wide;
    } else {
      t -= whole * wide;
      row = whole * kWide;
      const int three = (g.width + kWideOfThree - 1) / kWideOfThree;
      if (r.count[kTallTriples] && t < three) {
        rows = 3, step = kWideOfThree;
      } else {
        if (r.count[kTallTriples]) t -= three, row += 3;
        rows = n - row;   // a pair behind the fours, or a lone row
      }
    }
    const int j = t * step, left = g.width - j;
    at[0] = (first[e] + row) * g.width + j;
    at[1] = rows | ((left < step ? left : step) << 8);
  }
};

// Last i in [0, n) with at(i) <= x (ascending; at(0) <= x).
template <class At>
__device__ __forceinline__ int last_not_above(At&& at, int n, int x) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (at(mid) <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}

// LDS of a workgroup that builds the plan (in this order, four-byte words)
struct DmoeLds {
  int* first;     // [experts + 1] first block rows
  int* order;     // [experts] in order of descending R_e (255 at most counted), equal ones ascending
  int* base;      // [10][experts] entries of a list in front of the share of the o-th expert of the list's order
  int* tiles;     // [experts] tiles of stk_sdd in front of expert e's
  int* count;     // [11] entries of the lists, rows first; tiles of stk_sdd
  int* blocks;    // [10] blocks of one line per entry
  int* longest;   // [10] blocks of a line of the first entry
  float* ends;    // [kMaxTailSlices]
  uint32_t* keys; // [(experts + 3) / 4] min(R_e, 255), a byte each
  static __host__ __device__ size_t bytes(int experts) { return sizeof(int) * (13 * (size_t)experts + 1 + 31 + kMaxTailSlices + (experts + 3) / 4); }
  __device__ DmoeLds(int* p, int E)
      : first(p), order(p + E + 1), base(order + E), tiles(base + 10 * E), count(tiles + E), blocks(count + 11), longest(blocks + 10),
        ends(reinterpret_cast<float*>(longest + 10)), keys(reinterpret_cast<uint32_t*>(ends + kMaxTailSlices)) {}
};

template <bool FOURS>
__device__ __forceinline__ void dmoe_plan(const DmoeArgs& g, const DmoeLds& s, int group, int64_t thread, int64_t threads) {
  const int E = g.experts, width = g.width, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const DmoePlan<FOURS> plan{g, s.first};
  for (int w = tid; w < (E + 3) / 4; w += 256) {
    uint32_t v = 0;
    for (int i = 0; i < 4; i++)
      if (4 * w + i < E) v |= (uint32_t)min(plan.rows_of(4 * w + i), 255) << (8 * i);
    s.keys[w] = v;
  }
  __syncthreads();
  for (int e = tid; e < E; e += 256) {
    const int mine = min(plan.rows_of(e), 255);
    int rank = 0;
    for (int w = 0; w < (E + 3) / 4; w++) {   // (the bytes behind the last expert count as no rows and lie behind e)
      const uint32_t v = s.keys[w];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int other = (v >> (8 * i)) & 0xff;
        rank += other > mine || (other == mine && 4 * w + i < e);
      }
    }
    s.order[rank] = e;
  }
  // the rows' lists and the tiles of stk_sdd do not need the order; wavefront w adds up the lists w, w + 4, w + 8
  __syncthreads();
  for (int l = wave; l <= 10; l += 4) {
    const bool cols = l >= kPlanLists;
    const int kind = l % kPlanLists;
    int total = 0;
    if (l == 10 || !cols) {
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        const int n = e >= E ? 0 : l == 10 ? plan.sdd_tiles(e) : plan.share(false, kind, e);
        const int inc = wave_inclusive_scan(n, lane);
        if (e < E) (l == 10 ? s.tiles : s.base + l * E)[e] = total + inc - n;
        total += __shfl(inc, 63, 64);
      }
      if (lane == 0) {
        s.count[l] = total;
        if (l < 10) s.blocks[l] = total * width, s.longest[l] = width;
      }
      continue;
    }
    // Columns: a list of at most kSortedLines entries runs through the experts in order of descending R_e.  Both orders
    // hold the same entries, so the sum can be had first.
    int mine = 0;
    for (int e = lane; e < E; e += 64) mine += plan.share(true, kind, e);
    total = __shfl(wave_inclusive_scan(mine, lane), 63, 64);
    const bool sorted = total <= kSortedLines;
    int run = 0, sum_blocks = 0, head = -1;
    for (int o0 = 0; o0 < E; o0 += 64) {
      const int o = o0 + lane, e = o < E ? (sorted ? s.order[o] : o) : 0;
      const int n = o < E ? plan.share(true, kind, e) : 0;
      const int inc = wave_inclusive_scan(n, lane);
      if (o < E) s.base[l * E + o] = run + inc - n;
      run += __shfl(inc, 63, 64);
      sum_blocks += n * plan.rows_of(e);
      const uint64_t some = __ballot(n > 0);
      if (head < 0 && some) head = __shfl(e, __ffsll((unsigned long long)some) - 1, 64);
    }
    sum_blocks = __shfl(wave_inclusive_scan(sum_blocks, lane), 63, 64);
    if (lane == 0) s.count[l] = total, s.blocks[l] = sum_blocks, s.longest[l] = head >= 0 ? plan.rows_of(head) : 0;
  }
  __syncthreads();

  const int block_cols = E * width;
  int32_t* lists = reinterpret_cast<int32_t*>(g.plan + plan_list_offset(g.block_rows, block_cols));
  uint8_t* hints = g.plan + plan_slices_offset(g.block_rows, block_cols);
  const int64_t nnz = (int64_t)g.block_rows * width;
  for (int l = 0; l < 10; l++) {
    const bool cols = l >= kPlanLists, sorted = cols && s.count[l] <= kSortedLines;
    const int kind = l % kPlanLists, lines = cols ? block_cols : g.block_rows;
    int32_t* list = lists + 2 * kPlanLists + (cols ? kPlanLists * (int64_t)g.block_rows : 0) + (int64_t)kind * lines;
    const int* base = s.base + l * E;
    for (int64_t x = thread; x < s.count[l]; x += threads) {
      const int o = last_not_above([&](int i) { return base[i]; }, E, (int)x);   // (of equal ones the last: the one with entries)
      list[x] = plan.line(cols, kind, sorted ? s.order[o] : o, (int)x - base[o]);
    }
  }
  const int total_tiles = s.count[10];
  const bool fits = total_tiles <= g.max_sdd_tiles;
  for (int64_t t = thread; t < total_tiles && fits; t += threads) {
    const int e = last_not_above([&](int i) { return s.tiles[i]; }, E, (int)t);
    plan.sdd_tile(e, (int)t - s.tiles[e], g.sdd + 2 + 2 * t);
  }
  if (group == 0 && tid < 10) {
    lists[tid] = s.count[tid];
    // entries that go to one compute die at a time: a quarter of a die's share of the list's blocks (plan.hip)
    int entries = 1;
    const int fit = s.blocks[tid] / (32 * (s.longest[tid] > 0 ? s.longest[tid] : 1));
    while (s.count[tid] > 0 && entries < 32 && 2 * entries <= fit) entries *= 2;
    hints[(tid >= kPlanLists ? kPlanHintBytes : 0) + kGroupHint + tid % kPlanLists] = (uint8_t)entries;
    if (tid == 0) g.sdd[0] = fits ? total_tiles : 0, g.sdd[1] = 0;
  }
  if (group == 0 && wave < 2) {
    // wavefront 0 the rows, wavefront 1 the columns: do equal eighths of the lines hold about equal numbers of blocks?
    const bool cols = wave == 1;
    const int lines = cols ? block_cols : g.block_rows;
    uint8_t* h = hints + (cols ? kPlanHintBytes : 0);
    bool uneven = false;
    if (lane < 8) {
      auto offset_of = [&](int64_t line) -> int64_t {
        if (!cols) return line * width;
        const int e = (int)(line / width);
        return (int64_t)s.first[e] * width + (line % width) * (e < E ? plan.rows_of(e) : 0);
      };
      const int64_t share = offset_of((int64_t)(lane + 1) * lines / 8) - offset_of((int64_t)lane * lines / 8);
      uneven = share * 32 > nnz * 5;
    }
    const uint64_t any = __ballot(uneven);
    if (lane == 0) h[kSpreadHint] = any != 0;
    // from which width of the dense operand on stripes beat lines
    if (lane < 2) {
      const int* b = s.blocks + (cols ? kPlanLists : 0);
      const int64_t panels = lane == 0 ? (int64_t)b[kTallPairs] + b[kTallTriples] + b[kTallSingles] : (int64_t)b[kPairs] + b[kSingles];
      const int64_t saved = panels - (cols ? g.block_rows : block_cols);
      int from = 0;
      if (!FOURS && saved > 0) {
        const int64_t wide = (7 * nnz + saved - 1) / saved;
        from = wide > 255 ? 0 : (wide < 1 ? 1 : (int)wide);
      }
      h[kStripeHint + lane] = (uint8_t)from;
    }
  }
}

// The launches of one direction and width of the dense operand, a wavefront per number of slices.  All that they need of
// the plan is how many groups of each height a direction has, which every wavefront adds up for itself without the order
// of the experts and the shares in front of each.
constexpr int kSimulations = 2 * kTailSliceColumns;
static_assert(kMaxTailSlices == 4, "one wavefront per number of slices");
template <bool FOURS>
__device__ __forceinline__ void dmoe_simulation(const DmoeArgs& g, const DmoeLds& s, int item) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const DmoePlan<FOURS> plan{g, s.first};
  const bool cols = item >= kTailSliceColumns;
  const int column = item % kTailSliceColumns, ntn = column + 1, block_cols = g.experts * g.width, lines = cols ? block_cols : g.block_rows;
  int pairs = 0, triples = 0, singles = 0;
  for (int e = lane; e < g.experts; e += 64) {
    pairs += plan.share(cols, kTallPairs, e);
    triples += plan.share(cols, kTallTriples, e);
    singles += plan.share(cols, kTallSingles, e);
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) pairs += __shfl_xor(pairs, d, 64), triples += __shfl_xor(triples, d, 64), singles += __shfl_xor(singles, d, 64);
  const int kinds[3] = {uniform_int(pairs * ntn), uniform_int(triples * 2 * ntn), uniform_int(singles * ntn)};
  float end = 0.f;
  if (tail_slices_considered(kinds[0] + kinds[1] + kinds[2], g.compute_units)) {
    WaveSim sim;
    end = simulate_launch(sim, kinds, (float)((int64_t)g.block_rows * g.width) / (float)lines, g.compute_units, uniform_int(wave) + 1);
  }
  if (lane == 0) s.ends[wave] = end;
  __syncthreads();
  if (tid == 0) {
    const float all[kMaxTailSlices] = {s.ends[0], s.ends[1], s.ends[2], s.ends[3]};
    uint8_t* h = g.plan + plan_slices_offset(g.block_rows, block_cols) + (cols ? kPlanHintBytes : 0);
    h[column] = (uint8_t)choose_tail_slices(all);
  }
}

// The arrays of the topology; first(e) = first block row of expert e.
template <typename IDX, class First>
__device__ __forceinline__ void dmoe_arrays(const DmoeArgs& g, First&& first, int64_t thread, int64_t threads) {
  const int E = g.experts, width = g.width;
  const int64_t nnz = (int64_t)g.block_rows * width, columns = (int64_t)E * width;
  const int64_t work = nnz > columns + 1 ? nnz : columns + 1;
  IDX* row_indices = static_cast<IDX*>(g.row_indices);
  IDX* column_indices = static_cast<IDX*>(g.column_indices);
  IDX* column_indices_t = static_cast<IDX*>(g.column_indices_t);
  for (int64_t p = thread; p < work; p += threads) {
    if (p < nnz) {
      const int i = (int)(p / width), j = (int)(p % width);
      const int e = last_not_above(first, E, i);
      const int f = first(e);
      row_indices[p] = (IDX)i;
      column_indices[p] = (IDX)(e * width + j);
      if (j == 0) g.offsets[i] = i * width;
      const int64_t q = (int64_t)f * width + (int64_t)j * (first(e + 1) - f) + (i - f);
      if (q >= 0 && q < nnz) {   // (false for bins that do not ascend, without a plan, only)
        column_indices_t[q] = (IDX)i;
        g.block_offsets_t[q] = (int32_t)p;
      }
    }
    if (p <= columns) {
      if (p == columns) {
        g.offsets_t[p] = (int32_t)nnz;
        g.offsets[g.block_rows] = (int32_t)nnz;
      } else {
        const int e = (int)(p / width), j = (int)(p % width);
        g.offsets_t[p] = (int32_t)((int64_t)first(e) * width + (int64_t)j * (first(e + 1) - first(e)));
      }
    }
  }
}

template <typename IDX, bool FOURS>
__global__ __launch_bounds__(256) void dmoe_plan_kernel(DmoeArgs g) {
  extern __shared__ int lds[];
  const DmoeLds s(lds, g.experts);
  bool descends = false;
  for (int e = threadIdx.x; e <= g.experts; e += 256) {
    s.first[e] = first_row_of(g, e);
    descends |= e < g.experts && first_row_of(g, e + 1) < s.first[e];
  }
  // Bins that do not ascend are read as their running maximum: an expert whose bin lies below an earlier one has no rows.
  // The experts' rows then add up to block_rows, which is what the lengths of the plan's lists rest on.
  if (__syncthreads_or(descends)) {
    if (threadIdx.x == 0)
      for (int e = 1; e <= g.experts; e++) s.first[e] = max(s.first[e], s.first[e - 1]);
    __syncthreads();
  }
  // The workgroups in front simulate, the others write the arrays and the lists beside them.  One behind the other in the same
  // workgroups: 128 slots over 64 experts of 32 block columns 16.7 us, 15.4 like this; 16 384 slots 19.1 and 16.7 us.
  if (blockIdx.x < kSimulations) {
    dmoe_simulation<FOURS>(g, s, blockIdx.x);
    return;
  }
  const int group = (int)blockIdx.x - kSimulations;
  const int64_t thread = group * (int64_t)256 + threadIdx.x, threads = (int64_t)(gridDim.x - kSimulations) * 256;
  dmoe_arrays<IDX>(g, [&](int e) { return s.first[e]; }, thread, threads);
  dmoe_plan<FOURS>(g, s, group, thread, threads);
}

// Without a plan: any number of experts, the bins read where they are.
template <typename IDX>
__global__ __launch_bounds__(256) void dmoe_topology_kernel(DmoeArgs g) {
  const int64_t thread = blockIdx.x * (int64_t)256 + threadIdx.x, threads = (int64_t)gridDim.x * 256;
  dmoe_arrays<IDX>(g, [&](int e) { return first_row_of(g, e); }, thread, threads);
}

}  // namespace stk

extern "C" int stk_dmoe_topology(const int32_t* padded_bins, int64_t num_experts, int blocking, int64_t block_rows,
                                 int64_t blocks_per_row, int index_dtype, int32_t* offsets, void* row_indices,
                                 void* column_indices, int32_t* offsets_t, void* column_indices_t, int32_t* block_offsets_t,
                                 stk_stream_t stream) {
  return stk_dmoe_topology_plan(padded_bins, num_experts, blocking, block_rows, blocks_per_row, index_dtype, offsets, row_indices, column_indices,
                                offsets_t, column_indices_t, block_offsets_t, nullptr, 0, stream);
}

extern "C" int stk_dmoe_topology_plan(const int32_t* padded_bins, int64_t num_experts, int blocking, int64_t block_rows,
                                      int64_t blocks_per_row, int index_dtype, int32_t* offsets, void* row_indices,
                                      void* column_indices, int32_t* offsets_t, void* column_indices_t, int32_t* block_offsets_t,
                                      uint8_t* plan, size_t plan_bytes, stk_stream_t stream) {
  using namespace stk;
  const char* who = plan ? "stk_dmoe_topology_plan" : "stk_dmoe_topology";
  if (index_dtype != STK_I16 && index_dtype != STK_I32) return fail(STK_ERR_UNSUPPORTED, "%s: index dtype %d", who, index_dtype);
  if (num_experts <= 0 || blocking <= 0 || block_rows < 0 || blocks_per_row <= 0)
    return fail(STK_ERR_DIMS, "%s: %lld experts, blocking %d, %lld block rows of %lld blocks", who, (long long)num_experts,
                blocking, (long long)block_rows, (long long)blocks_per_row);
  const int64_t nnz = block_rows * blocks_per_row, columns = num_experts * blocks_per_row;
  if (nnz > INT32_MAX || columns >= INT32_MAX || block_rows * blocking > INT32_MAX)
    return fail(STK_ERR_UNSUPPORTED, "%s: size exceeds 32-bit range", who);
  if (index_dtype == STK_I16 && (block_rows > 32767 || columns > 32767))
    return fail(STK_ERR_DIMS, "%s: %lld block rows x %lld block columns do not fit 16-bit indices", who, (long long)block_rows, (long long)columns);
  if (!padded_bins || !offsets || !offsets_t || (nnz > 0 && (!row_indices || !column_indices || !column_indices_t || !block_offsets_t)))
    return fail(STK_ERR_DIMS, "%s: missing pointer", who);
  DmoeArgs g{padded_bins, (int)num_experts, blocking, (int)block_rows, (int)blocks_per_row, offsets, row_indices, column_indices,
             offsets_t, column_indices_t, block_offsets_t, nullptr, nullptr, 0, 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t work = nnz > columns + 1 ? nnz : columns + 1;
  const int64_t groups = (work + 255) / 256;
  if (!plan) {
    const dim3 grid((unsigned)(groups < 65536 ? groups : 65536));
    if (index_dtype == STK_I32) hipLaunchKernelGGL((dmoe_topology_kernel<int32_t>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((dmoe_topology_kernel<int16_t>), grid, dim3(256), 0, s, g);
    return check_launch(who);
  }
  if (blocking != 64 && blocking != 128) return fail(STK_ERR_UNSUPPORTED, "%s: a plan for blocking %d (64 or 128)", who, blocking);
  if (num_experts > kPlanExperts) return fail(STK_ERR_UNSUPPORTED, "%s: a plan for %lld experts (at most %d)", who, (long long)num_experts, kPlanExperts);
  if (nnz == 0) return fail(STK_ERR_UNSUPPORTED, "%s: a plan for no blocks", who);
  if (plan_bytes < stk_plan_bytes(block_rows, columns, nnz))
    return fail(STK_ERR_WORKSPACE, "%s: plan buffer of %zu bytes needed", who, stk_plan_bytes(block_rows, columns, nnz));
  if (reinterpret_cast<uintptr_t>(plan) & 3u) return fail(STK_ERR_UNSUPPORTED, "%s: plan buffer needs 4-byte alignment", who);
  g.sdd = reinterpret_cast<int32_t*>(plan);
  g.plan = plan + plan_sdd_bytes(block_rows, nnz);
  g.max_sdd_tiles = sdd_max_tiles(block_rows, nnz);
  g.compute_units = compute_units();
  const dim3 grid((unsigned)(kSimulations + (groups < 1024 ? groups : 1024)));
  const size_t lds = DmoeLds::bytes((int)num_experts);
#define STK_DMOE_CASE(I32, T, FOURS)                                                                    \
  if ((index_dtype == STK_I32) == I32 && (blocking == 64) == FOURS) {                                   \
    static const int once = (set_lds_limit(&dmoe_plan_kernel<T, FOURS>, (int)DmoeLds::bytes(kPlanExperts)), 0); \
    (void)once;                                                                                         \
    hipLaunchKernelGGL((dmoe_plan_kernel<T, FOURS>), grid, dim3(256), lds, s, g);                       \
  }
  STK_DMOE_CASE(true, int32_t, true) STK_DMOE_CASE(true, int32_t, false) STK_DMOE_CASE(false, int16_t, true) STK_DMOE_CASE(false, int16_t, false)
#undef STK_DMOE_CASE
  return check_launch(who);
}
